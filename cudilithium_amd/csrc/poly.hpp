// Polynomial data movement for one wavefront: loads and stores in the NTT
// register layouts (A: j = 64r + l, D: j = 4l + r) and little-endian
// bit-field packing, the byte format of every packed polynomial on the path
// (t1 10-bit, t0 13-bit, eta 3/4-bit, z 18/20-bit, w1 6/4-bit; see
// keypair.cu:116-130,268-301 and sign.cu:662-683,1151-1192).
#pragma once

#include <hip/hip_runtime.h>

#include "field.hpp"
#include "ntt.hpp"
#include "params.hpp"

namespace dil {

// Words per polynomial row of an LDS array that lanes walk in step, each in
// its own row (ExpandA lanes folding coefficient ctr of many rows at about
// the same ctr): with rows of N = 256 words every lane would hit the same
// bank.  Four words of padding spread 16 consecutive rows over the 64 banks
// and keep the rows 16-byte aligned (with uniform_poly's shorter test:
// verification of 65,536 Dilithium5 items 4.80 -> 4.23 ms, 16,384 Dilithium3
// keys 0.975 -> 0.867 ms).
constexpr int LDS_ROW = N + 4;

// Little-endian loads and stores at any byte address.  The GPU reads and
// writes global memory at any alignment in one instruction, so a packed
// polynomial in a caller's unaligned row is moved a word at a time.
template <class T>
__device__ __forceinline__ T load_any(const uint8_t *p) {
    T v;
    __builtin_memcpy(&v, p, sizeof(T));
    return v;
}
template <class T>
__device__ __forceinline__ void store_any(uint8_t *p, T v) {
    __builtin_memcpy(p, &v, sizeof(T));
}

// W-bit field j of a little-endian bit-packed polynomial (N fields, N * W / 8
// bytes) at any byte alignment: one 32-bit load, moved back at the end of the
// polynomial so that it stays inside (every field and its shift fit 32 bits).
template <int W>
__device__ __forceinline__ uint32_t field_at(const uint8_t *p, int j) {
    static_assert(W + 7 <= 32, "a field starting inside a byte fits one word");
    const int bit = j * W, off = min(bit >> 3, N * W / 8 - 4);
    return __builtin_amdgcn_ubfe(load_any<uint32_t>(p + off), (uint32_t)(bit - 8 * off), W);
}

// Stores the low NB bytes of a little-endian word array, any alignment.
template <int NB, int NW>
__device__ __forceinline__ void store_bytes(uint8_t *out, const uint32_t (&w)[NW]) {
    static_assert(NB <= 4 * NW, "enough words");
#pragma unroll
    for (int i = 0; i + 4 <= NB; i += 4) store_any<uint32_t>(out + i, w[i / 4]);
    if constexpr (NB & 2) store_any<uint16_t>(out + (NB & ~3), (uint16_t)w[NB / 4]);
    if constexpr (NB & 1) out[NB - 1] = (uint8_t)(w[NB / 4] >> (8 * ((NB - 1) & 3)));
}

// Packs C fields of W bits (C * W a multiple of 8) to out, any alignment.
template <int W, int C>
__device__ __forceinline__ void pack_store(uint8_t *out, const uint32_t (&c)[C]) {
    static_assert(C * W % 8 == 0, "whole bytes");
    constexpr int NW = (C * W + 31) / 32;
    uint32_t acc[NW];
#pragma unroll
    for (int i = 0; i < NW; ++i) acc[i] = 0;
#pragma unroll
    for (int i = 0; i < C; ++i) {
        const int bit = i * W, wi = bit >> 5, sh = bit & 31;
        acc[wi] |= c[i] << sh;
        if (sh + W > 32) acc[wi + 1] |= c[i] >> (32 - sh);
    }
    store_bytes<C * W / 8>(out, acc);
}

// Wave-level packing of a polynomial in layout D whose lane values are the
// W-bit fields: each lane packs its 4 coefficients when they fill whole
// bytes of at least 4, else even lanes pack 8 with their neighbour's.
template <int W>
__device__ __forceinline__ void wave_pack_D(uint8_t *out, const uint32_t (&v)[4]) {
    const int l = lane_id();
    if constexpr (W >= 8 && 4 * W % 8 == 0) {
        pack_store<W>(out + l * (W / 2), v);
    } else {
        uint32_t n[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) n[r] = (uint32_t)__shfl_down((int)v[r], 1);
        if ((l & 1) == 0) {
            const uint32_t c[8] = {v[0], v[1], v[2], v[3], n[0], n[1], n[2], n[3]};
            pack_store<W>(out + (l >> 1) * W, c);
        }
    }
}

// Wave-level unpack of W-bit fields into layout D (4 consecutive fields of
// W / 2 whole bytes per lane), any alignment.
template <int W>
__device__ __forceinline__ void wave_fields_D(uint32_t (&v)[4], const uint8_t *p) {
    static_assert(W % 2 == 0 && W > 16 && W <= 20, "9 or 10 bytes per lane");
    const uint8_t *q = p + lane_id() * (W / 2);
    const uint64_t lo = load_any<uint64_t>(q);
    const uint32_t d0 = (uint32_t)lo, d1 = (uint32_t)(lo >> 32);
    const uint32_t d2 = W == 18 ? (uint32_t)q[8] : (uint32_t)load_any<uint16_t>(q + 8);
    constexpr uint32_t M = (1u << W) - 1u;
    v[0] = d0 & M;
    v[1] = __builtin_amdgcn_alignbit(d1, d0, W) & M;
    v[2] = (d1 >> (2 * W - 32)) & M;
    v[3] = __builtin_amdgcn_alignbit(d2, d1, 3 * W - 32) & M;
}

// Wave-level unpack of W-bit fields into layout A.
template <int W>
__device__ __forceinline__ void wave_fields_A(uint32_t (&v)[4], const uint8_t *p) {
    const int l = lane_id();
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = field_at<W>(p, 64 * r + l);
}

__device__ __forceinline__ void wave_load_A(int32_t (&v)[4], const int32_t *p) {
    const int l = lane_id();
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = p[64 * r + l];
}
__device__ __forceinline__ void wave_store_A(int32_t *p, const int32_t (&v)[4]) {
    const int l = lane_id();
#pragma unroll
    for (int r = 0; r < 4; ++r) p[64 * r + l] = v[r];
}
__device__ __forceinline__ void wave_load_D(int32_t (&v)[4], const int32_t *p) {
    const int4 t = reinterpret_cast<const int4 *>(p)[lane_id()];
    v[0] = t.x;
    v[1] = t.y;
    v[2] = t.z;
    v[3] = t.w;
}
__device__ __forceinline__ void wave_store_D(int32_t *p, const int32_t (&v)[4]) {
    reinterpret_cast<int4 *>(p)[lane_id()] = make_int4(v[0], v[1], v[2], v[3]);
}
// Challenge polynomial from its masks (nz[8] | neg[8], see challenge()) in
// layout A: lane l, register r holds c[64 r + l] in {-1, 0, 1}.
__device__ __forceinline__ void wave_load_challenge_A(int32_t (&v)[4], const uint32_t *masks) {
    const int l = lane_id(), sh = l & 31, hi = l >> 5;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const uint32_t nzw = masks[2 * r + hi], ngw = masks[8 + 2 * r + hi];
        const int32_t nzb = (int32_t)((nzw >> sh) & 1u), ngb = (int32_t)((ngw >> sh) & 1u);
        v[r] = nzb - 2 * (nzb & ngb);
    }
}

// Wave-wide OR of a per-lane predicate.
__device__ __forceinline__ bool wave_any(bool p) { return __ballot(p) != 0ull; }

}  // namespace dil
