// Device-side stages of deterministic signing, shared by the device-driven
// rounds, the per-stage form (host-driven rejection rounds) and the persistent
// kernel; hash_row.hpp has the hashes with more lanes each.
//
// Fixed part per item (api.cu:117-182):
//   mu = SHAKE256(tr || m), rhoprime = SHAKE256(key || mu)   lane pair, row or wave per item
//   A = ExpandA(rho)                                         lane or wave per entry
//   s2 | s1 and the limbs of t0 as int8 (unpack of sk)        lane per 8 coefficients
// One attempt (item, nonce) in a "slot" (sign.cu:463-1196):
//   y    per (slot, l)        raw ExpandMask squeeze of rhoprime || L*nonce+l
//   w    wave per slot        NTT(y), A y^, INTT, caddq -> w; pack w1
//   c    per slot             c~ = SHAKE256(mu || w1), c = SampleInBall(c~)
//   z    wave per slot        c s2, c s1, c t0 on the matrix cores
//                             (ringmul.hpp), the norm checks, z = y + c s1,
//                             MakeHint, pack z and h
#pragma once

#include <hip/hip_runtime.h>

#include "layout.hpp"
#include "pipelines.hpp"
#include "poly.hpp"
#include "ringmul.hpp"
#include "sample.hpp"

namespace dil {

struct SignArgs {
    uint8_t *sig;  // final signatures
    size_t sig_pitch;
    const uint8_t *sk;
    size_t sk_pitch;
    MsgRef m;
    uint8_t *rows;  // SignLayout rows (item state)
    size_t row_pitch;
    size_t off_ints;  // byte offset of the expanded arrays (A, then s2 | s1 | t0 limbs as int8) in a row
    size_t n;
    // Resident keys (optional): when key_idx is set, item i signs with key
    // k = min(key_idx[i], nkeys - 1); its secret key is sk + k * sk_pitch and
    // its expanded arrays (A, s2, s1, t0) sit at key_ints + k * key_pitch
    // instead of in the item's row.  (Out-of-range indices are clamped so
    // that no access leaves the store.)
    const uint32_t *key_idx;
    const uint8_t *key_ints;
    size_t key_pitch;
    uint32_t nkeys;
    // Randomized signing (optional): item i's rhoprime is the 64 bytes at
    // rnd + i * rnd_pitch instead of SHAKE256(key || mu) (api.cu:143-148).
    const uint8_t *rnd;
    size_t rnd_pitch;
    // Long messages: mu / rhoprime with one sponge per 16-lane row at least,
    // whatever the batch size.
    int row_mu;
};

__device__ __forceinline__ size_t sk_index(const SignArgs &a, size_t i) {
    if (!a.key_idx) return i;
    const uint32_t k = a.key_idx[i];
    return k < a.nkeys ? k : a.nkeys - 1;
}

// Control block of one chain of signing rounds (SignLayout::CHAIN of the
// chain's first row).
struct ChainCtl {
    uint32_t left;   // items without a signature: entries of list `cur`
    uint32_t count;  // entries [0, count) take part in the current round
    uint32_t m;      // attempts (consecutive nonces) per item of the round
    uint32_t cur;    // which of the two lists
    uint32_t head;   // the finishing persistent kernel's queue head
};
static_assert(sizeof(ChainCtl) <= 256 - 136, "control block fits the row's mu area");

// One chain of rounds.  The items without a signature are a list of entries
// {item, next nonce}; two lists alternate.  They lie in chunks of 512 entries
// (8 KiB: both lists) `chunk_pitch` bytes apart, so that a caller's pool rows
// can hold them.
constexpr uint32_t CHAIN_CHUNK = 512;
constexpr size_t CHAIN_CHUNK_BYTES = CHAIN_CHUNK * 2 * sizeof(uint2);
struct Chain {
    uint8_t *rows;  // row of the chain's first item
    uint8_t *lists;
    size_t chunk_pitch;
    uint32_t first, n;
    uint32_t nslots;  // attempt slots of the chain
    uint32_t target;  // attempts a round aims at when fewer items are left
};

template <class P>
__device__ __forceinline__ ChainCtl *chain_ctl(const Chain &ch) {
    return reinterpret_cast<ChainCtl *>(ch.rows + SignLayout<P>::CHAIN);
}
__device__ __forceinline__ uint2 *chain_entry(const Chain &ch, uint32_t list, uint32_t e) {
    return reinterpret_cast<uint2 *>(ch.lists + (e / CHAIN_CHUNK) * ch.chunk_pitch) + list * CHAIN_CHUNK +
           e % CHAIN_CHUNK;
}

// Scratch and signature destination of attempt slots.
struct SlotRef {
    uint8_t *base;  // SlotLayout of slot s at base + s * pitch
    size_t pitch;
    uint8_t *sig;  // signature bytes of slot s at sig + s * sig_pitch
    size_t sig_pitch;
};

template <class P>
struct ItemView {
    using Z = Sizes<P>;
    using SLy = SignLayout<P>;
    uint8_t *row;
    const int32_t *mat;
    const int8_t *s8;  // s2 (K polynomials) | s1 (L)
    const int8_t *t8;  // t0's low limbs (K) | high limbs (K)
    __device__ ItemView(const SignArgs &a, size_t item) {
        row = a.rows + item * a.row_pitch;
        mat = a.key_idx ? reinterpret_cast<const int32_t *>(a.key_ints + sk_index(a, item) * a.key_pitch)
                        : reinterpret_cast<const int32_t *>(row + a.off_ints);
        s8 = reinterpret_cast<const int8_t *>(mat + P::K * P::L * N);
        t8 = s8 + (P::K + P::L) * N;
    }
};

__device__ __forceinline__ void load_words8(uint64_t (&w)[8], const uint8_t *p) {
#pragma unroll
    for (int i = 0; i < 8; ++i) w[i] = reinterpret_cast<const uint64_t *>(p)[i];
}

// ---------------------------------------------------------------- fixed part

// mu and rhoprime with two lanes per item (keccak_f1600_pair): lane h of the pair
// holds the 32-bit halves h of the state.  A permutation takes 2/3 of the
// one-lane form's time for 1.2 x its instructions, so the serial absorb of
// the batch's longest message, which bounds the fixed stage, is shorter.
template <class P>
__device__ __forceinline__ void stage_mu_pair(const SignArgs &a, size_t i, uint32_t h) {
    using Z = Sizes<P>;
    using SLy = SignLayout<P>;
    const uint8_t *sk = a.sk + sk_index(a, i) * a.sk_pitch;
    const uint8_t *m = a.m.ptr(i);
    const uint32_t mlen = a.m.len(i);
    uint32_t s[25];
    shake_pair<SHAKE256_RATE>(s, h, SEEDBYTES + mlen, [&](uint32_t w) -> uint32_t {
        if (w < 4) return load_half_bytes(sk + Z::SK_TR, 8 * w + 4 * h, SEEDBYTES);
        return load_half_bytes(m, 8 * (w - 4) + 4 * h, mlen);
    });
    uint32_t *row = reinterpret_cast<uint32_t *>(a.rows + i * a.row_pitch);
#pragma unroll
    for (int w = 0; w < 8; ++w) row[SLy::MU / 4 + 2 * w + h] = s[w];
    if (a.rnd) {
        const uint8_t *r = a.rnd + i * a.rnd_pitch;
#pragma unroll
        for (int w = 0; w < 8; ++w) row[SLy::RHOPRIME / 4 + 2 * w + h] = load_half_bytes(r, 8 * w + 4 * h, CRHBYTES);
        return;
    }
    // rhoprime = SHAKE256(key || mu): 96 bytes, one block
    uint32_t t[25];
#pragma unroll
    for (int w = 0; w < 25; ++w) t[w] = 0u;
#pragma unroll
    for (int w = 0; w < 4; ++w) t[w] = load_half_bytes(sk + Z::SK_KEY, 8 * w + 4 * h, SEEDBYTES);
#pragma unroll
    for (int w = 0; w < 8; ++w) t[4 + w] = s[w];
    if (h == 0) t[12] ^= 0x1Fu;
    if (h == 1) t[SHAKE256_RATE / 8 - 1] ^= 0x80000000u;
    keccak_f1600_pair(t, h);
#pragma unroll
    for (int w = 0; w < 8; ++w) row[SLy::RHOPRIME / 4 + 2 * w + h] = t[w];
}

template <class P>
__device__ __forceinline__ void stage_expand_a(const SignArgs &a, size_t i, int k, int l) {
    const uint8_t *sk = a.sk + i * a.sk_pitch;
    uint64_t rho[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) rho[w] = load_le64(sk + 8 * w);
    int32_t *dst = reinterpret_cast<int32_t *>(a.rows + i * a.row_pitch + a.off_ints) + (k * P::L + l) * N;
    // Four consecutive coefficients per 16-byte store: lanes write different
    // rows, so each store instruction touches one cache line per lane, and a
    // store per coefficient made the kernel wait on its writes.  (Row pitches
    // and the int32 area offset are multiples of 16; the entry points check.)
    int4 *dst4 = reinterpret_cast<int4 *>(dst);
    int32_t b0 = 0, b1 = 0, b2 = 0;  // the last three accepted coefficients
    uniform_poly(rho, (uint32_t)((k << 8) | l), [&](int ctr, int32_t v) {
        if ((ctr & 3) == 3) dst4[ctr >> 2] = make_int4(b0, b1, b2, v);
        b0 = b1;
        b1 = b2;
        b2 = v;
    });
}

// Coefficients 8c .. 8c + 7 (c < 32) of poly p of the item's secret key as
// int8, for the products with the challenge: p < L: s1[p], p < L + K: s2,
// else t0, whose 13-bit coefficients become a low limb in [-64, 64) and a
// high limb, t0 = lo + 128 hi.  dst: the item's s8 area (ItemView).
template <class P>
__device__ __forceinline__ void stage_prep(const uint8_t *sk, int8_t *dst, int p, int c) {
    using Z = Sizes<P>;
    uint32_t lo[2] = {0, 0}, hi[2] = {0, 0};
    if (p < P::L + P::K) {
        const uint8_t *src = sk + Z::SK_S1 + p * Z::POLYETA_BYTES + c * Z::ETA_BITS;
        uint32_t v;
        if constexpr (Z::ETA_BITS == 4)
            v = load_any<uint32_t>(src);
        else
            v = load_any<uint16_t>(src) | (uint32_t)src[2] << 16;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int32_t x = P::ETA - (int32_t)((v >> (j * Z::ETA_BITS)) & ((1u << Z::ETA_BITS) - 1u));
            lo[j >> 2] |= ((uint32_t)x & 0xFFu) << (8 * (j & 3));
        }
        const int row = p < P::L ? P::K + p : p - P::L;
        *reinterpret_cast<uint2 *>(dst + row * N + 8 * c) = make_uint2(lo[0], lo[1]);
    } else {
        const int k = p - P::L - P::K;
        const uint8_t *src = sk + Z::SK_T0 + k * POLYT0_BYTES + c * 13;
        const uint64_t a = load_any<uint64_t>(src), b = load_any<uint64_t>(src + 5);  // bits 0.., 40..
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t f = (uint32_t)(j < 4 ? a >> (13 * j) : b >> (13 * j - 40)) & 0x1FFFu;
            const int32_t x = (1 << (D - 1)) - (int32_t)f, h = (x + 64) >> 7;
            lo[j >> 2] |= ((uint32_t)(x - 128 * h) & 0xFFu) << (8 * (j & 3));
            hi[j >> 2] |= ((uint32_t)h & 0xFFu) << (8 * (j & 3));
        }
        int8_t *t8 = dst + (P::K + P::L) * N;
        *reinterpret_cast<uint2 *>(t8 + k * N + 8 * c) = make_uint2(lo[0], lo[1]);
        *reinterpret_cast<uint2 *>(t8 + (P::K + k) * N + 8 * c) = make_uint2(hi[0], hi[1]);
    }
}

// ------------------------------------------------------------- attempt part

template <class P>
__device__ __forceinline__ void stage_y(const SignArgs &a, size_t item, uint32_t nonce, int l, uint8_t *slot) {
    using Z = Sizes<P>;
    uint64_t rp[8];
    load_words8(rp, a.rows + item * a.row_pitch + SignLayout<P>::RHOPRIME);
    mask_raw(rp, (uint32_t)(P::L * nonce + l) & 0xFFFF,
             reinterpret_cast<uint64_t *>(slot + SlotLayout<P>::YRAW + l * Z::YRAW_BYTES));
}

// stage_y with two lanes per sponge (both lanes of the pair call it)
template <class P>
__device__ __forceinline__ void stage_y_pair(const SignArgs &a, size_t item, uint32_t nonce, int l, uint8_t *slot,
                                             uint32_t h) {
    using Z = Sizes<P>;
    mask_raw_pair(reinterpret_cast<const uint32_t *>(a.rows + item * a.row_pitch + SignLayout<P>::RHOPRIME),
                  (uint32_t)(P::L * nonce + l) & 0xFFFF,
                  reinterpret_cast<uint32_t *>(slot + SlotLayout<P>::YRAW + l * Z::YRAW_BYTES), h);
}

template <class P>
__device__ __forceinline__ void load_y_A(int32_t (&v)[4], const uint8_t *slot, int l) {
    using Z = Sizes<P>;
    uint32_t f[4];
    wave_fields_A<Z::Z_BITS>(f, slot + SlotLayout<P>::YRAW + l * Z::YRAW_BYTES);
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = P::GAMMA1 - (int32_t)f[r];
}

template <class P>
__device__ __forceinline__ void load_y_D(int32_t (&v)[4], const uint8_t *slot, int l) {
    using Z = Sizes<P>;
    uint32_t f[4];
    wave_fields_D<Z::Z_BITS>(f, slot + SlotLayout<P>::YRAW + l * Z::YRAW_BYTES);
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = P::GAMMA1 - (int32_t)f[r];
}

// One coefficient's decomposition in a word of the slot's w area: high bits
// above bit 20, low bits (|w0| <= gamma2 < 2^19) below.
__device__ __forceinline__ uint32_t pack_w(int32_t w1, int32_t w0) { return (uint32_t)w1 << 20 | ((uint32_t)w0 & 0xFFFFFu); }
__device__ __forceinline__ int32_t packed_w0(uint32_t p) { return (int32_t)(p << 12) >> 12; }
__device__ __forceinline__ uint32_t packed_w1(uint32_t p) { return p >> 20; }

// w for M attempts of the same item (slots[0..M)) in one wave: every A row
// is loaded once for all M products, and the M transforms give the wave
// independent work to overlap with the loads.
// ylds: with M > 1 and L = 7 the M x 7 transformed y polynomials live in
// this wave's LDS area (M * L * N words) instead of registers, where they
// would not fit beside the A rows and the INTT
template <class P, int M>
__device__ __forceinline__ void stage_w_multi(const SignArgs &a, size_t item, uint8_t *const (&slots)[M], int32_t *x,
                                              const ZetaLds &zt, int32_t *ylds = nullptr) {
    using Z = Sizes<P>;
    using SL = SlotLayout<P>;
// smallest L whose paired y vectors go to LDS (for L = 4 and 5 moving them
// there freed 10-27 VGPRs and changed nothing measurable)
#ifndef DIL_W_Y_LDS_MIN_L
#define DIL_W_Y_LDS_MIN_L 6
#endif
    constexpr bool Y_LDS = M > 1 && P::L >= DIL_W_Y_LDS_MIN_L;
    const ItemView<P> it(a, item);
    // A rows are streamed from HBM with the next row's loads issued before
    // the current row's products and INTTs (software prefetch)
    int32_t an[P::L][4];
#pragma unroll
    for (int l = 0; l < P::L; ++l) wave_load_D(an[l], it.mat + l * N);
    int32_t yh[Y_LDS ? 1 : M][Y_LDS ? 1 : P::L][4];
#pragma unroll
    for (int j = 0; j < M; ++j)
#pragma unroll
        for (int l = 0; l < P::L; ++l) {
            int32_t t[4];
            load_y_A<P>(t, slots[j], l);
            ntt_wave(t, x, zt);
            if constexpr (Y_LDS) {
                wave_store_D(ylds + (j * P::L + l) * N, t);
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) yh[j][l][r] = t[r];
            }
        }
    for (int k = 0; k < P::K; ++k) {
        // the L products of a coefficient are summed in 64 bits (one
        // v_mad_i64_i32 each) and reduced once; |sum| < 7 q 2^26.1 < 2^53, so
        // the reduced sum is below q / 2 + 2^21 and the INTT cannot overflow
        int64_t sum[M][4];
        int32_t acc[M][4];
        int32_t ac[P::L][4];
#pragma unroll
        for (int l = 0; l < P::L; ++l)
#pragma unroll
            for (int r = 0; r < 4; ++r) ac[l][r] = an[l][r];
        if (k + 1 < P::K) {
#pragma unroll
            for (int l = 0; l < P::L; ++l) wave_load_D(an[l], it.mat + ((k + 1) * P::L + l) * N);
        }
#pragma unroll
        for (int j = 0; j < M; ++j) {
#pragma unroll
            for (int r = 0; r < 4; ++r) sum[j][r] = 0;
#pragma unroll
            for (int l = 0; l < P::L; ++l) {
                if constexpr (Y_LDS) {
                    int32_t yv[4];
                    wave_load_D(yv, ylds + (j * P::L + l) * N);
#pragma unroll
                    for (int r = 0; r < 4; ++r) sum[j][r] += (int64_t)ac[l][r] * yv[r];
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r) sum[j][r] += (int64_t)ac[l][r] * yh[j][l][r];
                }
            }
        }
#pragma unroll
        for (int j = 0; j < M; ++j) {
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[j][r] = mont_reduce(sum[j][r]);
            intt_wave(acc[j], x, zt);
            int32_t w1[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                int32_t w0;
                w1[r] = decompose<P>(caddq(acc[j][r]), w0);
                acc[j][r] = (int32_t)pack_w(w1[r], w0);
            }
            wave_store_A(reinterpret_cast<int32_t *>(slots[j] + SL::W) + k * N, acc[j]);
            layout_A_to_D(w1, x);
            uint32_t u[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) u[r] = (uint32_t)w1[r];
            wave_pack_D<Z::W1_BITS>(slots[j] + SL::W1PK + k * Z::POLYW1_BYTES, u);
        }
    }
}

template <class P>
__device__ __forceinline__ void stage_w(const SignArgs &a, size_t item, uint8_t *slot, int32_t *x, const ZetaLds &zt) {
    uint8_t *const slots[1] = {slot};
    stage_w_multi<P, 1>(a, item, slots, x, zt);
}

template <class P>
__device__ __forceinline__ void stage_c(const SignArgs &a, size_t item, uint8_t *slot, uint8_t *sig_out) {
    using Z = Sizes<P>;
    using SL = SlotLayout<P>;
    const uint64_t *mu = reinterpret_cast<const uint64_t *>(a.rows + item * a.row_pitch + SignLayout<P>::MU);
    const uint64_t *w1 = reinterpret_cast<const uint64_t *>(slot + SL::W1PK);
    Lane64 s[25];
    shake_absorb<SHAKE256_RATE>(s, [&](uint32_t w, uint32_t) { return w < 8 ? mu[w] : w1[w - 8]; },
                                (uint32_t)Z::CHASH_IN_BYTES);
    uint64_t ct[4];
    squeeze_words<4>(s, ct);
#pragma unroll
    for (int w = 0; w < 4; ++w)
#pragma unroll
        for (int b = 0; b < 8; ++b) sig_out[8 * w + b] = (uint8_t)(ct[w] >> (8 * b));
    challenge<P::TAU>(ct, reinterpret_cast<uint32_t *>(slot + SL::CP));
}

// stage_c over a lane pair (keccak_f1600_pair): lanes 2j and 2j + 1 hash the
// same slot, each holding one 32-bit half of every state word, so a wave
// runs the challenge hash of 32 slots with a chain a third shorter than one
// state per lane.  h = lane & 1; both lanes of the pair must call it.
template <class P>
__device__ __forceinline__ void stage_c_pair(const SignArgs &a, size_t item, uint8_t *slot, uint8_t *sig_out,
                                             uint32_t h) {
    using Z = Sizes<P>;
    using SL = SlotLayout<P>;
    const uint32_t *mu = reinterpret_cast<const uint32_t *>(a.rows + item * a.row_pitch + SignLayout<P>::MU);
    const uint32_t *w1 = reinterpret_cast<const uint32_t *>(slot + SL::W1PK);
    uint32_t s[25];
    shake_absorb_pair<SHAKE256_RATE, Z::CHASH_IN_BYTES>(
        s, [&](uint32_t w) { return w < 8 ? mu[2 * w + h] : w1[2 * (w - 8) + h]; }, h);
    keccak_f1600_pair(s, h);
    uint64_t ct[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) ct[w] = pair_word(s, w, h);
    // c~: each lane of the pair writes its 4-byte halves (16 bytes)
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const uint32_t v = s[w];
#pragma unroll
        for (int b = 0; b < 4; ++b) sig_out[8 * w + 4 * h + b] = (uint8_t)(v >> (8 * b));
    }
    // the challenge block squeezed in the pair layout as well (one state per
    // lane: ~1 % slower loop for Dilithium3)
#ifndef DIL_CHALLENGE_PAIR
#define DIL_CHALLENGE_PAIR 1
#endif
    if constexpr (DIL_CHALLENGE_PAIR)
        challenge_pair<P::TAU>(ct, reinterpret_cast<uint32_t *>(slot + SL::CP), h);
    else
        challenge<P::TAU>(ct, reinterpret_cast<uint32_t *>(slot + SL::CP), h == 0);
}

// One wave's LDS area in the z stage: the challenge's operand table and the
// rows c s2 (K) | c s1 (L); once z is written, the rows c t0 of half of the
// K polynomials at a time (low limbs K / 2, high limbs K / 2) take the place
// of c s1.
template <class P, bool CHECK_ONLY = false>
struct ZScratch {
    static constexpr int ROWS = P::K + (CHECK_ONLY || P::L > P::K ? P::L : P::K);
    uint32_t toep[TOEP_WORDS];
    uint16_t rows[ROWS * RING_ROW];
};

// Returns true (wave-uniform) when the attempt passes every check; then
// sig_out holds the complete signature.  An attempt is accepted iff all of
// ||r0|| < gamma2 - beta, ||z|| < gamma1 - beta, ||c t0|| < gamma2 and
// #hints <= omega hold (sign.cu:986-1196), so the order of the checks does
// not change any result: c s2 and c s1 come from one set of matrix products,
// r0 is checked first because it rejects most often (about 2/3 of Dilithium3
// attempts), then z, and only the remaining fifth computes c t0 and the
// hints.  All values are exact integers below q / 2, where the reference's
// representatives mod q agree with them.  Fields of a rejected attempt's
// sig_out are left partly written.
// CHECK_ONLY: r0 and z are checked and nothing is written; c t0 and the hints
// (which reject about 2 % of what is left) are not looked at.
template <class P, bool CHECK_ONLY = false>
__device__ __forceinline__ bool stage_z(const SignArgs &a, size_t item, uint8_t *slot, uint8_t *sig_out,
                                        ZScratch<P, CHECK_ONLY> &zs) {
    using Z = Sizes<P>;
    using SL = SlotLayout<P>;
    const ItemView<P> it(a, item);
    const int lane = lane_id();
    // every load that the first check needs is issued before the first use
    const uint32_t *masks = reinterpret_cast<const uint32_t *>(slot + SL::CP) + toeplitz_word(lane);
    const uint32_t nzw = masks[0], ngw = masks[8];
    v4i B[4];
    wave_ring_load(B, it.s8 + min(lane & 15, P::K + P::L - 1) * N);
    const uint4 *wbase = reinterpret_cast<const uint4 *>(slot + SL::W) + lane;  // layout D
    uint4 w[P::K];
#pragma unroll
    for (int k = 0; k < P::K; ++k) w[k] = wbase[k * (N / 4)];
    wave_toeplitz(zs.toep, nzw, ngw);
    wave_ring_mul<P::K + P::L>(zs.rows, zs.toep, B);
    wave_lds_sync();

    // r0 = w0 - c s2
#pragma unroll
    for (int k = 0; k < P::K; ++k) {
        int32_t cs[4];
        wave_ring_row(cs, zs.rows + k * RING_ROW);
        const uint32_t wp[4] = {w[k].x, w[k].y, w[k].z, w[k].w};
        bool big = false;
#pragma unroll
        for (int r = 0; r < 4; ++r) big |= abs(packed_w0(wp[r]) - cs[r]) >= P::GAMMA2 - P::BETA;
        if (wave_any(big)) return false;
    }

    // z = y + c s1
    int32_t y[P::L][4];
#pragma unroll
    for (int l = 0; l < P::L; ++l) load_y_D<P>(y[l], slot, l);
#pragma unroll
    for (int l = 0; l < P::L; ++l) {
        int32_t cs[4];
        wave_ring_row(cs, zs.rows + (P::K + l) * RING_ROW);
        bool big = false;
        uint32_t f[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int32_t z = y[l][r] + cs[r];
            big |= abs(z) >= P::GAMMA1 - P::BETA;
            f[r] = (uint32_t)(P::GAMMA1 - z);
        }
        if (wave_any(big)) return false;
        if constexpr (!CHECK_ONLY) wave_pack_D<Z::Z_BITS>(sig_out + Z::SIG_Z + l * Z::POLYZ_BYTES, f);
    }
    if constexpr (CHECK_ONLY) return true;

    // c t0 in two halves of K / 2 polynomials; the hints in ascending
    // coefficient order j = 4 lane + r
    uint8_t *h = sig_out + Z::SIG_H;
    int pos = 0;
#pragma unroll 1
    for (int k0 = 0; k0 < P::K; k0 += P::K / 2) {
        const int col = min(lane & 15, P::K - 1);  // low limbs, then high limbs
        wave_ring_load(B, it.t8 + (col < P::K / 2 ? k0 + col : P::K / 2 + k0 + col) * N);
        wave_lds_sync();  // the rows are read by now
        wave_ring_mul<P::K>(zs.rows + P::K * RING_ROW, zs.toep, B);
        wave_lds_sync();
#pragma unroll 1
        for (int k = k0; k < k0 + P::K / 2; ++k) {
            int32_t cs[4], lo[4], hi[4];
            wave_ring_row(cs, zs.rows + k * RING_ROW);
            wave_ring_row(lo, zs.rows + (P::K + k - k0) * RING_ROW);
            wave_ring_row(hi, zs.rows + (P::K + P::K / 2 + k - k0) * RING_ROW);
            const uint4 wk = wbase[k * (N / 4)];
            const uint32_t wp[4] = {wk.x, wk.y, wk.z, wk.w};
            bool big = false;
            int hb[4], before = 0, cnt = 0;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int32_t ct0 = lo[r] + 128 * hi[r];
                big |= abs(ct0) >= P::GAMMA2;
                hb[r] = make_hint<P>(packed_w0(wp[r]) - cs[r] + ct0, (int32_t)packed_w1(wp[r]));
                const uint64_t m = __ballot(hb[r]);
                before += __popcll(m & ((1ull << lane) - 1ull));  // hints of lower lanes
                cnt += __popcll(m);
            }
            if (wave_any(big) || pos + cnt > P::OMEGA) return false;
            int idx = pos + before;
            pos += cnt;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (hb[r]) h[idx++] = (uint8_t)(4 * lane + r);
            if (lane == 0) h[P::OMEGA + k] = (uint8_t)pos;
        }
    }
    for (int j = pos + lane; j < P::OMEGA; j += 64) h[j] = 0;
    return true;
}

}  // namespace dil
