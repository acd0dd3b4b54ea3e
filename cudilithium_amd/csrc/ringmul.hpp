// Products of the challenge polynomial with small polynomials, on the matrix
// cores.
//
// c has coefficients in {-1, 0, 1} and s1, s2 and the two limbs of t0 fit
// int8, so c * s in Z[X] / (X^256 + 1) is an exact int8 contraction: with
// C~[d] = c[d] for d >= 0 and -c[256 + d] for d < 0,
//     (c s)[i] = sum_j C~[i - j] s[j],
// a 256 x 256 Toeplitz matrix times one column per polynomial.  One wave
// multiplies up to 16 polynomials with 64 v_mfma_i32_16x16x64_i8 (16 row
// tiles x 4 steps of 64 along j), 1,100 cycles of the matrix pipe for what
// one forward transform, 11 pointwise products and 11 inverse transforms
// (Dilithium3: s1 and s2) take about 10,000 cycles of vector ALU for, and the
// key's part of a signature's operands shrinks from 17 KiB of transformed
// int32 to 6 KiB of int8.  |c s| <= tau * 128 < 2^15, so results are int16.
#pragma once

#include <hip/hip_runtime.h>

#include "ntt.hpp"
#include "params.hpp"

namespace dil {

typedef int v4i __attribute__((ext_vector_type(4)));

// Operand table of one challenge in LDS: the bytes Rv[x] = C~[255 - x],
// x < 512, in four copies shifted by 0..3 bytes, so that a lane's 16 operand
// bytes (which start at any byte) are whole words.  The copies lie 16 banks
// apart: the 64 lanes of an operand read touch 64 different banks.
constexpr int TOEP_STRIDE = 128 + 16;
constexpr int TOEP_WORDS = 4 * TOEP_STRIDE;
// Result rows (one per polynomial): 256 int16 and 16 of padding.
constexpr int RING_ROW = N + 16;

// bit b of a nibble to byte b
__device__ __forceinline__ uint32_t nibble_bytes(uint32_t nib) { return (nib * 0x00204081u) & 0x01010101u; }

// Fills T from the challenge masks nz[8] | neg[8] (neg is a subset of nz):
// lane l passes words w = toeplitz_word(l) of both.
__device__ __forceinline__ int toeplitz_word(int l) { return 7 - (l >> 3); }
__device__ __forceinline__ void wave_toeplitz(uint32_t *T, uint32_t nz_word, uint32_t neg_word) {
    const int l = lane_id();
    // word l holds x = 4l .. 4l + 3, i.e. c[255 - 4l] downwards: nibble l of
    // the bit-reversed masks
    const int sh = 4 * (l & 7);
    const uint32_t nz = nibble_bytes((__brev(nz_word) >> sh) & 15u);
    const uint32_t ng = nibble_bytes((__brev(neg_word) >> sh) & 15u);
    wave_lds_sync();
    T[l] = nz + ng * 0xFEu;              // 0x01 or, negative, 0xFF
    T[64 + l] = nz + (nz ^ ng) * 0xFEu;  // the negated half, x >= 256
    wave_lds_sync();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int y = 64 * h + l;
        const uint32_t a = T[y], b = T[y == 127 ? 127 : y + 1];  // the bytes after x = 511 are never used
#pragma unroll
        for (int s = 1; s < 4; ++s) T[s * TOEP_STRIDE + y] = __builtin_amdgcn_alignbyte(b, a, s);
    }
    wave_lds_sync();
}

// The right-hand operands of wave_ring_mul: lane (n, g) = (lane & 15,
// lane >> 4) holds bytes 64b + 16g .. + 15 of its column's polynomial, a
// 16-byte aligned int8 polynomial of N bytes at `poly`.
__device__ __forceinline__ void wave_ring_load(v4i (&B)[4], const int8_t *poly) {
    const int8_t *src = poly + 16 * (lane_id() >> 4);
#pragma unroll
    for (int b = 0; b < 4; ++b) B[b] = *reinterpret_cast<const v4i *>(src + 64 * b);
}

// rows[n] = c * (column n) for n < NCOL, int16 rows of RING_ROW.
//
// Row tile a (coefficients 16a .. 16a + 15) and step b (j = 64b ..) need, in
// lane (m, g), the 16 bytes C~[16a + m - 64b - 16g - t], t < 16: Rv from
// x = 16 (15 - (a - 4b) + g) + (15 - m).  They are read from the table for
// each product (half the LDS bandwidth) rather than held: 64 registers fewer
// let one or two more waves run on each SIMD.
template <int NCOL>
__device__ __forceinline__ void wave_ring_mul(uint16_t *rows, const uint32_t *T, const v4i (&B)[4]) {
    static_assert(NCOL <= 16, "one column tile");
    const int l = lane_id(), n = l & 15, g = l >> 4;
    const uint32_t *tl = T + ((15 - n) & 3) * TOEP_STRIDE + ((15 - n) >> 2) + 4 * (15 + g);
    uint16_t *dst = rows + n * RING_ROW + 4 * g;
#pragma unroll 1
    for (int A = 0; A < 4; ++A, tl -= 16, dst += 64) {
        v4i acc[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = v4i{0, 0, 0, 0};
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t *p = tl - 4 * (i - 4 * b);
                const v4i op{(int)p[0], (int)p[1], (int)p[2], (int)p[3]};
                acc[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(op, B[b], acc[i], 0, 0, 0);
            }
        if (n < NCOL) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                // low halves of two results per word
                const uint32_t lo = __builtin_amdgcn_perm((uint32_t)acc[i][1], (uint32_t)acc[i][0], 0x05040100u);
                const uint32_t hi = __builtin_amdgcn_perm((uint32_t)acc[i][3], (uint32_t)acc[i][2], 0x05040100u);
                *reinterpret_cast<uint2 *>(dst + 16 * i) = make_uint2(lo, hi);
            }
        }
    }
}

// a result row in layout D
__device__ __forceinline__ void wave_ring_row(int32_t (&v)[4], const uint16_t *row) {
    const uint2 t = reinterpret_cast<const uint2 *>(row)[lane_id()];
    v[0] = (int32_t)(t.x << 16) >> 16;
    v[1] = (int32_t)t.x >> 16;
    v[2] = (int32_t)(t.y << 16) >> 16;
    v[3] = (int32_t)t.y >> 16;
}

}  // namespace dil
