// Keccak-f[1600] with one state per wavefront, for the shortest chain.
//
// A sponge's permutations depend on each other, so a small batch's hashes take
// as long as their chains, whatever the card could do beside them.  The 16-lane
// row form (keccak_row.hpp) issues 54 vector instructions per round, one every
// 4.5 cycles, plus an LDS round trip: 350 cycles.  One 64-bit word per lane
// leaves 24 and five LDS instructions:
//
//   lane 8 y + p: word (x, y) with x = p for p < 5; p = 5 and p = 7 hold copies
//   of x = 0 and x = 4, so that neighbours along x are one lane away in both
//   directions; p = 6 and the lanes from 40 on hold zeros
//
//   theta  column parities: one DPP rotation by 8 joins the two y of a 16-lane
//          row; permlane32_swap of the two halves' registers then puts the low
//          halves' sums into lanes 0..31 and the high halves' into 32..63, one
//          permlane16_swap joins the rows, and a last permlane32_swap gives
//          every lane both halves of its column's parity.  C[x - 1] and
//          C[x + 1] come from the neighbouring lanes by DPP (the copies supply
//          the wrap; a column's parity is the same for every y, so the lane
//          rotation may cross rows of the state)
//   rho    two funnel shifts; as in the row form the shift yields the halves
//          in swapped places for R > 32 and R = 0, and the write address swaps
//          them back
//   pi     two LDS writes to per-lane addresses; reading the words x, x + 1,
//          x + 2 of the new row (three LDS reads) also serves chi
//
// A chained permutation takes 2.2 us on MI355X while a SIMD has one such wave
// (row form 3.5, lane pair 5.9, lane 8.6); 1,024 / 2,048 / 3,072 / 4,096 states
// on the card take 2.6 / 3.2 / 4.1 / 5.0 us, where the row form takes 3.5 to
// 3.9 us up to 4,096: the wave form is for up to 2,000 states, or 3,000 where the
// work around the hash gains from whole waves too.
//
// All 64 lanes must execute every call.  The round constants and rotation
// offsets are those of keccak.hpp.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "keccak.hpp"
#include "keccak_row.hpp"  // xor_dpp, DPP_ROW_ROR8

namespace dil {

// LDS words per wave: the 25 words of the pi exchange (word x + 5 y at 2 (x +
// 5 y)), a zero word that idle lanes read, a dummy word that they write
constexpr int WAVE_LDS_WORDS = 54;
constexpr int DPP_ROW_ROR1 = 0x121, DPP_ROW_SHL1 = 0x101;

struct WaveLane {
    uint32_t w;             // index x + 5 y of this lane's word, 25 for idle lanes
    bool main;              // the word's own lane (not a copy, not idle)
    uint32_t sh;            // rho funnel-shift amount
    uint32_t wlo, whi;      // pi destination of the two rotated halves
    uint32_t r0, r1, r2;    // words x, x + 1, x + 2 of the row after pi
    uint32_t iota_mask;     // all ones on the lanes of word 0
};

// base: first of the wave's WAVE_LDS_WORDS words (8-byte aligned) in lds
__device__ __forceinline__ WaveLane wave_lane_setup(uint32_t *lds, uint32_t base) {
    WaveLane r;
    const uint32_t lane = (uint32_t)lane_id(), p = lane & 7, y = lane >> 3;
    const uint32_t x = p < 5 ? p : (p == 5 ? 0 : 4);
    const bool active = y < 5 && p != 6;
    r.main = y < 5 && p < 5;
    r.w = active ? x + 5 * y : 25;
    if (lane < 2) lds[base + 50 + lane] = 0u;
    const int R = r.main ? kKeccak.rho[x + 5 * y] : 0;
    const bool swapped = R == 0 || R > 32;  // see row_lane_setup
    r.sh = (uint32_t)(swapped ? (64 - R) & 31 : 32 - R);
    const uint32_t dst = base + (r.main ? 2 * ((2 * x + 3 * y) % 5 * 5 + y) : 52);
    r.wlo = dst + (uint32_t)swapped;
    r.whi = dst + (uint32_t)!swapped;
    r.r0 = base + 2 * r.w;
    r.r1 = active ? base + 2 * ((x + 1) % 5 + 5 * y) : base + 50;
    r.r2 = active ? base + 2 * ((x + 2) % 5 + 5 * y) : base + 50;
    r.iota_mask = r.w == 0 ? 0xFFFFFFFFu : 0u;
    return r;
}

// acc ^ (v moved by a DPP row pattern)
template <int CTRL>
__device__ __forceinline__ uint32_t xor_into_dpp(uint32_t acc, uint32_t v) {
    return acc ^ (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, true);
}

__device__ __forceinline__ void keccak_round_wave(uint32_t &lo, uint32_t &hi, const WaveLane &r, uint32_t *lds,
                                                  uint32_t rc_lo, uint32_t rc_hi) {
    const auto a = __builtin_amdgcn_permlane32_swap(xor_dpp<DPP_ROW_ROR8>(lo), xor_dpp<DPP_ROW_ROR8>(hi), false, false);
    uint32_t s = a[0] ^ a[1];
    const auto b = __builtin_amdgcn_permlane16_swap(s, s, false, false);
    s = b[0] ^ b[1];
    const auto c = __builtin_amdgcn_permlane32_swap(s, s, false, false);
    const uint32_t cl = c[0], ch = c[1], rl = funnel(cl, ch, 31), rh = funnel(ch, cl, 31);
    lo = xor_into_dpp<DPP_ROW_ROR1>(lo, cl);
    hi = xor_into_dpp<DPP_ROW_ROR1>(hi, ch);
    asm("" : "+v"(lo), "+v"(hi));  // keeps the two updates apart: each is one DPP instruction
    lo = xor_into_dpp<DPP_ROW_SHL1>(lo, rl);
    hi = xor_into_dpp<DPP_ROW_SHL1>(hi, rh);
    lds[r.wlo] = funnel(lo, hi, r.sh);
    lds[r.whi] = funnel(hi, lo, r.sh);
    wave_lds_sync();
    const uint2 b0 = *reinterpret_cast<const uint2 *>(lds + r.r0), b1 = *reinterpret_cast<const uint2 *>(lds + r.r1),
                b2 = *reinterpret_cast<const uint2 *>(lds + r.r2);
    wave_lds_sync();  // reads done before the next round's writes
    lo = bitop3<kChi>(b0.x, b1.x, b2.x) ^ (rc_lo & r.iota_mask);
    hi = bitop3<kChi>(b0.y, b1.y, b2.y) ^ (rc_hi & r.iota_mask);
}

// unrolled as in the row form
template <int I = 0>
__device__ __forceinline__ void keccak_f1600_wave(uint32_t &lo, uint32_t &hi, const WaveLane &r, uint32_t *lds) {
    constexpr uint64_t rc = kKeccak.rc[I];
    keccak_round_wave(lo, hi, r, lds, (uint32_t)rc, (uint32_t)(rc >> 32));
    if constexpr (I + 1 < 24) keccak_f1600_wave<I + 1>(lo, hi, r, lds);
}

// shake_row for a wave: get_word(i) returns input word i (bytes past the end
// zero; only called for i < ceil(len / 8)); afterwards the lanes hold the
// words of the first output block.
template <int RATE, class GetWord>
__device__ __forceinline__ void shake_wave(uint32_t &lo, uint32_t &hi, const WaveLane &r, uint32_t *lds, uint32_t len,
                                           GetWord get_word) {
    constexpr uint32_t RW = RATE / 8;
    lo = hi = 0u;
    const uint32_t nwords = (len + 7) / 8, nfull = len / RATE;
    auto fetch = [&](uint32_t blk) -> uint64_t {
        const uint32_t i = blk * RW + r.w;
        return r.w < RW && i < nwords ? get_word(i) : 0ull;
    };
    uint64_t cur = fetch(0);
#pragma unroll 1
    for (uint32_t blk = 0; blk < nfull; ++blk) {
        lo ^= (uint32_t)cur;
        hi ^= (uint32_t)(cur >> 32);
        cur = fetch(blk + 1);  // overlaps the permutation
        keccak_f1600_wave(lo, hi, r, lds);
    }
    // last (partial) block and padding: 0x1F at byte rem, 0x80 at byte RATE - 1
    const uint32_t rem = len - nfull * RATE;
    if (r.w == rem / 8) cur ^= 0x1Full << (8 * (rem % 8));
    if (r.w == RW - 1) cur ^= 0x80ull << 56;
    lo ^= (uint32_t)cur;
    hi ^= (uint32_t)(cur >> 32);
    keccak_f1600_wave(lo, hi, r, lds);
}

// words [0, nwords) of the state to dst (4-byte aligned)
__device__ __forceinline__ void wave_store_words(uint32_t lo, uint32_t hi, const WaveLane &r, uint32_t *dst,
                                                 uint32_t nwords) {
    if (r.main && r.w < nwords) {
        dst[2 * r.w] = lo;
        dst[2 * r.w + 1] = hi;
    }
}

}  // namespace dil
