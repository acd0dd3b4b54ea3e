// Hashes with one sponge per 16-lane row or per wavefront, for the launches
// whose chains of permutations are longer than the card's work beside them:
// mu / rhoprime, the mask sponges and the challenges.
#pragma once

#include <hip/hip_runtime.h>

#include "keccak_row.hpp"
#include "keccak_wave.hpp"
#include "sign_stages.hpp"

namespace dil {

constexpr int ROW_ITEMS_PER_BLOCK = 16;

// a[x] holds half r.h of output word x + 5 y: lanes with word < nwords
// store their half to dst (32-bit stores; dst 4-byte aligned)
__device__ __forceinline__ void row_store_words(const uint32_t (&a)[5], const RowLane &r, uint32_t *dst,
                                                uint32_t nwords) {
#pragma unroll
    for (int x = 0; x < 5; ++x) {
        const uint32_t w = row_word(r, x);
        if (r.active && w < nwords) dst[2 * w + r.h] = a[x];
    }
}

// shares output words [0, nwords) of the group through LDS (the state's pi
// area, free after the permutation): returns half h of word w
struct RowShare {
    uint32_t base;
    __device__ void put(uint32_t *lds, const uint32_t (&a)[5], const RowLane &r, uint32_t nwords) const {
#pragma unroll
        for (int x = 0; x < 5; ++x) {
            const uint32_t w = row_word(r, x);
            if (r.active && w < nwords) lds[base + 2 * w + r.h] = a[x];
        }
    }
    __device__ uint32_t get(const uint32_t *lds, uint32_t w, uint32_t h) const { return lds[base + 2 * w + h]; }
};

// mu = SHAKE256(tr || m) and rhoprime = SHAKE256(key || mu) (or the caller's
// rhoprime) of item i, by the 16 lanes of a row; lds as for row_lane_setup.
template <class P>
__device__ __forceinline__ void stage_mu_row(const SignArgs &a, size_t i, const RowLane &r, uint32_t *lds,
                                             uint32_t wave) {
    using Z = Sizes<P>;
    using SLy = SignLayout<P>;
    const uint8_t *sk = a.sk + sk_index(a, i) * a.sk_pitch;
    const uint8_t *m = a.m.ptr(i);
    const uint32_t mlen = a.m.len(i);
    const uint32_t h = r.h;
    uint32_t s[5];
    // mu = SHAKE256(tr || m)
    shake_row<SHAKE256_RATE>(s, r, lds, SEEDBYTES + mlen, [&](uint32_t w) -> uint32_t {
        if (w < 4) return load_half_bytes(sk + Z::SK_TR, 8 * w + 4 * h, SEEDBYTES);
        return load_half_bytes(m, 8 * (w - 4) + 4 * h, mlen);
    });
    uint8_t *row = a.rows + i * a.row_pitch;
    row_store_words(s, r, reinterpret_cast<uint32_t *>(row + SLy::MU), 8);
    if (a.rnd) {
        const uint8_t *rnd = a.rnd + i * a.rnd_pitch;
        const uint32_t g = (uint32_t)lane_id() & 15;  // 16 lanes x 4 bytes
        reinterpret_cast<uint32_t *>(row + SLy::RHOPRIME)[g] = load_half_bytes(rnd, 4 * g, CRHBYTES);
        return;
    }
    // rhoprime = SHAKE256(key || mu): mu's words cross rows, through LDS
    const RowShare sh{wave * 4 * ROW_LDS_WORDS + ((uint32_t)lane_id() >> 4) * ROW_LDS_WORDS};
    sh.put(lds, s, r, 8);
    wave_lds_sync();
    uint32_t t[5];
    shake_row<SHAKE256_RATE>(t, r, lds, SEEDBYTES + CRHBYTES, [&](uint32_t w) -> uint32_t {
        if (w < 4) return load_half_bytes(sk + Z::SK_KEY, 8 * w + 4 * h, SEEDBYTES);
        return sh.get(lds, w - 4, h);
    });
    row_store_words(t, r, reinterpret_cast<uint32_t *>(row + SLy::RHOPRIME), 8);
}

// LDS words per row of challenge_row: the block, the accepted positions, the
// masks; 4 words of padding.
constexpr int CHALLENGE_ROW_WORDS = 2 * (SHAKE256_RATE / 8) + 16 + 16 + 6;

// SampleInBall from the state a (c~ absorbed, not yet permuted) by the 16
// lanes of a row; masks: nz[8] | neg[8] as challenge() stores them.
//
// The step (c[i] = c[b]; c[b] = +-1) moves whatever was placed at b earlier to
// i, so the place of the j-th sign follows from the accepted bytes alone: it
// starts at b_j, and every later step whose byte equals its place moves it.
// Each lane follows four signs through all steps, which takes about 8
// instructions per step instead of the 45 of one lane updating bit masks.
template <int TAU>
__device__ __forceinline__ void challenge_row(uint32_t (&a)[5], uint32_t *masks, const RowLane &r, uint32_t *lds,
                                              uint32_t *my, bool run) {
    static_assert(TAU <= 64, "four signs per lane");
    constexpr int BLOCK = 2 * (SHAKE256_RATE / 8);
    const uint32_t g = (uint32_t)lane_id() & 15;
    uint32_t *list = my + BLOCK, *mk = list + 16;
    uint8_t *lb = reinterpret_cast<uint8_t *>(list);
    uint32_t n = 0, sign0 = 0, sign1 = 0;
    for (uint32_t start = 2;; start = 0) {
        keccak_f1600_row(a, r, lds);
#pragma unroll
        for (int x = 0; x < 5; ++x) {
            const uint32_t w = row_word(r, x);
            if (r.active && w < SHAKE256_RATE / 8) my[2 * w + r.h] = a[x];
        }
        wave_lds_sync();
        if (start) {
            sign0 = my[0];
            sign1 = my[1];
        }
        // the accepted bytes: b <= i, i = N - TAU + n; every lane of the row
        // runs the same steps, lane 0 writes
        for (uint32_t k = start; k < BLOCK && n < TAU; ++k) {
            uint32_t v = my[k];
#pragma unroll
            for (int b = 0; b < 4; ++b, v >>= 8) {
                const uint32_t byte = v & 0xFFu;
                if (byte <= N - TAU + n && n < TAU) {
                    if (g == 0) lb[n] = (uint8_t)byte;
                    ++n;
                }
            }
        }
        if (__ballot(n < TAU) == 0ull) break;
        wave_lds_sync();  // the block is read before the next one overwrites it
    }
    mk[g] = 0u;
    wave_lds_sync();
    uint32_t pos[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) pos[q] = 0xFFFFu;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
#pragma unroll 4
        for (int t = 0; t < 16; ++t) {
            const int j = 16 * q + t;
            if (j >= TAU) break;
            const uint32_t b = lb[j];
#pragma unroll
            for (int p = 0; p <= q; ++p) pos[p] = pos[p] == b ? (uint32_t)(N - TAU + j) : pos[p];
            pos[q] = g == (uint32_t)t ? b : pos[q];
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const uint32_t j = 16 * q + g;
        if (j < TAU) {
            const uint32_t bit = 1u << (pos[q] & 31), neg = ((j < 32 ? sign0 : sign1) >> (j & 31)) & 1u;
            atomicOr(&mk[pos[q] >> 5], bit);
            if (neg) atomicOr(&mk[8 + (pos[q] >> 5)], bit);
        }
    }
    wave_lds_sync();
    if (run) masks[g] = mk[g];
}

// stage_c by the 16 lanes of a row
template <class P>
__device__ __forceinline__ void stage_c_row(const uint32_t *mu, const uint32_t *w1, uint32_t *ct, uint32_t *masks,
                                            const RowLane &r, uint32_t *lds, uint32_t *my, bool run) {
    uint32_t a[5];
    shake_row<SHAKE256_RATE>(a, r, lds, Sizes<P>::CHASH_IN_BYTES, [&](uint32_t w) -> uint32_t {
        return !run ? 0u : (w < 8 ? mu[2 * w + r.h] : w1[2 * (w - 8) + r.h]);
    });
    if (run) row_store_words(a, r, ct, SEEDBYTES / 8);
    // c~ is words 0..3, held by the y = 0 lanes: 32 input bytes, the domain
    // byte at byte 32, the final bit in the high half of word 16
#pragma unroll
    for (int x = 0; x < 5; ++x) {
        const uint32_t w = row_word(r, x);
        a[x] = r.active && w < 4 ? a[x] : 0u;
        if (r.active && w == 4 && r.h == 0) a[x] = 0x1Fu;
        if (r.active && w == SHAKE256_RATE / 8 - 1 && r.h == 1) a[x] = 0x80000000u;
    }
    challenge_row<P::TAU>(a, masks, r, lds, my, run);
}

// ------------------------------------------------- one sponge per wavefront

// 8 bytes at off of a buffer of len bytes (bytes past the end zero)
__device__ __forceinline__ uint64_t load_word_bytes(const uint8_t *p, uint32_t off, uint32_t len) {
    if (off + 8 <= len) return load_any<uint64_t>(p + off);
    uint64_t v = 0;
    for (uint32_t b = 0; off + b < len; ++b) v |= (uint64_t)p[off + b] << (8 * b);
    return v;
}

// stage_mu_row by a wave; lds: its WAVE_LDS_WORDS words at base
template <class P>
__device__ __forceinline__ void stage_mu_wave(const SignArgs &a, size_t i, const WaveLane &r, uint32_t *lds,
                                              uint32_t base) {
    using Z = Sizes<P>;
    using SLy = SignLayout<P>;
    const uint8_t *sk = a.sk + sk_index(a, i) * a.sk_pitch;
    const uint8_t *m = a.m.ptr(i);
    const uint32_t mlen = a.m.len(i);
    uint32_t lo, hi;
    shake_wave<SHAKE256_RATE>(lo, hi, r, lds, SEEDBYTES + mlen, [&](uint32_t w) -> uint64_t {
        return w < 4 ? load_word_bytes(sk + Z::SK_TR, 8 * w, SEEDBYTES) : load_word_bytes(m, 8 * (w - 4), mlen);
    });
    uint8_t *row = a.rows + i * a.row_pitch;
    wave_store_words(lo, hi, r, reinterpret_cast<uint32_t *>(row + SLy::MU), 8);
    uint32_t *rhoprime = reinterpret_cast<uint32_t *>(row + SLy::RHOPRIME);
    if (a.rnd) {
        const uint32_t g = (uint32_t)lane_id();
        if (g < CRHBYTES / 4) rhoprime[g] = load_half_bytes(a.rnd + i * a.rnd_pitch, 4 * g, CRHBYTES);
        return;
    }
    // rhoprime = SHAKE256(key || mu): mu's words change lanes through LDS (the
    // area of the pi exchange, free after the permutation)
    wave_store_words(lo, hi, r, lds + base, 8);
    wave_lds_sync();
    shake_wave<SHAKE256_RATE>(lo, hi, r, lds, SEEDBYTES + CRHBYTES, [&](uint32_t w) -> uint64_t {
        return w < 4 ? load_word_bytes(sk + Z::SK_KEY, 8 * w, SEEDBYTES)
                     : *reinterpret_cast<const uint64_t *>(lds + base + 2 * (w - 4));
    });
    wave_store_words(lo, hi, r, rhoprime, 8);
}

// mask_raw by a wave: 5 squeezed SHAKE256 blocks of rhoprime || le16(nonce)
__device__ __forceinline__ void mask_raw_wave(const uint32_t *rhoprime, uint32_t nonce, uint32_t *out,
                                              const WaveLane &r, uint32_t *lds) {
    // 66 input bytes: le16(nonce) and the domain byte 0x1F in word 8, the final
    // bit in word 16
    uint32_t lo = r.w < 8 ? rhoprime[2 * r.w] : 0u, hi = r.w < 8 ? rhoprime[2 * r.w + 1] : 0u;
    if (r.w == 8) lo = (nonce & 0xFFFFu) | (0x1Fu << 16);
    if (r.w == SHAKE256_RATE / 8 - 1) hi = 0x80000000u;
#pragma unroll 1
    for (int b = 0; b < 5; ++b) {
        keccak_f1600_wave(lo, hi, r, lds);
        wave_store_words(lo, hi, r, out + 2 * 17 * b, SHAKE256_RATE / 8);
    }
}

// challenge_row by a wave, each lane following one sign; my: as for a row
template <int TAU>
__device__ __forceinline__ void challenge_wave(uint32_t lo, uint32_t hi, uint32_t *masks, const WaveLane &r,
                                               uint32_t *lds, uint32_t *my) {
    static_assert(TAU <= 64, "a sign per lane");
    constexpr uint32_t BLOCK = 2 * (SHAKE256_RATE / 8);
    const uint32_t lane = (uint32_t)lane_id();
    uint32_t *list = my + BLOCK, *mk = list + 16;
    uint8_t *lb = reinterpret_cast<uint8_t *>(list);
    uint32_t n = 0, sign0 = 0, sign1 = 0;
    for (uint32_t start = 2; n < TAU; start = 0) {
        keccak_f1600_wave(lo, hi, r, lds);
        wave_store_words(lo, hi, r, my, SHAKE256_RATE / 8);
        wave_lds_sync();
        if (start) {
            sign0 = my[0];
            sign1 = my[1];
        }
        for (uint32_t k = start; k < BLOCK && n < TAU; ++k) {
            uint32_t v = my[k];
#pragma unroll
            for (int b = 0; b < 4; ++b, v >>= 8) {
                const uint32_t byte = v & 0xFFu;
                if (byte <= N - TAU + n && n < TAU) {
                    if (lane == 0) lb[n] = (uint8_t)byte;
                    ++n;
                }
            }
        }
        wave_lds_sync();  // the block is read before the next one overwrites it
    }
    if (lane < 16) mk[lane] = 0u;
    wave_lds_sync();
    uint32_t pos = 0xFFFFu;
#pragma unroll 8
    for (int j = 0; j < TAU; ++j) {
        const uint32_t b = lb[j];
        pos = pos == b ? (uint32_t)(N - TAU + j) : pos;
        pos = lane == (uint32_t)j ? b : pos;
    }
    if (lane < TAU) {
        const uint32_t bit = 1u << (pos & 31), neg = ((lane < 32 ? sign0 : sign1) >> (lane & 31)) & 1u;
        atomicOr(&mk[pos >> 5], bit);
        if (neg) atomicOr(&mk[8 + (pos >> 5)], bit);
    }
    wave_lds_sync();
    if (lane < 16) masks[lane] = mk[lane];
}

// stage_c by a wave
template <class P>
__device__ __forceinline__ void stage_c_wave(const uint32_t *mu, const uint32_t *w1, uint32_t *ct, uint32_t *masks,
                                             const WaveLane &r, uint32_t *lds, uint32_t *my) {
    uint32_t lo, hi;
    shake_wave<SHAKE256_RATE>(lo, hi, r, lds, Sizes<P>::CHASH_IN_BYTES, [&](uint32_t w) -> uint64_t {
        const uint32_t *src = w < 8 ? mu + 2 * w : w1 + 2 * (w - 8);
        return src[0] | (uint64_t)src[1] << 32;
    });
    wave_store_words(lo, hi, r, ct, SEEDBYTES / 8);
    lo = r.w < 4 ? lo : (r.w == 4 ? 0x1Fu : 0u);
    hi = r.w < 4 ? hi : (r.w == SHAKE256_RATE / 8 - 1 ? 0x80000000u : 0u);
    challenge_wave<P::TAU>(lo, hi, masks, r, lds, my);
}

// LDS words of expand_a_wave's block: 42 and one that the last candidates'
// second word reads
constexpr int EXPAND_WAVE_WORDS = 2 * (SHAKE128_RATE / 8) + 2;

// One polynomial of ExpandA by a wave: a[N] from rho (32 bytes) and
// nonce = k << 8 | l.  The 56 candidates of a block are tested at once, one
// per lane; an accepted one's place is the number accepted before it.
__device__ __forceinline__ void expand_a_wave(int32_t *a, const uint8_t *rho, uint32_t nonce, const WaveLane &r,
                                              uint32_t *lds, uint32_t *block) {
    constexpr uint32_t CAND = SHAKE128_RATE / 3;
    const uint32_t lane = (uint32_t)lane_id(), byte = 3 * lane;
    const uint64_t seed = r.w < 4 ? load_any<uint64_t>(rho + 8 * r.w) : 0ull;
    uint32_t lo = (uint32_t)seed, hi = (uint32_t)(seed >> 32);
    if (r.w == 4) lo = (nonce & 0xFFFFu) | (0x1Fu << 16);
    if (r.w == SHAKE128_RATE / 8 - 1) hi = 0x80000000u;
    for (uint32_t n = 0; n < N;) {
        keccak_f1600_wave(lo, hi, r, lds);
        wave_store_words(lo, hi, r, block, SHAKE128_RATE / 8);
        wave_lds_sync();
        uint32_t t = Q;
        if (lane < CAND) {
            const uint32_t *q = block + (byte >> 2);
            t = __builtin_amdgcn_alignbyte(q[1], q[0], byte & 3) & 0x7FFFFFu;
        }
        const bool ok = t < (uint32_t)Q;
        const uint64_t mask = __ballot(ok);
        const uint32_t at = n + __popcll(mask & ((1ull << lane) - 1ull));
        if (ok && at < N) a[at] = (int32_t)t;
        n += __popcll(mask);
        wave_lds_sync();  // the block is read before the next one overwrites it
    }
}

}  // namespace dil
