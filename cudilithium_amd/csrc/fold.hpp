// ExpandA folded into a matrix-vector product: one wave computes A v^ for the
// K rows of IPW items without storing A.
//
// Lane (item, k, l) runs the sponge of entry A[k][l] and folds each accepted
// coefficient a into sum[k][ctr] += mont(a, v^[l][ctr]) with an LDS atomic; the
// int32 sums are exact, so their order does not matter.  A block of 168 bytes
// holds 56 candidates, of which 0.1 % are rejected, so all lanes of a wave walk
// the coefficients nearly in step and only a window of them is live: the sums
// of WIN = 60 coefficients per row sit in LDS, and when every lane is past the
// window's first 56 they are final and replace the entries of v^ that no lane
// reads any more.  One item thus takes K rows of 1 KiB and K windows of 240
// bytes (instead of K + L full rows), which decides how many waves a CU holds.
//
// Bound by VALU issue (Keccak three quarters of it).  65,536 Dilithium5
// verifications 4.80 -> 3.26 ms (the form with full rows and a workgroup per
// item group spent its time on LDS bank conflicts, on barriers and on the half
// of its lanes without a sponge), 16,384 Dilithium3 keys 0.975 -> 0.777 ms.
//
// A lane that meets more than 4 rejections in the first 56 (b + 1) candidates
// falls behind the window (about one wave in 5,000); the wave then goes on in
// a form in which every lane squeezes and pauses on its own.
#pragma once

#include <hip/hip_runtime.h>

#include "field.hpp"
#include "ntt.hpp"
#include "params.hpp"
#include "poly.hpp"
#include "sample.hpp"

namespace dil {

template <class P>
struct FoldCfg {
    // items per wave: their K * L sponges fill 64, 60 and 56 of 64 lanes
    static constexpr int IPW = P::MODE == 2 ? 4 : (P::MODE == 3 ? 2 : 1);
    static_assert(IPW * P::K * P::L <= 64 && P::K >= P::L, "one sponge per lane, sums replace v^");
};

constexpr int FOLD_CAND = SHAKE128_RATE / 3;  // 56 candidates per block
constexpr int FOLD_SLACK = 4;                 // rejections a window allows for
constexpr int FOLD_WIN = FOLD_CAND + FOLD_SLACK;

// rows 16-byte aligned; LDS_ROW and FOLD_WIN spread 16 rows over the banks
template <class P>
struct FoldLds {
    int32_t row[FoldCfg<P>::IPW * P::K][LDS_ROW];
    int32_t win[FoldCfg<P>::IPW * P::K][FOLD_WIN];
};

// One block's candidates from number `ci` on into sink(t) while ctr < limit.
// FREE: all 56, no limit (the caller knows that they fit).
template <bool FREE, class Sink>
__device__ __forceinline__ void fold_block(const Lane64 (&s)[25], int &ctr, int &ci, int limit, Sink &&sink) {
    static_for<0, FOLD_CAND / 8>([&](auto g) {
        if (!FREE && __ballot(ctr < limit) == 0ull) return;
        static_for<0, 8>([&](auto c) {
            constexpr int C = 8 * decltype(g)::value + decltype(c)::value;
            const uint32_t t = block_bits<24 * C, 23>(s);
            if constexpr (FREE) {
                if (t < (uint32_t)Q) {
                    sink(ctr, (int32_t)t);
                    ++ctr;
                }
            } else {
                if (C >= ci && ctr < limit) {
                    ci = C + 1;
                    if (t < (uint32_t)Q) {
                        sink(ctr, (int32_t)t);
                        ++ctr;
                    }
                }
            }
        });
    });
}

// On entry f.row[i * K + l] = v^ of item i (layout D order, l < L); on exit
// f.row[i * K + k] = sum over l of mont(A[k][l], v^[l]).  Lane (i, k, l) =
// lane i * K * L + k * L + l passes its item's rho; `run` is false for lanes
// without an item and for items to skip.
template <class P>
__device__ __forceinline__ void expand_fold(FoldLds<P> &f, const uint64_t (&rho)[4], bool run) {
    constexpr int KL = P::K * P::L, ROWS = FoldCfg<P>::IPW * P::K;
    const int lane = lane_id();
    const int i = min(lane / KL, FoldCfg<P>::IPW - 1), k = lane % KL / P::L, l = lane % P::L;
    wave_lds_sync();  // the transforms that used the windows as their exchange buffer are through
    for (int j = lane; j < ROWS * (FOLD_WIN / 4); j += 64)
        reinterpret_cast<int4 *>(f.win)[j] = make_int4(0, 0, 0, 0);
    Lane64 s[25];
    const uint64_t in[5] = {rho[0], rho[1], rho[2], rho[3], (uint64_t)(k << 8 | l)};
    shake_absorb_regs<SHAKE128_RATE, SEEDBYTES + 2>(s, in);
    const int32_t *v = f.row[i * P::K + l];
    int32_t *win = f.win[i * P::K + k];
    int ctr = run ? 0 : N, ci = FOLD_CAND;
    int base = 0;  // first coefficient of the window
    wave_lds_sync();
    auto sink = [&](int c, int32_t t) { atomicAdd(&win[c - base], mont_reduce((int64_t)t * v[c])); };
    // the window's first `step` sums are final: into the rows; the rest becomes
    // the start of the next window, `step` coefficients on
    auto advance = [&](int step) {
        wave_lds_sync();
        const int q = lane - base / 4;  // this lane's coefficients 4 lane .. + 3 in the window
        if (q >= 0 && q < step / 4) {
#pragma unroll
            for (int r = 0; r < ROWS; ++r)
                reinterpret_cast<int4 *>(f.row[r])[lane] = reinterpret_cast<const int4 *>(f.win[r])[q];
        }
        // (every lane's load before any lane's store, four rows at a time)
        const int from = lane + step / 4;
        const bool keep = from < FOLD_WIN / 4;
#pragma unroll
        for (int r0 = 0; r0 < ROWS; r0 += 4) {
            int4 old[4];
#pragma unroll
            for (int r = r0; r < min(r0 + 4, ROWS); ++r)
                old[r - r0] = reinterpret_cast<const int4 *>(f.win[r])[keep ? from : 0];
            wave_lds_sync();
            if (lane < FOLD_WIN / 4) {
#pragma unroll
                for (int r = r0; r < min(r0 + 4, ROWS); ++r)
                    reinterpret_cast<int4 *>(f.win[r])[lane] = keep ? old[r - r0] : make_int4(0, 0, 0, 0);
            }
        }
        wave_lds_sync();
        base += step;
    };
    bool own_pace = false;
#pragma unroll 1
    for (int b = 0; b < 5; ++b) {
        const bool last = b == 4;
        const int target = last ? N : FOLD_CAND * (b + 1) - FOLD_SLACK;
        if (!own_pace && !last) {
            if (run) {
                keccak_f1600(s);
                fold_block<true>(s, ctr, ci, 0, sink);
            }
            own_pace = __ballot(ctr < target) != 0ull;
        }
        if (own_pace || last) {
            const int limit = min(base + FOLD_WIN, N);
            while (__ballot(ctr < target)) {
                if (ctr < target) {
                    if (ci == FOLD_CAND) {
                        keccak_f1600(s);
                        ci = 0;
                    }
                    fold_block<false>(s, ctr, ci, limit, sink);
                }
            }
        }
        advance(b == 0 ? FOLD_CAND - FOLD_SLACK : last ? FOLD_WIN : FOLD_CAND);
    }
}

}  // namespace dil
