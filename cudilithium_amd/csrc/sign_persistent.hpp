// Persistent work-queue signing engine.
//
// Replaces the reference's host rejection scheduler (api.cu:208-441: one
// stream synchronisation and ~8 host<->device transfers per round) with one
// launch in which every workgroup loops until the batch is done:
//
//   refill   claim items from a global queue (one atomicAdd per refill) until
//            the workgroup owns `claim` (at most S) undone items or the queue
//            is empty
//   assign   S attempt slots round-robin over the owned items: item o gets
//            slots o, o + U, o + 2U, ... with consecutive nonces, so freed
//            slots turn into speculative nonces of unfinished items instead of
//            idling at the end of the batch
//   y w c    the first three attempt stages on the S slots (sign_stages.hpp),
//            with the lane mapping each stage wants, separated by barriers
//   z        one wave per item: its slots in slot order = nonce order; the
//            first that passes is the smallest successful nonce -- the
//            sequential specification's result -- and writes the signature
//            (z, h and c~ straight into the item's signature row)
//
// Workgroups never wait on each other (the queue is only read-modify-written
// by atomicAdd), so there is no co-residency requirement and no deadlock: a
// workgroup that starts after the queue has drained exits at once.  Every
// round gives each owned item at least one attempt, so each workgroup
// finishes with probability 1, as the reference's loop does.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>

#include "internal.hpp"
#include "sign_stages.hpp"

namespace dil {

// threads per workgroup (4 waves; a build may choose 2 with -DDIL_PERSIST_THREADS=128,
// then with 16 slots per workgroup so that the y stage's S * L sponges fit one pass)
#ifndef DIL_PERSIST_THREADS
#define DIL_PERSIST_THREADS 256
#endif
constexpr int PERSIST_THREADS = DIL_PERSIST_THREADS;
constexpr int PERSIST_MAX_IDLE_ROUNDS = 20000;  // of one workgroup, without a signature
// control words (uint32): 0 queue head, 1 status, 2 attempts executed.
// Optional phase profile: PERSIST_PHASES uint64 cycle sums (assign, y, w, c,
// z, commit) at a separate pointer, null when not profiling.
constexpr int PERSIST_PHASES = 6;
// wave priority (s_setprio) of the Keccak stages; 0 elsewhere.  Measured on
// 16384-item batches: +2-3 % signatures/s for Dilithium3 over no priority.
#ifndef DIL_KECCAK_PRIO
#define DIL_KECCAK_PRIO 2
#endif
constexpr int KECCAK_PRIO = DIL_KECCAK_PRIO;
// waves per SIMD the register allocation must allow (256 VGPRs).  Three or
// four (w unpaired, no spills) measured slower: 16,384 Dilithium3 items 2.85 /
// 3.05 against 2.82 ms.
constexpr int PERSIST_WPE = 2;

// claim: at most this many items owned per workgroup (1..S); below S every
// owned item gets at least S / claim slots (nonces) per round, which trades
// speculative attempts for fewer rounds on small batches
// the items are those left in the chain's list, claimed through its head
template <class P, int S>
__global__ __launch_bounds__(PERSIST_THREADS) __attribute__((amdgpu_waves_per_eu(PERSIST_WPE))) void
sg_persistent_kernel(SignArgs a, SlotRef sr, Chain chain, uint32_t *ctl, int claim, unsigned long long *phase_sums) {
    __shared__ ZetaLds zt;
    __shared__ int32_t x[PERSIST_THREADS / 64][NTT_XBUF];
    // L = 7: the paired w stage's transformed y vectors (56 KiB per workgroup,
    // which leaves room for two workgroups per CU)
    constexpr bool W_Y_LDS = P::L >= DIL_W_Y_LDS_MIN_L;
    union StageLds {
        int32_t y[W_Y_LDS ? 2 * P::L * N : 1];  // w stage
        ZScratch<P> z;                          // z stage
    };
    __shared__ StageLds stage_lds[PERSIST_THREADS / 64];
    __shared__ uint32_t own_item[S], own_next[S];
    __shared__ int own_done[S];
    __shared__ uint32_t slot_own[S], slot_nonce[S];
    __shared__ uint8_t w_unit[S];  // w work units: slot s, paired with s + u when s / u is even
    __shared__ int n_own, queue_empty, n_units, idle;
    const int tid = threadIdx.x, wave = tid >> 6, lane = lane_id();
    constexpr int NW = PERSIST_THREADS / 64;
    const size_t slot0 = (size_t)blockIdx.x * S;
    auto slot_base = [&](int s) { return sr.base + (slot0 + s) * sr.pitch; };
    auto slot_ct = [&](int s) { return slot_base(s) + SlotLayout<P>::CT; };  // c~ until the attempt passes
    zeta_lds_load(zt);
    if (tid == 0) {
        n_own = 0;
        queue_empty = 0;
        idle = 0;
    }
    __syncthreads();
    // optional phase profile: workgroup cycles per phase, summed over
    // workgroups; kept in LDS (only thread 0 uses it) so that it holds no
    // registers through the loop
    __shared__ unsigned long long tph[PERSIST_PHASES + 1];  // [PERSIST_PHASES]: last mark
    const bool prof = phase_sums != nullptr;
    if (prof && tid == 0) {
        for (int p = 0; p < PERSIST_PHASES; ++p) tph[p] = 0;
        tph[PERSIST_PHASES] = clock64();
    }
    auto mark = [&](int ph) {
        if (prof && tid == 0) {
            const unsigned long long t = clock64();
            tph[ph] += t - tph[PERSIST_PHASES];
            tph[PERSIST_PHASES] = t;
        }
    };

    for (;;) {
        if (tid == 0) {
            const int cap = claim > 0 && claim < S ? claim : S;
            int u = n_own;
            if (u < cap && !queue_empty) {
                ChainCtl *const cc = chain_ctl<P>(chain);
                const size_t end = cc->left;
                const uint32_t list = cc->cur;
                const uint32_t start = atomicAdd(&cc->head, (uint32_t)(cap - u));
                for (int j = 0; j < cap - u && (size_t)start + j < end; ++j) {
                    const uint2 e = *chain_entry(chain, list, start + j);
                    own_item[n_own] = e.x;
                    own_next[n_own] = e.y;
                    ++n_own;
                }
                if ((size_t)start + (cap - u) >= end) queue_empty = 1;
            }
            u = n_own;
            for (int s = 0; s < S && u > 0; ++s) {
                const int o = s % u;
                slot_own[s] = o;
                slot_nonce[s] = own_next[o] + s / u;
            }
            for (int o = 0; o < u; ++o) {
                own_next[o] += (S - o + u - 1) / u;
                own_done[o] = 0;
            }
            // slots s and s + u carry consecutive nonces of the same item: the
            // w stage takes them as one unit (one pass over that item's A)
            int nu = 0;
            for (int s = 0; s < S && u > 0; ++s)
                if ((s / u) % 2 == 0) w_unit[nu++] = (uint8_t)s;
            n_units = nu;
        }
        __syncthreads();
        mark(0);
        const int u = n_own;
        if (u == 0) break;
        if (idle == PERSIST_MAX_IDLE_ROUNDS) {
            // no correct run gets here (each round succeeds per item with
            // probability >= 1/5); stop instead of spinning and report it
            if (tid == 0) atomicOr(ctl + 1, SIGN_STATUS_ROUND_CAP);
            break;
        }
        if (tid == 0) atomicAdd(ctl + 2, (uint32_t)S);  // attempts executed (incl. speculative)

        // the Keccak stages (y, c) run few serial permutation chains that the
        // whole workgroup then waits for; their waves get issue priority over
        // the transform stages of other workgroups on the same SIMDs
        __builtin_amdgcn_s_setprio(KECCAK_PRIO);
        // When the S * L sponges fit two lanes each, the pair form's shorter
        // chain (Dilithium2 16,384 items 2.41 -> 2.28 ms per batch; 16 slots per
        // workgroup: Dilithium3 / 5 4,096 items 1.79 / 1.73 -> 1.67 / 1.67 ms)
#ifndef DIL_Y_PAIR
#define DIL_Y_PAIR 1
#endif
        if constexpr (DIL_Y_PAIR && 2 * S * P::L <= PERSIST_THREADS) {
            if (tid < 2 * S * P::L) {
                const int q = tid >> 1, s = q / P::L;
                stage_y_pair<P>(a, own_item[slot_own[s]], slot_nonce[s], q % P::L, slot_base(s), tid & 1);
            }
        } else {
            for (int t = tid; t < S * P::L; t += PERSIST_THREADS) {
                const int s = t / P::L;
                stage_y<P>(a, own_item[slot_own[s]], slot_nonce[s], t % P::L, slot_base(s));
            }
        }
        __builtin_amdgcn_s_setprio(0);
        __syncthreads();
        mark(1);
        for (int t = wave; t < n_units; t += NW) {
            const int s = w_unit[t];
            const size_t item = own_item[slot_own[s]];
            if (s + u < S) {
                uint8_t *const pair[2] = {slot_base(s), slot_base(s + u)};
                stage_w_multi<P, 2>(a, item, pair, x[wave], zt, stage_lds[wave].y);
                continue;
            }
            stage_w<P>(a, item, slot_base(s), x[wave], zt);
        }
        __syncthreads();
        mark(2);
        __builtin_amdgcn_s_setprio(KECCAK_PRIO);
        // two lanes per slot (keccak_f1600_pair): S slots on 2 S lanes
        for (int t = tid; t < 2 * S; t += PERSIST_THREADS) {
            const int s = t >> 1;
            stage_c_pair<P>(a, own_item[slot_own[s]], slot_base(s), slot_ct(s), (uint32_t)(t & 1));
        }
        __builtin_amdgcn_s_setprio(0);
        __syncthreads();
        mark(3);
        // z and commit, one wave per owned item: its slots o, o + u, ... carry
        // increasing nonces, so they are checked in that order and the first
        // that passes -- the sequential specification's result -- ends the
        // item; later (speculative) slots of the item are skipped.  An attempt
        // writes z and h straight into the item's signature; a rejected one
        // leaves them partly written, and the accepted attempt rewrites every
        // byte (c~ is copied from the slot where the c stage put it).
        for (int o = wave; o < u; o += NW) {
            const size_t item = own_item[o];
            uint8_t *dst = a.sig + item * a.sig_pitch;
            for (int s = o; s < S; s += u) {
                if (stage_z<P>(a, item, slot_base(s), dst, stage_lds[wave].z)) {
                    const uint8_t *src = slot_ct(s);
                    if (lane < SEEDBYTES) dst[lane] = src[lane];
                    if (lane == 0) {
                        own_done[o] = 1;
                        // attempts the sequential specification makes for this item
                        *reinterpret_cast<uint32_t *>(a.rows + item * a.row_pitch + SignLayout<P>::ATTEMPTS) =
                            slot_nonce[s] + 1;
                    }
                    break;
                }
            }
        }
        __syncthreads();
        mark(4);
        if (tid == 0) {
            int k = 0;
            for (int o = 0; o < u; ++o)
                if (!own_done[o]) {
                    own_item[k] = own_item[o];
                    own_next[k] = own_next[o];
                    ++k;
                }
            idle = k < u ? 0 : idle + 1;
            n_own = k;
        }
        __syncthreads();
        mark(5);
    }
    if (prof && tid == 0) {
        for (int p = 0; p < PERSIST_PHASES; ++p) atomicAdd(phase_sums + p, tph[p]);
    }
}

// clears the control words (and the phase sums when given); a kernel rather
// than a memset so that the sequence can be captured in a HIP graph
__global__ void zero_ctl_kernel(uint32_t *p, unsigned long long *phase_sums);

template <class P, int S>
static int launch_persistent_s(const SignArgs &a, const SlotRef &sr, const Chain &chain, size_t nslots, int blocks,
                               int claim, uint32_t *ctl, unsigned long long *phase_sums, hipStream_t st) {
    int nb = (int)(nslots / S);
    if (blocks > 0 && blocks < nb) nb = blocks;
    if (nb < 1) return -3;
    hipLaunchKernelGGL((sg_persistent_kernel<P, S>), dim3(nb), dim3(PERSIST_THREADS), 0, st, a, sr, chain, ctl,
                       claim & 0xFFFF, phase_sums);
    return (int)hipGetLastError();
}

// Defined once per mode (sign_persistent_<mode>.hip).
template <class P>
int launch_persistent_p(const SignArgs &a, const SlotRef &sr, const Chain &chain, size_t nslots, int slots_per_block,
                        int blocks, int claim, uint32_t *ctl, unsigned long long *phase_sums, hipStream_t st);

#define DIL_DEFINE_PERSISTENT_LAUNCHER(MODE)                                                                       \
    template <>                                                                                                  \
    int launch_persistent_p<Params<MODE>>(const SignArgs &a, const SlotRef &sr, const Chain &chain, size_t nslots, \
                                          int slots_per_block, int blocks, int claim, uint32_t *ctl,             \
                                          unsigned long long *ph, hipStream_t st) {                              \
        using P = Params<MODE>;                                                                                  \
        switch (slots_per_block) {                                                                               \
            case 1: return launch_persistent_s<P, 1>(a, sr, chain, nslots, blocks, claim, ctl, ph, st);          \
            case 8: return launch_persistent_s<P, 8>(a, sr, chain, nslots, blocks, claim, ctl, ph, st);          \
            case 16: return launch_persistent_s<P, 16>(a, sr, chain, nslots, blocks, claim, ctl, ph, st);        \
            case 32: return launch_persistent_s<P, 32>(a, sr, chain, nslots, blocks, claim, ctl, ph, st);        \
            default: return -1;                                                                                  \
        }                                                                                                        \
    }

}  // namespace dil
