// Signing in rounds over the whole card, driven by the device.
//
// The rejection loop's stages want very different launches: the mask and
// challenge hashes are serial permutation chains that need many waves with
// few registers, w and z are wave-per-attempt transforms and matrix products.
// In one persistent kernel (sign_persistent.hpp) they share 256 registers,
// two waves per SIMD and a barrier per stage, and the loop issues vector
// instructions less than half of its time.  Here every stage is a launch of
// its own over all attempts of a round:
//
//   fixed  mu / rhoprime, ExpandA and the int8 secret key, one launch whose
//          workgroups take one of the three roles
//   y      lane (or lane pair) per mask sponge
//   w      wave per attempt
//   c      lane pair per attempt
//   z      wave per attempt; the first in nonce order that passes is the
//          specification's signature of its item
//   plan   one workgroup lists the items without a signature and plans the
//          next round (how many items, how many consecutive nonces for each),
//          so the host issues a fixed sequence of launches and never waits.
//          (A shared queue that z pushes to with atomics was slower: some
//          thousand atomics on one address from eight XCDs' L2 caches take
//          about 50 ns each, 430 us per round of 16,384 attempts.)
//
// The sequence is as long as the expected decay of the batch needs; what is
// left after it (rarely anything) is finished by the persistent kernel, which
// takes its items from the same queue.  Large batches run as two chains of
// rounds on two streams, so that the hash launches of one fill the SIMDs that
// the other leaves idle.
//
// The reference issues its rounds from the host with a synchronisation and
// about eight small copies per round (api.cu:208-441).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "hash_row.hpp"
#include "internal.hpp"
#include "sign_stages.hpp"

namespace dil {

constexpr int ROUND_WAVES = 4;
constexpr uint32_t ROUND_MAX_M = 32;  // attempts per item and round
// Messages hashed with a 16-lane row each up to this batch: beyond, the rows'
// fourfold instruction count costs ExpandA beside them more than the shorter
// chain gives (3,001 Dilithium5 items with messages up to 4 KiB: fixed stage
// 394 us with lane pairs, 174 us with rows).
constexpr uint32_t FIXED_ROW_MAX = 4096;
// Larger batches go to the persistent kernel, whose workgroups need no
// launches between stages: 10,000 Dilithium2 items (drop-in) 2.79 ms in
// rounds, 2.82 ms persistent; 16,384 Dilithium3 items 3.14 and 2.82 ms; 3,001
// Dilithium5 items 1.18 and 1.43 ms; 1,000 Dilithium2 items 0.44 and 0.81 ms;
// 17 Dilithium3 items 0.30 and 0.79 ms.
constexpr size_t ROUNDS_MAX_ITEMS = 4096;
// Attempts a round aims at when few items are left, and the least per item (a
// second attempt reads the item's A from L2).
constexpr size_t ROUND_TARGET = 8192;
constexpr uint32_t ROUND_MIN_M = 2;

// items and attempts per item of a round over u waiting items
__host__ __device__ inline void plan_round(uint32_t u, uint32_t nslots, uint32_t target, uint32_t &count,
                                           uint32_t &m) {
    m = u ? target / u : 0;
    m = m < ROUND_MIN_M ? ROUND_MIN_M : (m > ROUND_MAX_M ? ROUND_MAX_M : m);
    m = m > nslots ? nslots : m;
    count = nslots / m;
    count = count < u ? count : u;
}

// ------------------------------------------------------------------ kernels

struct FixedGrid {
    uint32_t mu, expand, prep;  // workgroups of each role
};

template <class P, bool ROW>
__global__ __launch_bounds__(256) void sg_fixed_kernel(SignArgs a, Chain ch, FixedGrid g) {
    constexpr int KL = P::K * P::L, PREP = (P::L + 2 * P::K) * (N / 8);
    __shared__ uint32_t lds[ROW ? 4 * 4 * ROW_LDS_WORDS : 1];
    uint32_t b = blockIdx.x;
    if (b < g.mu) {
        // serial chains, which end the stage: highest issue priority
        __builtin_amdgcn_s_setprio(3);
        const uint32_t t = threadIdx.x;
        const uint32_t i = ROW ? b * ROW_ITEMS_PER_BLOCK + (t >> 4) : b * 128 + (t >> 1);
        RowLane r;
        if constexpr (ROW) r = row_lane_setup(lds, (t >> 6) * 4 * ROW_LDS_WORDS);
        if (i >= ch.n) return;  // whole rows / pairs of lanes
        if ((t & (ROW ? 15 : 1)) == 0) {
            if (ch.lists) *chain_entry(ch, 0, i) = make_uint2(ch.first + i, 0);
            if (ch.lists && i == 0) {
                ChainCtl c{ch.n, 0, 0, 0, 0};
                plan_round(ch.n, ch.nslots, ch.target, c.count, c.m);
                *chain_ctl<P>(ch) = c;
            }
        }
        if constexpr (ROW)
            stage_mu_row<P>(a, ch.first + i, r, lds, t >> 6);
        else
            stage_mu_pair<P>(a, ch.first + i, t & 1);
        return;
    }
    b -= g.mu;
    if (b < g.expand) {
        const size_t t = (size_t)b * 256 + threadIdx.x;
        if (t >= (size_t)ch.n * KL) return;
        const int e = (int)(t % KL);
        stage_expand_a<P>(a, ch.first + t / KL, e / P::L, e % P::L);
        return;
    }
    const size_t t = (size_t)(b - g.expand) * 256 + threadIdx.x;
    if (t >= (size_t)ch.n * PREP) return;
    const size_t i = ch.first + t / PREP;
    const int u = (int)(t % PREP);
    int8_t *dst = reinterpret_cast<int8_t *>(a.rows + i * a.row_pitch + a.off_ints) + KL * N * 4;
    stage_prep<P>(a.sk + i * a.sk_pitch, dst, u / (N / 8), u % (N / 8));
}

// item and nonce of slot s of the current round
struct Attempt {
    uint32_t item, nonce;
};
__device__ __forceinline__ Attempt slot_attempt(const Chain &ch, const ChainCtl &c, uint32_t s) {
    const uint32_t o = s / c.m;
    const uint2 e = *chain_entry(ch, c.cur, o);
    return {e.x, e.y + (s - o * c.m)};
}

// Layout of a round's hashes by their number.  A chained permutation of a
// lone wave takes 8.6 / 5.9 / 3.5 us with one, two or sixteen lanes per
// state, and the card runs 9.6 / 7.4 / 2.1 G permutations/s: the row form
// while its waves have SIMDs of their own, then the pair form, then one lane.
constexpr uint32_t Y_ROW_MAX = 4096, Y_PAIR_MAX = 32768, C_ROW_MAX = 4096;
constexpr uint32_t ROW_LDS = 4 * 4 * ROW_LDS_WORDS;

template <class P>
__global__ __launch_bounds__(256) void sg_ry_kernel(SignArgs a, SlotRef sr, Chain ch) {
    using SL = SlotLayout<P>;
    __shared__ uint32_t lds[ROW_LDS];
    const ChainCtl c = *chain_ctl<P>(ch);
    const uint32_t total = c.count * c.m * P::L, stride = gridDim.x * 256;
    uint32_t t = blockIdx.x * 256 + threadIdx.x;
    __builtin_amdgcn_s_setprio(2);
    if (total <= Y_ROW_MAX) {
        const RowLane r = row_lane_setup(lds, (threadIdx.x >> 6) * 4 * ROW_LDS_WORDS);
        // whole waves: rows past the end run along without storing
        for (; (t & ~63u) < 16 * total; t += stride) {
            const bool run = t < 16 * total;
            const uint32_t q = run ? t >> 4 : 0, s = q / P::L, l = q % P::L;
            const Attempt at = slot_attempt(ch, c, s);
            mask_raw_row(reinterpret_cast<const uint32_t *>(a.rows + at.item * a.row_pitch + SignLayout<P>::RHOPRIME),
                         P::L * at.nonce + l,
                         reinterpret_cast<uint32_t *>(sr.base + s * sr.pitch + SL::YRAW + l * Sizes<P>::YRAW_BYTES), r,
                         lds, run);
        }
    } else if (total <= Y_PAIR_MAX) {
        for (; t < 2 * total; t += stride) {
            const uint32_t q = t >> 1, s = q / P::L;
            const Attempt at = slot_attempt(ch, c, s);
            stage_y_pair<P>(a, at.item, at.nonce, (int)(q % P::L), sr.base + s * sr.pitch, t & 1);
        }
    } else {
        for (; t < total; t += stride) {
            const uint32_t s = t / P::L;
            const Attempt at = slot_attempt(ch, c, s);
            stage_y<P>(a, at.item, at.nonce, (int)(t % P::L), sr.base + s * sr.pitch);
        }
    }
}

template <class P>
__global__ __launch_bounds__(64 * ROUND_WAVES) void sg_rw_kernel(SignArgs a, SlotRef sr, Chain ch) {
    __shared__ ZetaLds zt;
    __shared__ int32_t x[ROUND_WAVES][NTT_XBUF];
    const ChainCtl c = *chain_ctl<P>(ch);
    const uint32_t slots = c.count * c.m;
    if (blockIdx.x * ROUND_WAVES >= slots) return;
    zeta_lds_load(zt);
    __syncthreads();
    const uint32_t w = threadIdx.x >> 6;
    for (uint32_t s = blockIdx.x * ROUND_WAVES + w; s < slots; s += gridDim.x * ROUND_WAVES)
        stage_w<P>(a, slot_attempt(ch, c, s).item, sr.base + s * sr.pitch, x[w], zt);
}

template <class P>
__global__ __launch_bounds__(256) void sg_rc_kernel(SignArgs a, SlotRef sr, Chain ch) {
    using SL = SlotLayout<P>;
    __shared__ uint32_t lds[ROW_LDS];
    __shared__ uint32_t chal[16 * CHALLENGE_ROW_WORDS];
    const ChainCtl c = *chain_ctl<P>(ch);
    const uint32_t slots = c.count * c.m, stride = gridDim.x * 256;
    uint32_t t = blockIdx.x * 256 + threadIdx.x;
    __builtin_amdgcn_s_setprio(2);
    if (slots <= C_ROW_MAX) {
        const RowLane r = row_lane_setup(lds, (threadIdx.x >> 6) * 4 * ROW_LDS_WORDS);
        for (; (t & ~63u) < 16 * slots; t += stride) {
            const bool run = t < 16 * slots;
            const uint32_t s = run ? t >> 4 : 0;
            uint8_t *slot = sr.base + s * sr.pitch;
            const uint8_t *row = a.rows + slot_attempt(ch, c, s).item * a.row_pitch;
            stage_c_row<P>(reinterpret_cast<const uint32_t *>(row + SignLayout<P>::MU),
                           reinterpret_cast<const uint32_t *>(slot + SL::W1PK),
                           reinterpret_cast<uint32_t *>(slot + SL::CT), reinterpret_cast<uint32_t *>(slot + SL::CP), r,
                           lds, chal + (threadIdx.x >> 4) * CHALLENGE_ROW_WORDS, run);
        }
    } else {
        for (; t < 2 * slots; t += stride) {
            const uint32_t s = t >> 1;
            uint8_t *slot = sr.base + s * sr.pitch;
            stage_c_pair<P>(a, slot_attempt(ch, c, s).item, slot, slot + SL::CT, t & 1);
        }
    }
}

constexpr uint32_t ENTRY_DONE = 0xFFFFFFFFu;  // item of an entry whose signature is written

// The attempts are latency-bound (a few dependent rounds of memory per
// attempt, little arithmetic), so an item's attempts are checked by waves of
// their own: W waves per item, the first attempt writing its signature as it
// goes; if only a later one passes, it is run again to write.
template <class P>
__global__ __launch_bounds__(64 * ROUND_WAVES) void sg_rz_kernel(SignArgs a, SlotRef sr, Chain ch) {
    using SL = SlotLayout<P>;
    __shared__ ZScratch<P> zs[ROUND_WAVES];
    __shared__ uint32_t best[ROUND_WAVES];
    const ChainCtl c = *chain_ctl<P>(ch);
    const uint32_t w = threadIdx.x >> 6, lane = (uint32_t)lane_id();
    const uint32_t W = c.m == 1 ? 1 : c.m == 2 ? 2 : 4, per = ROUND_WAVES / W, sub = w / W, j0 = w % W;
    for (uint32_t o0 = blockIdx.x * per; o0 < c.count; o0 += gridDim.x * per) {
        if (threadIdx.x < ROUND_WAVES) best[threadIdx.x] = c.m;
        __syncthreads();
        const uint32_t o = o0 + sub;
        const bool have = o < c.count;
        uint2 *const entry = chain_entry(ch, c.cur, have ? o : 0);
        const uint2 e = *entry;
        uint8_t *dst = a.sig + (size_t)e.x * a.sig_pitch;
        auto slot_of = [&](uint32_t j) { return sr.base + (size_t)(o * c.m + j) * sr.pitch; };
        if (have) {
            for (uint32_t j = j0; j < c.m && j < *(volatile uint32_t *)&best[sub]; j += W) {
                const bool ok = j == 0 ? stage_z<P, true>(a, e.x, slot_of(j), dst, zs[w])
                                       : stage_z<P, false>(a, e.x, slot_of(j), dst, zs[w]);
                if (ok) {
                    if (lane == 0) atomicMin(&best[sub], j);
                    break;
                }
            }
        }
        __syncthreads();
        if (have) {
            const uint32_t j = best[sub];
            if (j == c.m) {
                if (j0 == 0 && lane == 0) entry->y = e.y + c.m;
            } else if (j0 == j % W) {
                const uint8_t *ct = slot_of(j) + SL::CT;
                if (j) (void)stage_z<P, true>(a, e.x, slot_of(j), dst, zs[w]);
                if (lane < SEEDBYTES) dst[lane] = ct[lane];
                if (lane == 0) {
                    *reinterpret_cast<uint32_t *>(a.rows + (size_t)e.x * a.row_pitch + SignLayout<P>::ATTEMPTS) =
                        e.y + j + 1;
                    entry->x = ENTRY_DONE;
                }
            }
        }
        __syncthreads();  // best is read before the next items reset it
    }
}

// ctl: the call's control words (attempts executed at [2])
constexpr int PLAN_THREADS = 1024;
template <class P>
__global__ __launch_bounds__(PLAN_THREADS) void sg_plan_kernel(Chain ch, uint32_t *ctl) {
    __shared__ uint32_t sums[PLAN_THREADS / 64];
    ChainCtl *const cc = chain_ctl<P>(ch);
    const ChainCtl c = *cc;
    if (c.left == 0) return;  // count is 0 already
    const uint32_t t = threadIdx.x, w = t >> 6, lane = t & 63;
    // thread t keeps the order of entries [t * per, (t + 1) * per)
    const uint32_t per = (c.left + PLAN_THREADS - 1) / PLAN_THREADS, e0 = t * per, e1 = min(e0 + per, c.left);
    uint32_t alive = 0;
    for (uint32_t e = e0; e < e1; ++e) alive += chain_entry(ch, c.cur, e)->x != ENTRY_DONE;
    uint32_t incl = alive;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t v = (uint32_t)__shfl_up((int)incl, d);
        if (lane >= (uint32_t)d) incl += v;
    }
    if (lane == 63) sums[w] = incl;
    __syncthreads();
    uint32_t before = 0, total = 0;
#pragma unroll
    for (uint32_t i = 0; i < PLAN_THREADS / 64; ++i) {
        before += i < w ? sums[i] : 0u;
        total += sums[i];
    }
    uint32_t at = before + incl - alive;
    for (uint32_t e = e0; e < e1; ++e) {
        const uint2 v = *chain_entry(ch, c.cur, e);
        if (v.x != ENTRY_DONE) *chain_entry(ch, c.cur ^ 1, at++) = v;
    }
    if (t == 0) {
        ChainCtl nx{total, 0, 0, c.cur ^ 1, 0};
        plan_round(total, ch.nslots, ch.target, nx.count, nx.m);
        *cc = nx;
        atomicAdd(ctl + 2, c.count * c.m);
    }
}

// --------------------------------------------------------------------- host

namespace {

size_t chain_chunks(size_t n) { return (n + CHAIN_CHUNK - 1) / CHAIN_CHUNK; }

template <class P>
int launch_fixed(const SignArgs &a, const Chain &ch, hipStream_t st) {
    constexpr int KL = P::K * P::L, PREP = (P::L + 2 * P::K) * (N / 8);
    // one sponge per 16-lane row where the rows of all messages fit the card
    // beside the other roles, or on request
    const bool row = a.row_mu || ch.n <= FIXED_ROW_MAX;
    FixedGrid g;
    g.mu = row ? (ch.n + ROW_ITEMS_PER_BLOCK - 1) / ROW_ITEMS_PER_BLOCK : (ch.n + 127) / 128;
    g.expand = a.key_idx ? 0 : (uint32_t)(((size_t)ch.n * KL + 255) / 256);  // resident keys are expanded
    g.prep = a.key_idx ? 0 : (uint32_t)(((size_t)ch.n * PREP + 255) / 256);
    const dim3 grid(g.mu + g.expand + g.prep);
    if (row)
        hipLaunchKernelGGL((sg_fixed_kernel<P, true>), grid, dim3(256), 0, st, a, ch, g);
    else
        hipLaunchKernelGGL((sg_fixed_kernel<P, false>), grid, dim3(256), 0, st, a, ch, g);
    return (int)hipGetLastError();
}

template <class P>
int launch_round(const SignArgs &a, const SlotRef &sr, const Chain &ch, double &u, uint32_t *ctl, hipStream_t st) {
    // mean attempts per signature: 4.25, 5.1, 3.85
    const double fail = P::MODE == 2 ? 1.0 - 1.0 / 4.25 : P::MODE == 3 ? 1.0 - 1.0 / 5.1 : 1.0 - 1.0 / 3.85;
    uint32_t count, m;
    plan_round((uint32_t)std::ceil(u), ch.nslots, ch.target, count, m);
    // grids for the expected round (every kernel strides over what there is)
    const uint32_t slots = count * m;
    auto blocks = [](uint32_t units, uint32_t per, uint32_t cap) {
        return dim3(std::max(1u, std::min((units + per - 1) / per, cap)));
    };
    const uint32_t total = slots * P::L;
    const uint32_t lanes = total <= Y_ROW_MAX ? 16 * total : total <= Y_PAIR_MAX ? 2 * total : total;
    hipLaunchKernelGGL(sg_ry_kernel<P>, blocks(lanes, 256, 4096), dim3(256), 0, st, a, sr, ch);
    hipLaunchKernelGGL(sg_rw_kernel<P>, blocks(slots, ROUND_WAVES, 8192), dim3(64 * ROUND_WAVES), 0, st, a, sr, ch);
    hipLaunchKernelGGL(sg_rc_kernel<P>, blocks((slots <= C_ROW_MAX ? 16 : 2) * slots, 256, 4096), dim3(256), 0, st,
                       a, sr, ch);
    hipLaunchKernelGGL(sg_rz_kernel<P>, blocks(m == 1 ? (count + 3) / 4 : m == 2 ? (count + 1) / 2 : count, 1, 8192),
                       dim3(64 * ROUND_WAVES), 0, st, a, sr, ch);
    hipLaunchKernelGGL(sg_plan_kernel<P>, dim3(1), dim3(PLAN_THREADS), 0, st, ch, ctl);
    u = (u > count ? u - count : 0.0) + std::min(u, (double)count) * std::pow(fail, m);
    return (int)hipGetLastError();
}

template <class P>
int sign_impl(const SignArgs &a, const SlotRef &sr, size_t nslots, const ChunkRef &lists, const PersistTiling &tiling,
              uint32_t *ctl, unsigned long long *phase_sums, hipStream_t st, hipEvent_t fixed_done) {
    int e = launch_zero_ctl(ctl, phase_sums, st);
    if (e) return e;
    const bool rounds = !phase_sums && a.n <= ROUNDS_MAX_ITEMS;
    // two chains of at least 2,048 items
    const int nchain = rounds && a.n >= 4096 ? 2 : 1;
    AuxStreams *aux = nullptr;
    std::unique_lock<std::mutex> guard;
    if (nchain == 2) {
        aux = aux_streams(st);
        if (!aux) return (int)hipErrorOutOfMemory;
        guard = std::unique_lock<std::mutex>(aux->lock);
        if ((e = (int)hipEventRecord(aux->fork, st))) return e;
        if ((e = (int)hipStreamWaitEvent(aux->s[0], aux->fork, 0))) return e;
    }
    Chain ch[2];
    SlotRef csr[2];
    hipStream_t cs[2];
    double u[2];
    size_t first = 0, slot = 0;
    for (int k = 0; k < nchain; ++k) {
        const size_t n = a.n * (k + 1) / nchain - first, ns = nslots * (k + 1) / nchain - slot;
        ch[k].rows = a.rows + first * a.row_pitch;
        ch[k].lists = lists.base + (k ? chain_chunks(ch[0].n) * lists.pitch : 0);
        ch[k].chunk_pitch = lists.pitch;
        ch[k].first = (uint32_t)first;
        ch[k].n = (uint32_t)n;
        ch[k].nslots = (uint32_t)ns;
        ch[k].target = (uint32_t)std::min<size_t>(ns, ROUND_TARGET / nchain);
        csr[k] = sr;
        csr[k].base += slot * sr.pitch;
        cs[k] = k == 0 ? st : aux->s[0];
        u[k] = (double)n;
        first += n;
        slot += ns;
    }
    for (int k = 0; k < nchain; ++k) {
        if ((e = launch_fixed<P>(a, ch[k], cs[k]))) return e;
        if (k == 0 && fixed_done && (e = (int)hipEventRecord(fixed_done, cs[0]))) return e;
    }
    if (!rounds) {
        const size_t ns = tiling.nslots ? tiling.nslots : nslots;
        const int spb = tiling.slots_per_block ? tiling.slots_per_block : default_slots_per_block(ns);
        return launch_sign_persistent(P::MODE, a, sr, ch[0], ns, spb, tiling.blocks, tiling.claim, ctl, phase_sums,
                                      st);
    }
    // the chains' rounds in turn, so that neither stream waits for the host
    for (int r = 0; r < 48 && (u[0] > 0.05 || (nchain == 2 && u[1] > 0.05)); ++r)
        for (int k = 0; k < nchain; ++k)
            if (u[k] > 0.05 && (e = launch_round<P>(a, csr[k], ch[k], u[k], ctl, cs[k]))) return e;
    for (int k = 0; k < nchain; ++k)
        if ((e = launch_sign_persistent(P::MODE, a, csr[k], ch[k], ch[k].nslots, ch[k].nslots >= 8 ? 8 : 1, 64, 1, ctl,
                                        nullptr, cs[k])))
            return e;
    if (nchain == 2) {
        if ((e = (int)hipEventRecord(aux->join[0], aux->s[0]))) return e;
        return (int)hipStreamWaitEvent(st, aux->join[0], 0);
    }
    return 0;
}

}  // namespace

int launch_sign_fixed(int mode, const SignArgs &a, const Chain &ch, hipStream_t st) {
    if (ch.n == 0) return 0;
    switch (mode) {
        case 2: return launch_fixed<Params<2>>(a, ch, st);
        case 3: return launch_fixed<Params<3>>(a, ch, st);
        case 5: return launch_fixed<Params<5>>(a, ch, st);
        default: return -1;
    }
}

size_t sign_lists_chunks(size_t n) { return chain_chunks(n) + 1; }
size_t sign_lists_chunk_bytes() { return CHAIN_CHUNK_BYTES; }

int sign_call(int mode, const SignArgs &a, const SlotRef &sr, size_t nslots, const ChunkRef &lists,
              const PersistTiling &tiling, uint32_t *ctl, unsigned long long *phase_sums, hipStream_t st,
              hipEvent_t fixed_done) {
    if (a.n == 0) return 0;
    if (nslots == 0) return -3;
    switch (mode) {
        case 2: return sign_impl<Params<2>>(a, sr, nslots, lists, tiling, ctl, phase_sums, st, fixed_done);
        case 3: return sign_impl<Params<3>>(a, sr, nslots, lists, tiling, ctl, phase_sums, st, fixed_done);
        case 5: return sign_impl<Params<5>>(a, sr, nslots, lists, tiling, ctl, phase_sums, st, fixed_done);
        default: return -1;
    }
}

}  // namespace dil
