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
//   y      lane, lane pair or wave per mask sponge
//   w      wave per attempt
//   c      lane pair, 16-lane row or wave per attempt
//   z      wave per attempt: the checks of r0 and z
//   s      wave per item: the first of its attempts in nonce order that passed
//          them and passes c t0 and the hints is the specification's signature
//   plan   one workgroup lists the items without a signature and plans the
//          next round (how many items, how many consecutive nonces for each),
//          so the host issues a fixed sequence of launches and never waits.
//          (A shared queue that z pushes to with atomics was slower: some
//          thousand atomics on one address from eight XCDs' L2 caches take
//          about 50 ns each, 430 us per round of 16,384 attempts.)
//
// The sequence is as long as the expected decay of the batch needs; what is
// left after it (rarely anything) is finished by the persistent kernel, which
// takes its items from the same queue.  The largest batches run as two chains
// of rounds on two streams, so that the hash launches of one fill the SIMDs
// that the other leaves idle.
//
// 16,384 Dilithium3 items in one chain: fixed 401 us; the rounds' y 490, w
// 725, c 510, z 290, s 257 and plan 60 us.  y and c are serial chains of
// permutations in every round (c 64 us with lane pairs for any number up to
// 32,768), w and z bound by their vector instructions and memory waits.
//
// The reference issues its rounds from the host with a synchronisation and
// about eight small copies per round (api.cu:208-441).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <mutex>

#include "hash_row.hpp"
#include "internal.hpp"
#include "sign_stages.hpp"

namespace dil {

constexpr int ROUND_WAVES = 4;
constexpr uint32_t ROUND_MAX_M = 32;  // attempts per item and round
// Messages hashed with a 16-lane row each up to this batch: beyond, the rows'
// fourfold instruction count costs ExpandA beside them more than the shorter
// chain gives.  Whole calls, messages up to 4 KiB, rows / lane pairs: 5,000
// Dilithium3 items 1.19 / 1.36 ms, 6,000 Dilithium2 1.01 / 1.20, 8,000
// Dilithium3 1.59 / 1.62 (resident 1.46 / 1.61), 8,000 Dilithium5 1.67 / 1.66,
// 12,000 Dilithium3 2.11 / 2.06; 32-byte messages 6,000 Dilithium3 1.27 / 1.26.
constexpr size_t FIXED_ROW_MAX = 8192;
// With a wave each up to these, the second with resident keys, where nothing
// runs beside the hashes (messages up to 4 KiB, whole call with waves / rows:
// 1,000 Dilithium3 items 465 / 517 us, 2,000 Dilithium5 691 / 713, 3,001
// Dilithium5 960 / 938; resident 3,000 Dilithium5 862 / 910).
constexpr uint32_t FIXED_WAVE_MAX = 2048, FIXED_WAVE_MAX_RESIDENT = 3072;
// The persistent kernel, which needs no launches between stages, runs what is
// left after the rounds, and alone the calls with so many items per slot that
// the sequence of rounds would leave most of them.  Rounds / persistent with two
// slots per item: 17 Dilithium3 items 0.53 / 0.75 ms, 1,000 Dilithium2 0.50 /
// 0.78, 3,001 Dilithium5 0.97 / 1.18, 10,000 Dilithium2 1.27 / 1.42, 16,384
// Dilithium3 2.49 / 2.79; with 8 items per slot 1,000 Dilithium2 2.95 / 8.06,
// 10,000 Dilithium2 4.8 / 7.7; 32: 36 / 52 and 29 / 31; 64: 122 / 67 and 67 / 69.
constexpr size_t ROUNDS_MAX_ITEMS_PER_SLOT = 32;
// Two chains from this batch on: 16,384 Dilithium3 items 2.45 ms (one chain
// 2.60), 40,000 5.03 (5.36), 14,000 2.19 (2.29), 16,384 Dilithium5 2.87
// (2.84); smaller ones lose as much as they gain (12,288 Dilithium2 1.46 and
// 1.44 ms, Dilithium3 2.13 and 2.14, 10,000 Dilithium2 1.29 and 1.28).
constexpr size_t TWO_CHAINS_MIN = 12288;
// Attempts a round aims at when few items are left, and the least per item.
// A second attempt reads the item's A from L2 and saves rounds: 40,000
// Dilithium3 items 5.03 ms, 5.62 with a least of one; 16,384 2.50 and 2.71.
// Targets of 8,192 / 16,384 attempts: 10,000 Dilithium2 items 1.41 / 1.28 ms,
// 16,384 Dilithium3 2.69 / 2.60, 8,000 Dilithium5 1.74 / 1.73.
constexpr size_t ROUND_TARGET = 16384;
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
    uint32_t expand_wave;       // ExpandA with a wave per entry instead of a lane
};
// Up to this many entries of A (with waves for the message hashes too): the
// chain of a lane's five permutations is 48 us, a wave's 12.  Whole calls with
// 32-byte messages: 1 Dilithium2 item 92 us (lanes 140), 500 Dilithium2 292
// (307), 270 Dilithium3 265 (282), 146 Dilithium5 238 (256).
constexpr size_t EXPAND_WAVE_MAX = 8192;

// lanes per message hash
enum { MU_PAIR = 2, MU_ROW = 16, MU_WAVE = 64 };

template <class P, int LANES>
__global__ __launch_bounds__(256) void sg_fixed_kernel(SignArgs a, Chain ch, FixedGrid g) {
    constexpr int KL = P::K * P::L, PREP = (P::L + 2 * P::K) * (N / 8);
    __shared__ __align__(8) uint32_t
        lds[LANES == MU_WAVE ? 4 * WAVE_LDS_WORDS : LANES == MU_ROW ? 4 * 4 * ROW_LDS_WORDS : 1];
    uint32_t b = blockIdx.x;
    if (b < g.mu) {
        // serial chains, which end the stage: highest issue priority
        __builtin_amdgcn_s_setprio(3);
        const uint32_t t = threadIdx.x;
        const uint32_t i = b * (256 / LANES) + t / LANES;
        RowLane r;
        if constexpr (LANES == MU_ROW) r = row_lane_setup(lds, (t >> 6) * 4 * ROW_LDS_WORDS);
        if (i >= ch.n) return;  // whole waves / rows / pairs of lanes
        if (t % LANES == 0) {
            if (ch.lists) *chain_entry(ch, 0, i) = make_uint2(ch.first + i, 0);
            if (ch.lists && i == 0) {
                ChainCtl c{ch.n, 0, 0, 0, 0};
                plan_round(ch.n, ch.nslots, ch.target, c.count, c.m);
                *chain_ctl<P>(ch) = c;
            }
        }
        if constexpr (LANES == MU_WAVE) {
            const uint32_t base = (t >> 6) * WAVE_LDS_WORDS;
            stage_mu_wave<P>(a, ch.first + i, wave_lane_setup(lds, base), lds, base);
        } else if constexpr (LANES == MU_ROW)
            stage_mu_row<P>(a, ch.first + i, r, lds, t >> 6);
        else
            stage_mu_pair<P>(a, ch.first + i, t & 1);
        return;
    }
    b -= g.mu;
    if (b < g.expand) {
        if constexpr (LANES == MU_WAVE) {
            if (g.expand_wave) {
                __shared__ __align__(8) uint32_t block[4][EXPAND_WAVE_WORDS];
                const uint32_t w = threadIdx.x >> 6, t = b * 4 + w, i = t / KL, e = t % KL;
                if (i >= ch.n) return;  // whole waves
                const size_t item = ch.first + i;
                expand_a_wave(reinterpret_cast<int32_t *>(a.rows + item * a.row_pitch + a.off_ints) + e * N,
                              a.sk + item * a.sk_pitch, e / P::L << 8 | e % P::L,
                              wave_lane_setup(lds, w * WAVE_LDS_WORDS), lds, block[w]);
                return;
            }
        }
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
// lone wave takes 8.6 / 5.9 / 3.5 / 2.2 us with one, two, sixteen or 64 lanes
// per state, and the card runs 9.6 / 7.4 / 2.1 / 0.9 G permutations/s: the
// wave form while its waves are few, then (challenges) rows, pairs and one
// lane; the mask chains are shorter and have no rows.  17 resident Dilithium3
// items 151 us (157 with 2,048 for both limits, 218 without the wave form).
// Challenges, whole calls with 32-byte messages and rounds of that many
// attempts, waves / rows: 2,500 Dilithium3 1067 / 1098 us, 3,000 Dilithium2
// 883 / 905, 3,000 Dilithium5 657 / 674; 4,000 Dilithium3 1301 / 1200, 4,096
// Dilithium2 618 / 578, 4,096 Dilithium5 806 / 754; rows / pairs: one round of
// 8,192 40 / 64 us.
constexpr uint32_t Y_WAVE_MAX = 4096, Y_PAIR_MAX = 32768;
constexpr uint32_t C_WAVE_MAX = 3072, C_ROW_MAX = 8192;
constexpr uint32_t ROW_LDS = 4 * 4 * ROW_LDS_WORDS;
static_assert(ROW_LDS >= 4 * WAVE_LDS_WORDS, "the row form's LDS also serves the wave form");

template <class P>
__global__ __launch_bounds__(256) void sg_ry_kernel(SignArgs a, SlotRef sr, Chain ch) {
    using SL = SlotLayout<P>;
    __shared__ __align__(8) uint32_t lds[4 * WAVE_LDS_WORDS];
    const ChainCtl c = *chain_ctl<P>(ch);
    const uint32_t total = c.count * c.m * P::L, stride = gridDim.x * 256;
    uint32_t t = blockIdx.x * 256 + threadIdx.x;
    __builtin_amdgcn_s_setprio(2);
    if (total <= Y_WAVE_MAX) {
        const WaveLane r = wave_lane_setup(lds, (threadIdx.x >> 6) * WAVE_LDS_WORDS);
        for (; t < 64 * total; t += stride) {
            const uint32_t q = t >> 6, s = q / P::L, l = q % P::L;
            const Attempt at = slot_attempt(ch, c, s);
            mask_raw_wave(reinterpret_cast<const uint32_t *>(a.rows + at.item * a.row_pitch + SignLayout<P>::RHOPRIME),
                          P::L * at.nonce + l,
                          reinterpret_cast<uint32_t *>(sr.base + s * sr.pitch + SL::YRAW + l * Sizes<P>::YRAW_BYTES),
                          r, lds);
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
    __shared__ __align__(8) uint32_t lds[ROW_LDS];
    __shared__ uint32_t chal[16 * CHALLENGE_ROW_WORDS];
    const ChainCtl c = *chain_ctl<P>(ch);
    const uint32_t slots = c.count * c.m, stride = gridDim.x * 256;
    uint32_t t = blockIdx.x * 256 + threadIdx.x;
    __builtin_amdgcn_s_setprio(2);
    if (slots <= C_WAVE_MAX) {
        const WaveLane r = wave_lane_setup(lds, (threadIdx.x >> 6) * WAVE_LDS_WORDS);
        for (; t < 64 * slots; t += stride) {
            const uint32_t s = t >> 6;
            uint8_t *slot = sr.base + s * sr.pitch;
            const uint8_t *row = a.rows + slot_attempt(ch, c, s).item * a.row_pitch;
            stage_c_wave<P>(reinterpret_cast<const uint32_t *>(row + SignLayout<P>::MU),
                            reinterpret_cast<const uint32_t *>(slot + SL::W1PK),
                            reinterpret_cast<uint32_t *>(slot + SL::CT), reinterpret_cast<uint32_t *>(slot + SL::CP),
                            r, lds, chal + (threadIdx.x >> 6) * CHALLENGE_ROW_WORDS);
        }
    } else if (slots <= C_ROW_MAX) {
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

// The attempts are latency-bound (a few dependent rounds of memory each, little
// arithmetic) and most end early, so r0 and z are checked by a wave and a
// workgroup per attempt, which leave the CU as soon as they are decided.
template <class P>
__global__ __launch_bounds__(64) void sg_rz_kernel(SignArgs a, SlotRef sr, Chain ch) {
    using SL = SlotLayout<P>;
    __shared__ ZScratch<P, true> zs;
    const ChainCtl c = *chain_ctl<P>(ch);
    const uint32_t slots = c.count * c.m;
    for (uint32_t s = blockIdx.x; s < slots; s += gridDim.x) {
        uint8_t *slot = sr.base + s * sr.pitch;
        const bool ok = stage_z<P, true>(a, slot_attempt(ch, c, s).item, slot, nullptr, zs);
        if (lane_id() == 0) *reinterpret_cast<uint32_t *>(slot + SL::FLAG) = ok;
    }
}

// Wave per item: the first of its attempts that passed the checks and also
// passes c t0 and the hints is its signature.
template <class P>
__global__ __launch_bounds__(64) void sg_rs_kernel(SignArgs a, SlotRef sr, Chain ch) {
    using SL = SlotLayout<P>;
    __shared__ ZScratch<P> zs;
    const ChainCtl c = *chain_ctl<P>(ch);
    const uint32_t lane = (uint32_t)lane_id();
    for (uint32_t o = blockIdx.x; o < c.count; o += gridDim.x) {
        uint2 *const entry = chain_entry(ch, c.cur, o);
        const uint2 e = *entry;
        uint8_t *const slots = sr.base + (size_t)o * c.m * sr.pitch;
        uint32_t passed = 0;  // m <= ROUND_MAX_M <= 32
        if (lane < c.m) passed = *reinterpret_cast<const uint32_t *>(slots + lane * sr.pitch + SL::FLAG);
        uint64_t left = __ballot(passed != 0);
        uint8_t *dst = a.sig + (size_t)e.x * a.sig_pitch;
        bool done = false;
        while (left && !done) {
            const uint32_t j = (uint32_t)__ffsll((unsigned long long)left) - 1;
            left &= left - 1;
            uint8_t *slot = slots + j * sr.pitch;
            done = stage_z<P>(a, e.x, slot, dst, zs);
            if (done) {
                if (lane < SEEDBYTES) dst[lane] = slot[SL::CT + lane];
                if (lane == 0) {
                    *reinterpret_cast<uint32_t *>(a.rows + (size_t)e.x * a.row_pitch + SignLayout<P>::ATTEMPTS) =
                        e.y + j + 1;
                    entry->x = ENTRY_DONE;
                }
            }
        }
        if (!done && lane == 0) entry->y = e.y + c.m;
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
    // wave w keeps the order of its run of entries, 64 at a time
    const uint32_t run = ((c.left + PLAN_THREADS - 1) / PLAN_THREADS) * 64, e0 = w * run, e1 = min(e0 + run, c.left);
    auto alive = [&](uint32_t e, uint2 &v) {
        v = e < e1 ? *chain_entry(ch, c.cur, e) : make_uint2(ENTRY_DONE, 0);
        return v.x != ENTRY_DONE;
    };
    uint32_t count = 0;
    uint2 v;
    for (uint32_t e = e0; e < e1; e += 64) count += __popcll(__ballot(alive(e + lane, v)));
    if (lane == 0) sums[w] = count;
    __syncthreads();
    uint32_t at = 0, total = 0;
#pragma unroll
    for (uint32_t i = 0; i < PLAN_THREADS / 64; ++i) {
        at += i < w ? sums[i] : 0u;
        total += sums[i];
    }
    for (uint32_t e = e0; e < e1; e += 64) {
        const bool keep = alive(e + lane, v);
        const uint64_t mask = __ballot(keep);
        if (keep) *chain_entry(ch, c.cur ^ 1, at + __popcll(mask & ((1ull << lane) - 1ull))) = v;
        at += __popcll(mask);
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
    // one sponge per wave or 16-lane row where those of all messages fit the
    // card beside the other roles, or (rows) on request
    const bool wave = ch.n <= (a.key_idx ? FIXED_WAVE_MAX_RESIDENT : FIXED_WAVE_MAX);
    const int lanes = wave ? MU_WAVE : a.row_mu || a.n <= FIXED_ROW_MAX ? MU_ROW : MU_PAIR;
    const uint32_t per = 256 / lanes;
    FixedGrid g;
    g.mu = (ch.n + per - 1) / per;
    const size_t entries = a.key_idx ? 0 : (size_t)ch.n * KL;  // resident keys are expanded
    g.expand_wave = lanes == MU_WAVE && entries <= EXPAND_WAVE_MAX;
    g.expand = (uint32_t)(g.expand_wave ? (entries + 3) / 4 : (entries + 255) / 256);
    g.prep = a.key_idx ? 0 : (uint32_t)(((size_t)ch.n * PREP + 255) / 256);
    const dim3 grid(g.mu + g.expand + g.prep);
    if (lanes == MU_WAVE)
        hipLaunchKernelGGL((sg_fixed_kernel<P, MU_WAVE>), grid, dim3(256), 0, st, a, ch, g);
    else if (lanes == MU_ROW)
        hipLaunchKernelGGL((sg_fixed_kernel<P, MU_ROW>), grid, dim3(256), 0, st, a, ch, g);
    else
        hipLaunchKernelGGL((sg_fixed_kernel<P, MU_PAIR>), grid, dim3(256), 0, st, a, ch, g);
    return (int)hipGetLastError();
}

template <class P>
int launch_round(const SignArgs &a, const SlotRef &sr, const Chain &ch, double &u, uint32_t *ctl, hipStream_t st) {
    // mean attempts per signature: 4.25, 5.1, 3.85
    const double fail = P::MODE == 2 ? 1.0 - 1.0 / 4.25 : P::MODE == 3 ? 1.0 - 1.0 / 5.1 : 1.0 - 1.0 / 3.85;
    uint32_t count, m;
    plan_round((uint32_t)std::ceil(u), ch.nslots, ch.target, count, m);
    // The count on the device differs from the expected one by a few percent, and
    // an attempt more than a hash grid holds costs its wave a second chain of
    // permutations (13,700 challenge hashes 62 us, 120 us with a grid for 13,600).
    // So the grids cover the largest need within an eighth of the expectation,
    // over every form and m that such a count selects; blocks without work exit.
    const uint32_t lo = count - count / 8, hi = std::min(count + count / 8 + 64, ch.n);
    const uint32_t most = std::min(ch.nslots, std::max(hi * ROUND_MIN_M, std::min(hi * ROUND_MAX_M, ch.target)));
    const uint32_t slots = std::min(most, count * m + count * m / 8 + 64);
    auto blocks = [](uint32_t units, uint32_t per, uint32_t cap) {
        return dim3(std::max(1u, std::min((units + per - 1) / per, cap)));
    };
    auto lanes_y = [](uint32_t t) {
        return t <= Y_WAVE_MAX ? 64 * t : t <= Y_PAIR_MAX ? 2 * t : t;
    };
    auto lanes_c = [](uint32_t t) { return t <= C_WAVE_MAX ? 64 * t : t <= C_ROW_MAX ? 16 * t : 2 * t; };
    auto widest = [](auto f, uint32_t from, uint32_t to, std::initializer_list<uint32_t> edges) {
        uint32_t most = f(to);
        for (const uint32_t e : edges) most = std::max(most, e >= from && e <= to ? f(e) : 0u);
        return most;
    };
    const uint32_t least = std::min(lo * ROUND_MIN_M, most);
    const uint32_t ly = widest(lanes_y, least * P::L, most * P::L, {Y_WAVE_MAX, Y_PAIR_MAX});
    const uint32_t lc = widest(lanes_c, least, most, {C_WAVE_MAX, C_ROW_MAX});
    const dim3 gy = blocks(ly, 256, 4096), gc = blocks(lc, 256, 4096);
    hipLaunchKernelGGL(sg_ry_kernel<P>, gy, dim3(256), 0, st, a, sr, ch);
    hipLaunchKernelGGL(sg_rw_kernel<P>, blocks(slots, ROUND_WAVES, 8192), dim3(64 * ROUND_WAVES), 0, st, a, sr, ch);
    hipLaunchKernelGGL(sg_rc_kernel<P>, gc, dim3(256), 0, st, a, sr, ch);
    hipLaunchKernelGGL(sg_rz_kernel<P>, blocks(slots, 1, 32768), dim3(64), 0, st, a, sr, ch);
    hipLaunchKernelGGL(sg_rs_kernel<P>, blocks(hi, 1, 32768), dim3(64), 0, st, a, sr, ch);
    hipLaunchKernelGGL(sg_plan_kernel<P>, dim3(1), dim3(PLAN_THREADS), 0, st, ch, ctl);
    u = (u > count ? u - count : 0.0) + std::min(u, (double)count) * std::pow(fail, m);
    return (int)hipGetLastError();
}

// A second stream forked from the caller's.  join() makes the caller's stream
// wait for it; a way out that did not join, an error on the way, joins in the
// destructor, so that buffers which the caller frees after draining its own
// stream are not in use and a capture is left without a loose branch.
struct ForkedStream {
    AuxStream *aux = nullptr;
    hipStream_t st = nullptr;
    std::unique_lock<std::mutex> guard;
    bool open = false;

    int fork(hipStream_t caller) {
        st = caller;
        if (!(aux = aux_stream(st))) return (int)hipErrorOutOfMemory;
        guard = std::unique_lock<std::mutex>(aux->lock);
        int e = (int)hipEventRecord(aux->fork, st);
        if (!e) e = (int)hipStreamWaitEvent(aux->s, aux->fork, 0);
        open = e == 0;
        return e;
    }
    int join() {
        if (!open) return 0;
        open = false;
        int e = (int)hipEventRecord(aux->join, aux->s);
        if (!e) e = (int)hipStreamWaitEvent(st, aux->join, 0);
        if (e) (void)hipStreamSynchronize(aux->s);
        return e;
    }
    ~ForkedStream() { (void)join(); }
};

template <class P>
int sign_impl(const SignArgs &a, const SlotRef &sr, size_t nslots, const ChunkRef &lists, const PersistTiling &tiling,
              uint32_t *ctl, unsigned long long *phase_sums, hipStream_t st, hipEvent_t *fixed_done) {
    int e = launch_zero_ctl(ctl, phase_sums, st);
    if (e) return e;
    const bool rounds = !phase_sums && a.n <= ROUNDS_MAX_ITEMS_PER_SLOT * nslots;
    const int nchain = rounds && a.n >= TWO_CHAINS_MIN ? 2 : 1;
    ForkedStream second;
    if (nchain == 2 && (e = second.fork(st))) return e;
    Chain ch[2];
    SlotRef csr[2];
    hipStream_t cs[2];
    double u[2] = {0.0, 0.0};
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
        cs[k] = k == 0 ? st : second.aux->s;
        u[k] = (double)n;
        first += n;
        slot += ns;
    }
    for (int k = 0; k < nchain; ++k) {
        if ((e = launch_fixed<P>(a, ch[k], cs[k]))) return e;
    }
    for (int k = 0; fixed_done && k < 2; ++k)
        if ((e = (int)hipEventRecord(fixed_done[k], cs[k < nchain ? k : 0]))) return e;
    if (!rounds) {
        const size_t ns = tiling.nslots ? tiling.nslots : nslots;
        const int spb = tiling.slots_per_block ? tiling.slots_per_block : default_slots_per_block(ns);
        return launch_sign_persistent(P::MODE, a, sr, ch[0], ns, spb, tiling.blocks, tiling.claim, ctl, phase_sums,
                                      st);
    }
    // the chains' rounds in turn, so that neither stream waits for the host
    for (int r = 0; r < 48 && (u[0] > 0.05 || u[1] > 0.05); ++r)
        for (int k = 0; k < nchain; ++k)
            if (u[k] > 0.05 && (e = launch_round<P>(a, csr[k], ch[k], u[k], ctl, cs[k]))) return e;
    for (int k = 0; k < nchain; ++k)
        if ((e = launch_sign_persistent(P::MODE, a, csr[k], ch[k], ch[k].nslots, ch[k].nslots >= 8 ? 8 : 1, 64, 1, ctl,
                                        nullptr, cs[k])))
            return e;
    return second.join();
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
              hipEvent_t *fixed_done) {
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
