// Batched verification (reference: gpu_verify, src/verify.cu:28-325, one
// 32-lane warp per item, A expanded into the pool and read back).
//
// Up to three launches:
//   vf_prep   lane per item: c = SampleInBall(c~).  Small batches leave it to
//             vf_main, one 16-lane row per item
//   vf_main   workgroups of two roles, side by side:
//             mu    tr = H(pk), mu = H(tr || m): a wave, a 16-lane row or
//                   a lane pair per item by batch size; only vf_final needs it
//             main  one wave per FoldCfg<P>::IPW items: hint decoding, z unpack
//                   + norm check + NTT, A z^ straight from the sponges
//                   (fold.hpp), then per row - c^ t1^ 2^d, INTT, caddq,
//                   UseHint, pack w1'.  With resident keys: one workgroup per
//                   G items, A z^ from the stored A.  The smallest batches:
//                   a workgroup per item and row of A (vf_small)
//   vf_final  c~' = H(mu || w1'), compare, write the verdict
// ret is 0 for a valid signature and -1 otherwise (api.cu:454-515).
#include <hip/hip_runtime.h>

#include "fold.hpp"
#include "hash_row.hpp"
#include "internal.hpp"
#include "layout.hpp"
#include "pipelines.hpp"
#include "poly.hpp"
#include "sample.hpp"

namespace dil {

// Batches up to this size (one row wave per SIMD) are latency-bound: hashes
// take a 16-lane row or a wave each and vf_main samples the challenges itself.  2,500
// resident Dilithium3 verifications with messages up to 4 KiB 655 -> 174 us,
// 16 Dilithium2 verifications 309 -> 141 us against one lane per hash.
constexpr size_t VERIFY_ROW_MAX = 4096;
// The smallest of them take a wave per hash, up to the second limit with
// resident keys, where no ExpandA runs beside the hashes (waves / rows: 16
// Dilithium2 items 128 / 141 us, 1,000 Dilithium5 138 / 151, 1,500 Dilithium2
// 205 / 151; resident, messages up to 4 KiB, 1,000 Dilithium3 52 / 72, 2,500
// Dilithium3 122 / 175, 4,000 Dilithium2 187 / 172).
constexpr size_t VERIFY_WAVE_MAX = 1024, VERIFY_WAVE_MAX_RESIDENT = 3072;
// Without resident keys, vf_small takes calls of up to this many entries of A
// (vf_small / vf_main, 32-byte messages: 16 Dilithium2 items 52 / 130 us, 512
// Dilithium2 87 / 132, 270 Dilithium3 98 / 121, 140 Dilithium5 95 / 120; 540
// Dilithium3 147 / 124, 290 Dilithium5 150 / 122).
constexpr size_t VERIFY_SMALL_WAVES = 8192;
static bool wave_hashes(const VerifyArgs &a) {
    return a.n <= (a.key_idx ? VERIFY_WAVE_MAX_RESIDENT : VERIFY_WAVE_MAX);
}
// Beyond, c~' = H(mu || w1') with two lanes per item while those waves fit the
// card twice, else one.
constexpr size_t VERIFY_PAIR_MAX = 32768;

template <class P>
__global__ __launch_bounds__(256) void vf_prep_kernel(VerifyArgs a) {
    using VL = VerifyLayout<P>;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    const uint8_t *sig = a.sig + i * a.sig_pitch;
    uint64_t ct[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) ct[w] = load_le64(sig + 8 * w);
    challenge<P::TAU>(ct, reinterpret_cast<uint32_t *>(a.work + i * a.work_pitch + VL::CP));
}

// ------------------------------------------------------------------ mu role

// lanes per message hash
enum MuForm { MU_PAIR = 2, MU_ROW = 16, MU_WAVE = 64 };
template <int FORM>
constexpr int mu_items(int threads) {
    return threads / FORM;
}

// tr = SHAKE256(pk)[0:32] (or the resident key's) and mu = SHAKE256(tr || m)
// into the work row, two lanes per item (keccak_f1600_pair)
template <class P>
__device__ __forceinline__ void mu_pair(const VerifyArgs &a, size_t i, uint32_t h) {
    using Z = Sizes<P>;
    using VL = VerifyLayout<P>;
    const uint8_t *key = a.key_idx ? a.keys + a.key_idx[i] * a.key_pitch : nullptr;
    uint32_t s[25], tr[4];
    if (key) {
#pragma unroll
        for (int w = 0; w < 4; ++w) tr[w] = load_half_bytes(key + KeyLayout<P>::TR, 8 * w + 4 * h, SEEDBYTES);
    } else {
        const uint8_t *pk = a.pk + i * a.pk_pitch;
        shake_pair<SHAKE256_RATE>(s, h, (uint32_t)Z::PK_BYTES,
                                  [&](uint32_t w) { return load_half_bytes(pk, 8 * w + 4 * h, Z::PK_BYTES); });
#pragma unroll
        for (int w = 0; w < 4; ++w) tr[w] = s[w];
    }
    const uint8_t *m = a.m.ptr(i);
    const uint32_t mlen = a.m.len(i);
    shake_pair<SHAKE256_RATE>(s, h, SEEDBYTES + mlen, [&](uint32_t w) -> uint32_t {
        if (w < 4) return w == 0 ? tr[0] : (w == 1 ? tr[1] : (w == 2 ? tr[2] : tr[3]));
        return load_half_bytes(m, 8 * (w - 4) + 4 * h, mlen);
    });
    uint32_t *hash = reinterpret_cast<uint32_t *>(a.work + i * a.work_pitch + VL::HASH);
#pragma unroll
    for (int w = 0; w < 8; ++w) hash[2 * w + h] = s[w];
}

// the same by the 16 lanes of a row
template <class P>
__device__ __forceinline__ void mu_row(const VerifyArgs &a, size_t i, const RowLane &r, uint32_t *lds, uint32_t wave) {
    using Z = Sizes<P>;
    using VL = VerifyLayout<P>;
    const uint32_t h = r.h;
    const RowShare sh{wave * 4 * ROW_LDS_WORDS + ((uint32_t)lane_id() >> 4) * ROW_LDS_WORDS};
    uint32_t s[5];
    const uint8_t *key = a.key_idx ? a.keys + a.key_idx[i] * a.key_pitch : nullptr;
    if (!key) {
        const uint8_t *pk = a.pk + i * a.pk_pitch;
        shake_row<SHAKE256_RATE>(s, r, lds, (uint32_t)Z::PK_BYTES,
                                 [&](uint32_t w) { return load_half_bytes(pk, 8 * w + 4 * h, Z::PK_BYTES); });
        sh.put(lds, s, r, 4);
        wave_lds_sync();
    }
    const uint8_t *m = a.m.ptr(i);
    const uint32_t mlen = a.m.len(i);
    shake_row<SHAKE256_RATE>(s, r, lds, SEEDBYTES + mlen, [&](uint32_t w) -> uint32_t {
        if (w < 4) return key ? load_half_bytes(key + KeyLayout<P>::TR, 8 * w + 4 * h, SEEDBYTES) : sh.get(lds, w, h);
        return load_half_bytes(m, 8 * (w - 4) + 4 * h, mlen);
    });
    row_store_words(s, r, reinterpret_cast<uint32_t *>(a.work + i * a.work_pitch + VL::HASH), 8);
}

// the same by a wave; lds: its WAVE_LDS_WORDS words at base
template <class P>
__device__ __forceinline__ void mu_wave(const VerifyArgs &a, size_t i, const WaveLane &r, uint32_t *lds,
                                        uint32_t base) {
    using Z = Sizes<P>;
    using VL = VerifyLayout<P>;
    uint32_t lo, hi;
    const uint8_t *key = a.key_idx ? a.keys + a.key_idx[i] * a.key_pitch : nullptr;
    if (!key) {
        const uint8_t *pk = a.pk + i * a.pk_pitch;
        shake_wave<SHAKE256_RATE>(lo, hi, r, lds, (uint32_t)Z::PK_BYTES,
                                  [&](uint32_t w) { return load_word_bytes(pk, 8 * w, Z::PK_BYTES); });
    } else if (r.w < 4) {
        const uint64_t v = load_word_bytes(key + KeyLayout<P>::TR, 8 * r.w, SEEDBYTES);
        lo = (uint32_t)v;
        hi = (uint32_t)(v >> 32);
    }
    // tr's words stay on their lanes: words 0..3 of the next input
    const uint64_t tr = r.w < 4 ? lo | (uint64_t)hi << 32 : 0ull;
    const uint8_t *m = a.m.ptr(i);
    const uint32_t mlen = a.m.len(i);
    shake_wave<SHAKE256_RATE>(lo, hi, r, lds, SEEDBYTES + mlen, [&](uint32_t w) -> uint64_t {
        return w < 4 ? tr : load_word_bytes(m, 8 * (w - 4), mlen);
    });
    wave_store_words(lo, hi, r, reinterpret_cast<uint32_t *>(a.work + i * a.work_pitch + VL::HASH), 8);
}

// one workgroup's share of the mu role; lds: ROW_LDS_WORDS * 4 words per wave,
// 8-byte aligned (row and wave forms)
template <class P, int FORM>
__device__ __forceinline__ void mu_role(const VerifyArgs &a, uint32_t block, uint32_t *lds) {
    // serial chains that end the call: highest issue priority
    __builtin_amdgcn_s_setprio(3);
    const uint32_t t = threadIdx.x;
    const size_t i = (size_t)block * mu_items<FORM>(blockDim.x) + t / FORM;
    RowLane r;
    if constexpr (FORM == MU_ROW) r = row_lane_setup(lds, (t >> 6) * 4 * ROW_LDS_WORDS);
    // whole waves / rows / pairs of lanes; vf_main rejects an index past the store
    if (i >= a.n || (a.key_idx && a.key_idx[i] >= a.nkeys)) return;
    if constexpr (FORM == MU_WAVE) {
        const uint32_t base = (t >> 6) * WAVE_LDS_WORDS;
        mu_wave<P>(a, i, wave_lane_setup(lds, base), lds, base);
    } else if constexpr (FORM == MU_ROW)
        mu_row<P>(a, i, r, lds, t >> 6);
    else
        mu_pair<P>(a, i, t & 1);
}

// ---------------------------------------------------------------- main role

// Hint decoding by one wave (verify.cu:52-93; spec unpack_sig): bits[k * 8 ..]
// = the 256-bit set of row k.  Returns false (wave-uniform) when the hint
// bytes break a rule: row ends ascending and at most omega, positions of a
// row strictly ascending, bytes after the last position zero.
template <class P>
__device__ __forceinline__ bool decode_hints(const uint8_t *h, uint32_t *bits) {
    const uint32_t lane = (uint32_t)lane_id();
    uint32_t end[P::K], prev = 0;
    bool bad = false;
#pragma unroll
    for (int k = 0; k < P::K; ++k) {
        end[k] = h[P::OMEGA + k];
        bad |= end[k] < prev || end[k] > (uint32_t)P::OMEGA;
        prev = end[k];
    }
    if (lane < P::K * 8) bits[lane] = 0;
    wave_lds_sync();
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        const uint32_t j = lane + 64 * half;
        if (j < (uint32_t)P::OMEGA) {
            const uint32_t idx = h[j], before = h[j ? j - 1 : 0];
            uint32_t row = 0, start = 0;
#pragma unroll
            for (int k = 0; k < P::K; ++k) {
                const bool past = end[k] <= j;
                row += past;
                start = past ? end[k] : start;
            }
            if (row < (uint32_t)P::K) {
                bad |= j > start && idx <= before;
                atomicOr(&bits[row * 8 + (idx >> 5)], 1u << (idx & 31));
            } else {
                bad |= idx != 0;
            }
        }
    }
    wave_lds_sync();
    return !wave_any(bad);
}

// z polynomial l of a signature: unpack, norm check, NTT (layout D).  Returns
// false (wave-uniform) when ||z|| >= gamma1 - beta.
template <class P>
__device__ __forceinline__ bool load_z_ntt(int32_t (&v)[4], const uint8_t *sig, int l, int32_t *x, const ZetaLds &zt) {
    using Z = Sizes<P>;
    uint32_t f[4];
    wave_fields_A<Z::Z_BITS>(f, sig + Z::SIG_Z + l * Z::POLYZ_BYTES);
    bool big = false;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        v[r] = P::GAMMA1 - (int32_t)f[r];
        big |= abs(v[r]) >= P::GAMMA1 - P::BETA;
    }
    if (wave_any(big)) return false;
    ntt_wave(v, x, zt);
    return true;
}

// w1' row k = UseHint(h, caddq(INTT(A z^ - c^ t1^ 2^d))), packed into the work row
template <class P>
__device__ __forceinline__ void finish_row(uint8_t *work, int k, int32_t (&w)[4], const int32_t (&c)[4],
                                           const int32_t (&t1)[4], const uint32_t *bits, int32_t *x,
                                           const ZetaLds &zt) {
    using Z = Sizes<P>;
    using VL = VerifyLayout<P>;
#pragma unroll
    for (int r = 0; r < 4; ++r) w[r] = reduce32(w[r] - mont_mul(c[r], t1[r]));
    intt_wave(w, x, zt);
    const int l = lane_id();
    int32_t w1[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int j = 64 * r + l;
        w1[r] = use_hint<P>(caddq(w[r]), (bits[k * 8 + (j >> 5)] >> (j & 31)) & 1);
    }
    layout_A_to_D(w1, x);
    uint32_t u[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) u[r] = (uint32_t)w1[r];
    wave_pack_D<Z::W1_BITS>(work + VL::HASH + CRHBYTES + k * Z::POLYW1_BYTES, u);
}

// one wave per workgroup: waves of the fold need no barriers
template <class P>
struct VfShared {
    ZetaLds zt;
    uint32_t bits[FoldCfg<P>::IPW][P::K * 8];
    uint32_t cp[FoldCfg<P>::IPW][16];  // challenge masks (OWN_C)
    union {
        FoldLds<P> f;                    // its windows double as the transforms' exchange buffer
        __align__(8) uint32_t mu[4 * ROW_LDS_WORDS];  // mu role
        struct {                         // sampling the challenges, before the rest
            uint32_t row[4 * ROW_LDS_WORDS];
            uint32_t chal[4 * CHALLENGE_ROW_WORDS];
        };
    };
    __device__ int32_t *x() {
        static_assert(sizeof(f.win) >= NTT_XBUF * 4, "the windows hold an exchange buffer");
        return &f.win[0][0];
    }
};

// OWN_C: the challenges are sampled here, one row of lanes per item
template <class P, int FORM, bool OWN_C>
__global__ __launch_bounds__(64) void vf_main_kernel(VerifyArgs a, uint32_t mu_blocks) {
    using Z = Sizes<P>;
    using VL = VerifyLayout<P>;
    constexpr int IPW = FoldCfg<P>::IPW, KL = P::K * P::L;
    __shared__ __align__(16) VfShared<P> sh;
    if (blockIdx.x < mu_blocks) return mu_role<P, FORM>(a, blockIdx.x, sh.mu);
    const int lane = lane_id();
    const size_t item0 = (size_t)(blockIdx.x - mu_blocks) * IPW;
    auto work_of = [&](size_t item) { return a.work + item * a.work_pitch; };
    zeta_lds_load(sh.zt);
    wave_lds_sync();
    if constexpr (OWN_C) {
        const RowLane r = row_lane_setup(sh.row, 0);
        const int i = lane >> 4;
        const bool run = i < IPW && item0 + i < a.n;
        const size_t item = run ? item0 + i : item0;
        uint32_t s[5];
#pragma unroll
        for (int x = 0; x < 5; ++x) {
            const uint32_t w = row_word(r, x);
            s[x] = r.active && w < 4 ? load_any<uint32_t>(a.sig + item * a.sig_pitch + 8 * w + 4 * r.h) : 0u;
            if (r.active && w == 4 && r.h == 0) s[x] = 0x1Fu;
            if (r.active && w == SHAKE256_RATE / 8 - 1 && r.h == 1) s[x] = 0x80000000u;
        }
        challenge_row<P::TAU>(s, sh.cp[run ? i : 0], r, sh.row, sh.chal + i * CHALLENGE_ROW_WORDS, run);
        wave_lds_sync();
    }

    // hints, z^; ok: bit i set when item i is still accepted (wave-uniform)
    uint32_t ok = 0;
#pragma unroll 1
    for (int i = 0; i < IPW; ++i) {
        const size_t item = item0 + i;
        if (item >= a.n) break;
        const uint8_t *sig = a.sig + item * a.sig_pitch;
        bool good = decode_hints<P>(sig + Z::SIG_H, sh.bits[i]);
#pragma unroll 1
        for (int l = 0; l < P::L && good; ++l) {
            int32_t v[4];
            good = load_z_ntt<P>(v, sig, l, sh.x(), sh.zt);
            if (good) wave_store_D(sh.f.row[i * P::K + l], v);
        }
        if (lane == 0) *reinterpret_cast<int32_t *>(work_of(item) + VL::FLAG) = good ? 0 : 1;
        ok |= (uint32_t)good << i;
    }
    if (ok == 0) return;

    {
        const int i = min(lane / KL, IPW - 1);
        const bool run = lane < IPW * KL && ((ok >> i) & 1u);
        const uint8_t *pk = a.pk + (run ? item0 + i : item0) * a.pk_pitch;
        uint64_t rho[4];
#pragma unroll
        for (int w = 0; w < 4; ++w) rho[w] = load_any<uint64_t>(pk + 8 * w);
        expand_fold<P>(sh.f, rho, run);
    }

#pragma unroll 1
    for (int i = 0; i < IPW; ++i) {
        if (!((ok >> i) & 1u)) continue;
        const size_t item = item0 + i;
        int32_t c[4];
        wave_load_challenge_A(c, OWN_C ? sh.cp[i] : reinterpret_cast<const uint32_t *>(work_of(item) + VL::CP));
        ntt_wave(c, sh.x(), sh.zt);
#pragma unroll 1
        for (int k = 0; k < P::K; ++k) {
            int32_t t1[4], w[4];
            uint32_t f[4];
            wave_fields_A<10>(f, a.pk + item * a.pk_pitch + SEEDBYTES + k * POLYT1_BYTES);
#pragma unroll
            for (int r = 0; r < 4; ++r) t1[r] = (int32_t)(f[r] << D);
            ntt_wave(t1, sh.x(), sh.zt);
            wave_load_D(w, sh.f.row[i * P::K + k]);
            finish_row<P>(work_of(item), k, w, c, t1, sh.bits[i], sh.x(), sh.zt);
        }
    }
}

// The smallest batches: a workgroup per item and row of A, a wave per entry.
// What ends such a call is the chain of one workgroup, in vf_main's form five
// lane permutations (9.6 us each) and the transforms of IPW items one after
// the other; here five wave permutations (2.3 us) and two transforms.  Every
// workgroup of an item checks and transforms z for itself.
template <class P>
struct VfSmallShared {
    ZetaLds zt;
    int32_t a[P::L][N], c[N], t1[N];
    int32_t x[P::L][NTT_XBUF];
    uint32_t wave[P::L][WAVE_LDS_WORDS + 2];
    uint32_t block[P::L][EXPAND_WAVE_WORDS];
    uint32_t chal[CHALLENGE_ROW_WORDS], cp[16], bits[P::K * 8];
    int fail;
};

template <class P>
__global__ __launch_bounds__(64 * P::L) void vf_small_kernel(VerifyArgs a, uint32_t mu_blocks) {
    using Z = Sizes<P>;
    using VL = VerifyLayout<P>;
    __shared__ __align__(16) VfSmallShared<P> sh;
    if (blockIdx.x < mu_blocks) {
        static_assert(sizeof(sh.a) >= 4 * P::L * WAVE_LDS_WORDS, "the mu role's waves");
        return mu_role<P, MU_WAVE>(a, blockIdx.x, reinterpret_cast<uint32_t *>(sh.a));
    }
    const uint32_t wave = threadIdx.x >> 6, b = blockIdx.x - mu_blocks, k = b % P::K;
    const size_t item = b / P::K;
    const uint8_t *sig = a.sig + item * a.sig_pitch, *pk = a.pk + item * a.pk_pitch;
    uint8_t *work = a.work + item * a.work_pitch;
    zeta_lds_load(sh.zt);
    if (threadIdx.x == 0) sh.fail = 0;
    __syncthreads();

    int32_t z[4];
    bool good = load_z_ntt<P>(z, sig, (int)wave, sh.x[wave], sh.zt);
    if (wave == 1) {
        good &= decode_hints<P>(sig + Z::SIG_H, sh.bits);
        uint32_t f[4];
        int32_t t1[4];
        wave_fields_A<10>(f, pk + SEEDBYTES + k * POLYT1_BYTES);
#pragma unroll
        for (int r = 0; r < 4; ++r) t1[r] = (int32_t)(f[r] << D);
        ntt_wave(t1, sh.x[wave], sh.zt);
        wave_store_D(sh.t1, t1);
    }
    if (!good && lane_id() == 0) sh.fail = 1;
    const WaveLane r = wave_lane_setup(sh.wave[wave], 0);
    if (wave == 0) {
        const uint64_t ct = r.w < 4 ? load_any<uint64_t>(sig + 8 * r.w) : 0ull;
        const uint32_t lo = r.w == 4 ? 0x1Fu : (uint32_t)ct;
        const uint32_t hi = r.w == SHAKE256_RATE / 8 - 1 ? 0x80000000u : (uint32_t)(ct >> 32);
        challenge_wave<P::TAU>(lo, hi, sh.cp, r, sh.wave[wave], sh.chal);
        wave_lds_sync();
        int32_t c[4];
        wave_load_challenge_A(c, sh.cp);
        ntt_wave(c, sh.x[wave], sh.zt);
        wave_store_D(sh.c, c);
    }
    expand_a_wave(sh.a[wave], pk, k << 8 | wave, r, sh.wave[wave], sh.block[wave]);
    int32_t av[4];
    wave_load_D(av, sh.a[wave]);
#pragma unroll
    for (int q = 0; q < 4; ++q) av[q] = mont_mul(av[q], z[q]);
    wave_store_D(sh.a[wave], av);
    __syncthreads();
    if (k == 0 && threadIdx.x == 0) *reinterpret_cast<int32_t *>(work + VL::FLAG) = sh.fail;
    if (wave != 0 || sh.fail) return;
    int32_t w[4] = {0, 0, 0, 0}, c[4], t1[4];
#pragma unroll
    for (int l = 0; l < P::L; ++l) {
        wave_load_D(av, sh.a[l]);
#pragma unroll
        for (int q = 0; q < 4; ++q) w[q] += av[q];
    }
    wave_load_D(c, sh.c);
    wave_load_D(t1, sh.t1);
    finish_row<P>(work, (int)k, w, c, t1, sh.bits, sh.x[0], sh.zt);
}

template <class P>
struct VfMainCfg {
    static constexpr int G = P::MODE == 2 ? 16 : (P::MODE == 3 ? 8 : 4);
};

// Resident keys: G items per workgroup (the compiled default VfMainCfg<P>::G,
// or the value a tiling chooses)
template <class P, int G>
struct VfResShared {
    ZetaLds zt;
    int32_t x[4][NTT_XBUF];
    int32_t zhat[G][P::L][N];
    int32_t chat[G][N];
    uint32_t bits[G][P::K * 8];
    int fail[G];
    uint32_t cp[G][16];                  // challenge masks (OWN_C)
    __align__(8) uint32_t mu[4 * 4 * ROW_LDS_WORDS];  // mu role
    uint32_t chal[16 * CHALLENGE_ROW_WORDS];
};

template <class P, int G, int FORM, bool OWN_C>
__global__ __launch_bounds__(256) void vf_res_kernel(VerifyArgs a, uint32_t mu_blocks) {
    using Z = Sizes<P>;
    using VL = VerifyLayout<P>;
    using KL = KeyLayout<P>;
    extern __shared__ __align__(16) uint8_t smem_raw[];
    VfResShared<P, G> &sh = *reinterpret_cast<VfResShared<P, G> *>(smem_raw);
    if (blockIdx.x < mu_blocks) return mu_role<P, FORM>(a, blockIdx.x, sh.mu);
    const size_t item0 = (size_t)(blockIdx.x - mu_blocks) * G;
    const int wave = threadIdx.x >> 6, lane = lane_id();
    zeta_lds_load(sh.zt);
    if constexpr (OWN_C) {
        static_assert(G <= 16, "a row of lanes per item");
        if (wave * 4 < G) {
            const RowLane r = row_lane_setup(sh.mu, wave * 4 * ROW_LDS_WORDS);
            const int g = threadIdx.x >> 4;
            const bool run = g < G && item0 + g < a.n;
            const size_t item = run ? item0 + g : item0;
            uint32_t s[5];
#pragma unroll
            for (int x = 0; x < 5; ++x) {
                const uint32_t w = row_word(r, x);
                s[x] = r.active && w < 4 ? load_any<uint32_t>(a.sig + item * a.sig_pitch + 8 * w + 4 * r.h) : 0u;
                if (r.active && w == 4 && r.h == 0) s[x] = 0x1Fu;
                if (r.active && w == SHAKE256_RATE / 8 - 1 && r.h == 1) s[x] = 0x80000000u;
            }
            challenge_row<P::TAU>(s, sh.cp[run ? g : 0], r, sh.mu, sh.chal + g * CHALLENGE_ROW_WORDS, run);
        }
    }
    // a wave per item: hints, and whether its key is in the store
    for (int g = wave; g < G; g += 4) {
        const size_t item = item0 + g;
        bool good = item < a.n && a.key_idx[item] < a.nkeys;
        if (good) good = decode_hints<P>(a.sig + item * a.sig_pitch + Z::SIG_H, sh.bits[g]);
        if (lane == 0) sh.fail[g] = good ? 0 : 1;
    }
    __syncthreads();

    // z: unpack, ||z|| < gamma1 - beta, NTT (verify.cu:96-126); NTT(c)
    for (int t = wave; t < G * (P::L + 1); t += 4) {
        const int g = t / (P::L + 1), l = t % (P::L + 1);
        const size_t item = item0 + g;
        if (*(volatile int *)&sh.fail[g]) continue;
        int32_t v[4];
        if (l < P::L) {
            if (load_z_ntt<P>(v, a.sig + item * a.sig_pitch, l, sh.x[wave], sh.zt))
                wave_store_D(sh.zhat[g][l], v);
            else if (lane == 0)
                sh.fail[g] = 1;
        } else {
            wave_load_challenge_A(
                v, OWN_C ? sh.cp[g] : reinterpret_cast<const uint32_t *>(a.work + item * a.work_pitch + VL::CP));
            ntt_wave(v, sh.x[wave], sh.zt);
            wave_store_D(sh.chat[g], v);
        }
    }
    __syncthreads();
    if (threadIdx.x < G && item0 + threadIdx.x < a.n)
        *reinterpret_cast<int32_t *>(a.work + (item0 + threadIdx.x) * a.work_pitch + VL::FLAG) = sh.fail[threadIdx.x];

    for (int t = wave; t < G * P::K; t += 4) {
        const int g = t / P::K, k = t % P::K;
        const size_t item = item0 + g;
        if (sh.fail[g]) continue;
        // A z^ from the stored A; the 64-bit sums are reduced once
        const uint8_t *key = a.keys + a.key_idx[item] * a.key_pitch;
        const int32_t *mat = reinterpret_cast<const int32_t *>(key + KL::MAT);
        int64_t sum[4] = {0, 0, 0, 0};
#pragma unroll
        for (int l = 0; l < P::L; ++l) {
            int32_t av[4], zv[4];
            wave_load_D(av, mat + (k * P::L + l) * N);
            wave_load_D(zv, sh.zhat[g][l]);
#pragma unroll
            for (int r = 0; r < 4; ++r) sum[r] += (int64_t)av[r] * zv[r];
        }
        int32_t t1[4], w[4], c[4];
        wave_load_D(t1, reinterpret_cast<const int32_t *>(key + KL::T1H) + k * N);
        wave_load_D(c, sh.chat[g]);
#pragma unroll
        for (int r = 0; r < 4; ++r) w[r] = mont_reduce(sum[r]);
        finish_row<P>(a.work + item * a.work_pitch, k, w, c, t1, sh.bits[g], sh.x[wave], sh.zt);
    }
}

// lanes per hash
enum FinalForm { FINAL_LANE = 1, FINAL_PAIR = 2, FINAL_ROW = 16, FINAL_WAVE = 64 };

// c~' = SHAKE256(mu || w1')[0:32] against c~, one wave / row / pair / lane per item
template <class P, int FORM>
__global__ __launch_bounds__(256) void vf_final_kernel(VerifyArgs a) {
    using Z = Sizes<P>;
    using VL = VerifyLayout<P>;
    __shared__ __align__(8) uint32_t
        lds[FORM == FINAL_WAVE ? 4 * WAVE_LDS_WORDS : FORM == FINAL_ROW ? 4 * 4 * ROW_LDS_WORDS : 1];
    constexpr int PER = FORM;
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x, i = t / PER;
    RowLane r;
    if constexpr (FORM == FINAL_ROW) r = row_lane_setup(lds, (threadIdx.x >> 6) * 4 * ROW_LDS_WORDS);
    if (i >= a.n) return;
    const uint8_t *work = a.work + i * a.work_pitch;
    int32_t *ret = a.ret + i * a.ret_pitch;
    if (*reinterpret_cast<const int32_t *>(work + VL::FLAG) != 0) {
        if (t % PER == 0) *ret = -1;
        if constexpr (FORM != FINAL_ROW) return;  // a row's lanes stay for the DPP of the others
    }
    const uint8_t *sig = a.sig + i * a.sig_pitch;
    const uint32_t *hin = reinterpret_cast<const uint32_t *>(work + VL::HASH);
    if constexpr (FORM == FINAL_WAVE) {
        const WaveLane wl = wave_lane_setup(lds, (threadIdx.x >> 6) * WAVE_LDS_WORDS);
        uint32_t lo, hi;
        shake_wave<SHAKE256_RATE>(lo, hi, wl, lds, Z::CHASH_IN_BYTES,
                                  [&](uint32_t w) { return hin[2 * w] | (uint64_t)hin[2 * w + 1] << 32; });
        const bool diff = wl.main && wl.w < 4 &&
                          (lo | (uint64_t)hi << 32) != load_any<uint64_t>(sig + 8 * wl.w);
        const bool bad = wave_any(diff);
        if (lane_id() == 0) *ret = bad ? -1 : 0;
    } else if constexpr (FORM == FINAL_ROW) {
        uint32_t s[5];
        shake_row<SHAKE256_RATE>(s, r, lds, Z::CHASH_IN_BYTES, [&](uint32_t w) { return hin[2 * w + r.h]; });
        bool diff = false;
#pragma unroll
        for (int x = 0; x < 4; ++x)
            if (r.active && r.y == 0) diff |= s[x] != load_any<uint32_t>(sig + 8 * x + 4 * r.h);
        const uint64_t rows = __ballot(diff);
        if (t % PER == 0 && *reinterpret_cast<const int32_t *>(work + VL::FLAG) == 0)
            *ret = (rows >> (lane_id() & 48) & 0xFFFFull) == 0 ? 0 : -1;
    } else if constexpr (FORM == FINAL_PAIR) {
        const uint32_t h = t & 1;
        uint32_t s[25];
        shake_absorb_pair<SHAKE256_RATE, Z::CHASH_IN_BYTES>(s, [&](uint32_t w) { return hin[2 * w + h]; }, h);
        keccak_f1600_pair(s, h);
        uint32_t diff = 0;
#pragma unroll
        for (int w = 0; w < 4; ++w) diff |= s[w] ^ load_any<uint32_t>(sig + 8 * w + 4 * h);
        diff |= pair_other(diff);
        if (h == 0) *ret = diff == 0 ? 0 : -1;
    } else {
        const uint64_t *hw = reinterpret_cast<const uint64_t *>(hin);
        Lane64 s[25];
        shake_absorb<SHAKE256_RATE>(s, [&](uint32_t w, uint32_t) { return hw[w]; }, (uint32_t)Z::CHASH_IN_BYTES);
        uint64_t c2[4];
        squeeze_words<4>(s, c2);
        uint64_t diff = 0;
#pragma unroll
        for (int w = 0; w < 4; ++w) diff |= c2[w] ^ load_any<uint64_t>(sig + 8 * w);
        *ret = diff == 0 ? 0 : -1;
    }
}

// The values a tiling may choose; they stayed as they were when the kernel's
// LDS shrank, so a recorded or refused value stays so.
template <class P, int G>
constexpr bool vf_fits() {
    return G * (P::L + P::K + 1) * N * 4 + 8 * 1024 <= 160 * 1024;
}

template <class P, int G>
static int launch_vf_res_g(const VerifyArgs &a, bool row, bool own_c, hipStream_t st) {
    if constexpr (!vf_fits<P, G>()) {
        return -1;
    } else {
        constexpr size_t smem = sizeof(VfResShared<P, G>);
        static_assert(smem <= 160 * 1024, "the LDS of a CU");
        auto go = [&](auto kernel, uint32_t per) {
            if (smem > 64 * 1024) {
                const hipError_t attr = hipFuncSetAttribute((const void *)kernel,
                                                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
                if (attr != hipSuccess) return (int)attr;
            }
            const uint32_t mu = (uint32_t)((a.n + per - 1) / per);
            hipLaunchKernelGGL(kernel, dim3(mu + (unsigned)((a.n + G - 1) / G)), dim3(256), smem, st, a, mu);
            return (int)hipGetLastError();
        };
        if (wave_hashes(a)) return go(vf_res_kernel<P, G, MU_WAVE, true>, mu_items<MU_WAVE>(256));
        if (own_c) return go(vf_res_kernel<P, G, MU_ROW, true>, mu_items<MU_ROW>(256));
        if (row) return go(vf_res_kernel<P, G, MU_ROW, false>, mu_items<MU_ROW>(256));
        return go(vf_res_kernel<P, G, MU_PAIR, false>, mu_items<MU_PAIR>(256));
    }
}

template <class P>
static int launch_vf_res(const VerifyArgs &a, bool row, bool own_c, hipStream_t st) {
    switch (tiling_get(TILE_VERIFY_ITEMS, P::MODE, a.n)) {
        case 2: return launch_vf_res_g<P, 2>(a, row, own_c, st);
        case 4: return launch_vf_res_g<P, 4>(a, row, own_c, st);
        case 8: return launch_vf_res_g<P, 8>(a, row, own_c, st);
        case 16: return launch_vf_res_g<P, 16>(a, row, own_c, st);
        default: return launch_vf_res_g<P, VfMainCfg<P>::G>(a, row, own_c, st);
    }
}

template <class P>
static int launch_vf_main(const VerifyArgs &a, bool row, bool own_c, hipStream_t st) {
    constexpr int IPW = FoldCfg<P>::IPW;
    if (a.n * P::K * P::L <= VERIFY_SMALL_WAVES) {
        const uint32_t mu = (uint32_t)((a.n + P::L - 1) / P::L);
        hipLaunchKernelGGL(vf_small_kernel<P>, dim3(mu + (unsigned)a.n * P::K), dim3(64 * P::L), 0, st, a, mu);
        return (int)hipGetLastError();
    }
    const bool wave = wave_hashes(a);
    const uint32_t per = wave ? mu_items<MU_WAVE>(64) : row ? mu_items<MU_ROW>(64) : mu_items<MU_PAIR>(64);
    const uint32_t mu = (uint32_t)((a.n + per - 1) / per);
    const dim3 grid(mu + (unsigned)((a.n + IPW - 1) / IPW));
    if (wave)
        hipLaunchKernelGGL((vf_main_kernel<P, MU_WAVE, true>), grid, dim3(64), 0, st, a, mu);
    else if (own_c)
        hipLaunchKernelGGL((vf_main_kernel<P, MU_ROW, true>), grid, dim3(64), 0, st, a, mu);
    else if (row)
        hipLaunchKernelGGL((vf_main_kernel<P, MU_ROW, false>), grid, dim3(64), 0, st, a, mu);
    else
        hipLaunchKernelGGL((vf_main_kernel<P, MU_PAIR, false>), grid, dim3(64), 0, st, a, mu);
    return (int)hipGetLastError();
}

template <class P>
static bool verify_items_ok(int g) {
    switch (g) {
        case 0: return true;
        case 2: return vf_fits<P, 2>();
        case 4: return vf_fits<P, 4>();
        case 8: return vf_fits<P, 8>();
        case 16: return vf_fits<P, 16>();
        default: return false;
    }
}

bool verify_items_supported(int mode, int g) {
    switch (mode) {
        case 2: return verify_items_ok<Params<2>>(g);
        case 3: return verify_items_ok<Params<3>>(g);
        case 5: return verify_items_ok<Params<5>>(g);
        default: return false;
    }
}

template <class P>
static int verify_impl(const VerifyArgs &a, hipStream_t st, hipEvent_t *ev) {
    if (a.n == 0) return 0;
    int e;
    const bool small = a.n <= VERIFY_ROW_MAX, row = a.row_mu || small;
    if (ev && (e = (int)hipEventRecord(ev[0], st))) return e;
    if (!small) {
        hipLaunchKernelGGL(vf_prep_kernel<P>, dim3((unsigned)((a.n + 255) / 256)), dim3(256), 0, st, a);
        if ((e = (int)hipGetLastError())) return e;
    }
    if (ev && (e = (int)hipEventRecord(ev[1], st))) return e;
    e = a.key_idx ? launch_vf_res<P>(a, row, small, st) : launch_vf_main<P>(a, row, small, st);
    if (e) return e;
    if (ev && (e = (int)hipEventRecord(ev[2], st))) return e;
    auto blocks = [&](size_t per) { return dim3((unsigned)((a.n * per + 255) / 256)); };
    if (wave_hashes(a))
        hipLaunchKernelGGL((vf_final_kernel<P, FINAL_WAVE>), blocks(64), dim3(256), 0, st, a);
    else if (small)
        hipLaunchKernelGGL((vf_final_kernel<P, FINAL_ROW>), blocks(16), dim3(256), 0, st, a);
    else if (a.n <= VERIFY_PAIR_MAX)
        hipLaunchKernelGGL((vf_final_kernel<P, FINAL_PAIR>), blocks(2), dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL((vf_final_kernel<P, FINAL_LANE>), blocks(1), dim3(256), 0, st, a);
    if (ev && (e = (int)hipEventRecord(ev[3], st))) return e;
    return (int)hipGetLastError();
}

int launch_verify(int mode, const VerifyArgs &a, hipStream_t st, hipEvent_t *ev) {
    switch (mode) {
        case 2: return verify_impl<Params<2>>(a, st, ev);
        case 3: return verify_impl<Params<3>>(a, st, ev);
        case 5: return verify_impl<Params<5>>(a, st, ev);
        default: return -1;
    }
}

}  // namespace dil
