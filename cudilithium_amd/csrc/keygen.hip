// Batched key generation (reference: gpu_keypair, src/keypair.cu:35-311, one
// 32-lane warp per key with ExpandA streamed through shared memory).
//
// Four launches, each with the lane mapping its work wants:
//   kg_seed   lane per key     seed (explicit or SHAKE128(le64(ctr))), then
//                              rho | rhoprime | key = SHAKE256(seed)
//   kg_eta    lane per s-poly  ExpandS, packed into sk
//   kg_main   one wave per FoldCfg<P>::IPW keys: NTT(s1), A s1^ straight from
//             the sponges (fold.hpp), then per row INTT, + s2, caddq,
//             Power2Round and packing of t1 / t0
//   kg_tr     tr = SHAKE256(pk)[0:32], a wave, a 16-lane row or a lane pair
//             per key
#include <hip/hip_runtime.h>

#include "fold.hpp"
#include "hash_row.hpp"
#include "internal.hpp"
#include "layout.hpp"
#include "pipelines.hpp"
#include "poly.hpp"
#include "sample.hpp"

namespace dil {

template <class P>
__global__ __launch_bounds__(256) void kg_seed_kernel(KeygenArgs a) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    uint64_t seed[4];
    Lane64 s[25];
    if (a.seeds) {
        const uint8_t *sp = a.seeds + i * a.seed_pitch;
#pragma unroll
        for (int w = 0; w < 4; ++w) seed[w] = load_le64(sp + 8 * w);
    } else {
        // keypair.cu:50-60: seed = SHAKE128(le64(rand_index + 2i + 1))[0:32]
        const uint64_t in[1] = {(uint64_t)a.rand_index + 2 * (uint64_t)i + 1};
        shake_absorb_regs<SHAKE128_RATE, 8>(s, in);
        squeeze_words<4>(s, seed);
    }
    uint64_t out[16];
    shake_absorb_regs<SHAKE256_RATE, SEEDBYTES>(s, seed);
    squeeze_words<16>(s, out);
    uint8_t *pk = a.pk + i * a.pk_pitch;
    uint8_t *sk = a.sk + i * a.sk_pitch;
    uint8_t *rp = a.scratch + i * a.scratch_pitch + KeypairLayout<P>::RHOPRIME - KeypairLayout<P>::SCRATCH;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        store_any<uint64_t>(pk + 8 * w, out[w]);
        store_any<uint64_t>(sk + 8 * w, out[w]);
        store_any<uint64_t>(sk + SEEDBYTES + 8 * w, out[12 + w]);
    }
#pragma unroll
    for (int w = 0; w < 8; ++w) store_any<uint64_t>(rp + 8 * w, out[4 + w]);
}

// ExpandS, lane per polynomial (keypair.cu:80-130), one wave per workgroup.
// Each lane writes every nibble to the next free byte of its LDS row and moves
// on only past an accepted one, so a nibble costs a field extract, a byte
// store, a compare and an add, with no branch.  The accepted nibbles are then
// packed a row at a time by the whole wave: eta - s is the nibble itself
// (eta 4) or the nibble mod 5 (eta 2).  16,384 Dilithium3 keys: 178 us when
// each lane branched per nibble and stored its own row, 96 us now.
constexpr int ETA_ROW = N + 4;  // bytes; an odd number of words apart
template <class P>
__global__ __launch_bounds__(64) void kg_eta_kernel(KeygenArgs a) {
    using Z = Sizes<P>;
    constexpr uint32_t NP = P::L + P::K, BOUND = P::ETA == 2 ? 15 : 9;
    __shared__ __align__(16) uint8_t rows[64 * ETA_ROW];
    const size_t t0 = (size_t)blockIdx.x * 64, total = a.n * NP;
    const int lane = lane_id();
    {
        const size_t t = min(t0 + lane, total - 1);
        const uint8_t *rp = a.scratch + t / NP * a.scratch_pitch + KeypairLayout<P>::RHOPRIME - KeypairLayout<P>::SCRATCH;
        Lane64 s[25];
        uint64_t in[9];
#pragma unroll
        for (int w = 0; w < 8; ++w) in[w] = load_any<uint64_t>(rp + 8 * w);
        in[8] = t % NP;  // nonce l for s1[l], L + k for s2[k] (keypair.cu:84-89, 202-207)
        shake_absorb_regs<SHAKE256_RATE, CRHBYTES + 2>(s, in);
        uint8_t *row = rows + lane * ETA_ROW;
        uint32_t ctr = 0;
#pragma unroll 1
        while (__ballot(ctr < N)) {
            keccak_f1600(s);
            static_for<0, 2 * (SHAKE256_RATE / 8)>([&](auto h) {
                if (__ballot(ctr < N) == 0ull) return;
                const uint32_t w = half_word<decltype(h)::value>(s);
#pragma unroll
                for (int b = 0; b < 8; ++b) {
                    const uint32_t v = (w >> (4 * b)) & 15u;
                    row[min(ctr, (uint32_t)N)] = (uint8_t)v;
                    ctr += v < BOUND;
                }
            });
        }
    }
    wave_lds_sync();
    const int count = (int)min((size_t)64, total - t0);
#pragma unroll 4
    for (int r = 0; r < count; ++r) {
        const size_t t = t0 + r;
        uint8_t *dst = a.sk + t / NP * a.sk_pitch + Z::SK_S1 + t % NP * Z::POLYETA_BYTES;
        const uint32_t d = reinterpret_cast<const uint32_t *>(rows + r * ETA_ROW)[lane];
        if constexpr (P::ETA == 4) {
            const uint32_t x = d | d >> 4;
            store_any<uint16_t>(dst + 2 * lane, (uint16_t)((x & 0xFFu) | (x >> 8 & 0xFF00u)));
        } else {
            // per byte: minus 5 for v >= 5 and again for v >= 10
            const uint32_t m = d - 5u * ((((d + 0x7B7B7B7Bu) >> 7) & 0x01010101u) + (((d + 0x76767676u) >> 7) & 0x01010101u));
            const uint32_t f = (m & 7u) | (m >> 5 & 7u << 3) | (m >> 10 & 7u << 6) | (m >> 15 & 7u << 9);
            const uint32_t v = f | pair_other(f) << 12;
            if ((lane & 1) == 0) {
                store_any<uint16_t>(dst + 3 * (lane >> 1), (uint16_t)v);
                dst[3 * (lane >> 1) + 2] = (uint8_t)(v >> 16);
            }
        }
    }
}

// one wave per workgroup: waves of the fold need no barriers
template <class P>
struct KgShared {
    ZetaLds zt;
    FoldLds<P> f;  // its windows double as the transforms' exchange buffer
    __device__ int32_t *x() {
        static_assert(sizeof(f.win) >= NTT_XBUF * 4, "the windows hold an exchange buffer");
        return &f.win[0][0];
    }
};

template <class P>
__global__ __launch_bounds__(64) void kg_main_kernel(KeygenArgs a) {
    using Z = Sizes<P>;
    constexpr int IPW = FoldCfg<P>::IPW;
    __shared__ __align__(16) KgShared<P> sh;
    const size_t item0 = (size_t)blockIdx.x * IPW;
    const int lane = lane_id(), count = (int)min((size_t)IPW, a.n - item0);
    // polynomial p of s1 | s2, packed in the secret key as eta - s
    auto load_s = [&](int32_t (&v)[4], int i, int p) {
        uint32_t f[4];
        wave_fields_A<Z::ETA_BITS>(f, a.sk + (item0 + i) * a.sk_pitch + Z::SK_S1 + p * Z::POLYETA_BYTES);
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = P::ETA - (int32_t)f[r];
    };
    zeta_lds_load(sh.zt);
    wave_lds_sync();

#pragma unroll 1
    for (int t = 0; t < count * P::L; ++t) {
        const int i = t / P::L, l = t % P::L;
        int32_t v[4];
        load_s(v, i, l);
        ntt_wave(v, sh.x(), sh.zt);
        wave_store_D(sh.f.row[i * P::K + l], v);
    }

    {
        const int i = lane / (P::K * P::L);
        const bool run = i < count;
        const uint8_t *pk = a.pk + (item0 + (run ? i : 0)) * a.pk_pitch;
        uint64_t rho[4];
#pragma unroll
        for (int w = 0; w < 4; ++w) rho[w] = load_any<uint64_t>(pk + 8 * w);
        expand_fold<P>(sh.f, rho, run);
    }

    // t = INTT(reduce32(t^)) + s2, caddq, Power2Round, pack (keypair.cu:251-301)
#pragma unroll 1
    for (int t = 0; t < count * P::K; ++t) {
        const int i = t / P::K, k = t % P::K;
        const size_t item = item0 + i;
        int32_t v[4];
        wave_load_D(v, sh.f.row[t]);
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = reduce32(v[r]);
        intt_wave(v, sh.x(), sh.zt);
        int32_t s2v[4], t1[4], t0[4];
        load_s(s2v, i, P::L + k);
#pragma unroll
        for (int r = 0; r < 4; ++r) t1[r] = power2round(caddq(v[r] + s2v[r]), t0[r]);
        layout_A_to_D(t1, sh.x());
        layout_A_to_D(t0, sh.x());
        uint32_t f1[4], f0[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            f1[r] = (uint32_t)t1[r];
            f0[r] = (uint32_t)((1 << (D - 1)) - t0[r]);
        }
        wave_pack_D<10>(a.pk + item * a.pk_pitch + SEEDBYTES + k * POLYT1_BYTES, f1);
        wave_pack_D<13>(a.sk + item * a.sk_pitch + Z::SK_T0 + k * POLYT0_BYTES, f0);
    }
}

// tr = SHAKE256(pk)[0:32] with one 16-lane row per key: for batches whose
// rows all find a place on the card, where the serial absorb of the public
// key (10 / 15 / 20 permutations) is the latency
template <class P>
__global__ __launch_bounds__(256) void kg_tr_row_kernel(KeygenArgs a) {
    using Z = Sizes<P>;
    __shared__ uint32_t lds[4 * 4 * ROW_LDS_WORDS];
    const RowLane r = row_lane_setup(lds, (threadIdx.x >> 6) * 4 * ROW_LDS_WORDS);
    const size_t i = (size_t)blockIdx.x * ROW_ITEMS_PER_BLOCK + (threadIdx.x >> 4);
    if (i >= a.n) return;  // whole rows
    const uint8_t *pk = a.pk + i * a.pk_pitch;
    uint32_t s[5];
    shake_row<SHAKE256_RATE>(s, r, lds, (uint32_t)Z::PK_BYTES,
                             [&](uint32_t w) { return load_half_bytes(pk, 8 * w + 4 * r.h, Z::PK_BYTES); });
    uint8_t *tr = a.sk + i * a.sk_pitch + Z::SK_TR;
    if (r.active && r.y == 0)
#pragma unroll
        for (int x = 0; x < 4; ++x) store_any<uint32_t>(tr + 8 * x + 4 * r.h, s[x]);
}

// ... and with a wave per key for the smallest batches
template <class P>
__global__ __launch_bounds__(256) void kg_tr_wave_kernel(KeygenArgs a) {
    using Z = Sizes<P>;
    __shared__ __align__(8) uint32_t lds[4 * WAVE_LDS_WORDS];
    const WaveLane r = wave_lane_setup(lds, (threadIdx.x >> 6) * WAVE_LDS_WORDS);
    const size_t i = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (i >= a.n) return;  // whole waves
    const uint8_t *pk = a.pk + i * a.pk_pitch;
    uint32_t lo, hi;
    shake_wave<SHAKE256_RATE>(lo, hi, r, lds, (uint32_t)Z::PK_BYTES,
                              [&](uint32_t w) { return load_word_bytes(pk, 8 * w, Z::PK_BYTES); });
    if (r.main && r.w < 4) store_any<uint64_t>(a.sk + i * a.sk_pitch + Z::SK_TR + 8 * r.w, lo | (uint64_t)hi << 32);
}

// tr = SHAKE256(pk)[0:32] with two lanes per key (keccak_f1600_pair): the
// serial absorb of the public key (10 / 15 / 20 permutations) is 2/3 as long
template <class P>
__global__ __launch_bounds__(256) void kg_tr_pair_kernel(KeygenArgs a) {
    using Z = Sizes<P>;
    const size_t i = (size_t)blockIdx.x * 128 + (threadIdx.x >> 1);
    const uint32_t h = threadIdx.x & 1;
    if (i >= a.n) return;  // both lanes of a pair
    const uint8_t *pk = a.pk + i * a.pk_pitch;
    uint32_t s[25];
    shake_pair<SHAKE256_RATE>(s, h, (uint32_t)Z::PK_BYTES,
                              [&](uint32_t w) { return load_half_bytes(pk, 8 * w + 4 * h, Z::PK_BYTES); });
    uint8_t *tr = a.sk + i * a.sk_pitch + Z::SK_TR;
#pragma unroll
    for (int w = 0; w < 4; ++w) store_any<uint32_t>(tr + 8 * w + 4 * h, s[w]);
}

// Keys-per-workgroup values that the tiling setter accepts (a wave's keys are
// fixed now; recorded tilings keep loading).
template <class P, int G>
constexpr bool kg_fits() {
    return G * (P::L + P::K) * N * 4 + 8 * 1024 <= 160 * 1024;
}

// tr with a wave per key, with a row per key, beyond that with lane pairs.
// Whole calls, row / wave: 10 Dilithium5 keys 206 / 173 us, 1,000 Dilithium3
// 199 / 175, 3,000 Dilithium3 236 / 229, 4,000 Dilithium5 393 / 396; pair /
// row: 6,000 Dilithium3 402 / 372, 8,000 Dilithium5 651 / 613, 10,000
// Dilithium2 366 / 370.
constexpr size_t KEYGEN_WAVE_MAX = 3072, KEYGEN_ROW_MAX = 8192;

template <class P>
static int keygen_impl(const KeygenArgs &a, hipStream_t st) {
    if (a.n == 0) return 0;
    constexpr int NP = P::L + P::K;
    const unsigned b1 = (unsigned)((a.n + 255) / 256);
    hipLaunchKernelGGL(kg_seed_kernel<P>, dim3(b1), dim3(256), 0, st, a);
    hipLaunchKernelGGL(kg_eta_kernel<P>, dim3((unsigned)((a.n * NP + 63) / 64)), dim3(64), 0, st, a);
    constexpr int IPW = FoldCfg<P>::IPW;
    hipLaunchKernelGGL(kg_main_kernel<P>, dim3((unsigned)((a.n + IPW - 1) / IPW)), dim3(64), 0, st, a);
    if (a.n <= KEYGEN_WAVE_MAX)
        hipLaunchKernelGGL(kg_tr_wave_kernel<P>, dim3((unsigned)((a.n + 3) / 4)), dim3(256), 0, st, a);
    else if (a.n <= KEYGEN_ROW_MAX)
        hipLaunchKernelGGL(kg_tr_row_kernel<P>, dim3((unsigned)((a.n + ROW_ITEMS_PER_BLOCK - 1) / ROW_ITEMS_PER_BLOCK)),
                           dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL(kg_tr_pair_kernel<P>, dim3((unsigned)((a.n + 127) / 128)), dim3(256), 0, st, a);
    return (int)hipGetLastError();
}

template <class P>
static bool keygen_items_ok(int g) {
    switch (g) {
        case 0: return true;
        case 2: return kg_fits<P, 2>();
        case 4: return kg_fits<P, 4>();
        case 8: return kg_fits<P, 8>();
        case 16: return kg_fits<P, 16>();
        default: return false;
    }
}

bool keygen_items_supported(int mode, int g) {
    switch (mode) {
        case 2: return keygen_items_ok<Params<2>>(g);
        case 3: return keygen_items_ok<Params<3>>(g);
        case 5: return keygen_items_ok<Params<5>>(g);
        default: return false;
    }
}

int launch_keygen(int mode, const KeygenArgs &a, hipStream_t st) {
    switch (mode) {
        case 2: return keygen_impl<Params<2>>(a, st);
        case 3: return keygen_impl<Params<3>>(a, st);
        case 5: return keygen_impl<Params<5>>(a, st);
        default: return -1;
    }
}

}  // namespace dil
