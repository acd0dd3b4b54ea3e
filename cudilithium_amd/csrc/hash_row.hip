// Message hashing with one sponge per 16-lane row (keccak_row.hpp), for
// batches of long messages, where the serial absorb of the longest message
// (floor((32 + mlen) / 136) + 1 permutations) sets the batch's latency.
//
//   vf_mu_row   tr = SHAKE256(pk) (or the resident key's) and
//               mu = SHAKE256(tr || m) into the verify work row, before
//               vf_prep (verify.cu:130-144), which then skips them
//
// Four items per wavefront, sixteen per 256-thread workgroup.
#include <hip/hip_runtime.h>

#include "hash_row.hpp"
#include "internal.hpp"
#include "layout.hpp"
#include "pipelines.hpp"
#include "sign_stages.hpp"

namespace dil {

template <class P>
__global__ __launch_bounds__(256) void vf_mu_row_kernel(VerifyArgs a) {
    using Z = Sizes<P>;
    using VL = VerifyLayout<P>;
    __shared__ uint32_t lds[4 * 4 * ROW_LDS_WORDS];
    __builtin_amdgcn_s_setprio(3);
    const uint32_t wave = threadIdx.x >> 6;
    const RowLane r = row_lane_setup(lds, wave * 4 * ROW_LDS_WORDS);
    const size_t i = (size_t)blockIdx.x * ROW_ITEMS_PER_BLOCK + wave * 4 + ((uint32_t)lane_id() >> 4);
    if (i >= a.n) return;
    if (a.key_idx && a.key_idx[i] >= a.nkeys) return;  // vf_prep rejects the item
    const uint32_t h = r.h;
    const RowShare sh{wave * 4 * ROW_LDS_WORDS + ((uint32_t)lane_id() >> 4) * ROW_LDS_WORDS};
    uint32_t s[5];
    const uint8_t *key = a.key_idx ? a.keys + a.key_idx[i] * a.key_pitch : nullptr;
    if (!key) {
        // tr = SHAKE256(pk)[0:32]
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

template <class P>
static int verify_mu_row_impl(const VerifyArgs &a, hipStream_t st) {
    if (a.n == 0) return 0;
    hipLaunchKernelGGL(vf_mu_row_kernel<P>, dim3((unsigned)((a.n + ROW_ITEMS_PER_BLOCK - 1) / ROW_ITEMS_PER_BLOCK)),
                       dim3(256), 0, st, a);
    return (int)hipGetLastError();
}

int launch_verify_mu_row(int mode, const VerifyArgs &a, hipStream_t st) {
    switch (mode) {
        case 2: return verify_mu_row_impl<Params<2>>(a, st);
        case 3: return verify_mu_row_impl<Params<3>>(a, st);
        case 5: return verify_mu_row_impl<Params<5>>(a, st);
        default: return -1;
    }
}

}  // namespace dil
