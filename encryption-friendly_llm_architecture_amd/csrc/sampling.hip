// Key and encryption samplers as kernels of their own (the streams: sampling.h).
#include "hemm_internal.hpp"
#include "sampling.h"

namespace {

struct KeyList {
    u64 key[HEMM_MAX_PRIMES];
};

// out[limb][i] uniform in [0, q_limb)
__global__ __launch_bounds__(256) void sample_uniform_kernel(KeyList keys, LimbList ll, const ModQ *__restrict__ modq,
                                                             u64 *__restrict__ out, int logN) {
    const int limb = blockIdx.y;
    const u64 i = (u64)blockIdx.x * 256 + threadIdx.x;
    out[((size_t)limb << logN) + i] = sample_uniform(keys.key[limb], i, modq[table_byte(ll.idx, limb)]);
}

// out[limb][i] = e_i mod q_limb for the centred-binomial error e of stream `key`
__global__ __launch_bounds__(256) void sample_error_kernel(u64 key, LimbList ll, const ModQ *__restrict__ modq,
                                                           u64 *__restrict__ out, int logN) {
    const int limb = blockIdx.y;
    const u64 i = (u64)blockIdx.x * 256 + threadIdx.x;
    const u64 q = modq[table_byte(ll.idx, limb)].q;
    const int e = sample_error(key, i);
    out[((size_t)limb << logN) + i] = e >= 0 ? (u64)e : q - (u64)(-e);
}

}  // namespace

void launch_sample_uniform(const hemm_context *c, const u64 *stream_keys, const LimbList &ll, int n_limbs, u64 *out,
                           hipStream_t s) {
    KeyList kl;
    for (int j = 0; j < n_limbs; j++) kl.key[j] = stream_keys[j];
    dim3 grid(c->N / 256, n_limbs), block(256);
    hipLaunchKernelGGL(sample_uniform_kernel, grid, block, 0, s, kl, ll, c->d_modq, out, c->logN);
}

void launch_sample_error(const hemm_context *c, u64 stream_key, const LimbList &ll, int n_limbs, u64 *out, hipStream_t s) {
    dim3 grid(c->N / 256, n_limbs), block(256);
    hipLaunchKernelGGL(sample_error_kernel, grid, block, 0, s, stream_key, ll, c->d_modq, out, c->logN);
}
