// Counter-based samplers on the device.  Every value is a pure function of (stream key, coefficient index):
//   sm64(x)          = splitmix64 finaliser of x + 0x9E3779B97F4A7C15
//   draw(key, i)     = sm64(key + i * 0x9E3779B97F4A7C15)
//   uniform mod q    : attempt t = 0, 1, ... draws draw(sm64(key + t), i) masked to the bit length of q and is
//                      accepted when below q (masked rejection: exactly uniform)
//   error            : centred binomial, popcount of bits 0..20 minus popcount of bits 21..41 of draw(key, i)
// so host code, the CPU oracle and these kernels produce identical keys and encryptions from a seed.
#pragma once
#include "modarith.h"

__device__ __forceinline__ u64 sm64(u64 x) {
    u64 z = x + 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
__device__ __forceinline__ u64 draw(u64 key, u64 ctr) { return sm64(key + ctr * 0x9E3779B97F4A7C15ull); }
// from attempt t on
__device__ __forceinline__ u64 sample_uniform(const u64 key, const u64 i, const ModQ &m, u64 t = 0) {
    const u64 mask = (1ull << m.k) - 1;
    u64 x = 0;
    // acceptance is at least 1/2 per attempt; 4096 attempts cannot all fail in practice and bound the loop
    for (; t < 4096; t++) {
        x = draw(sm64(key + t), i) & mask;
        if (x < m.q) break;
    }
    return x;
}
// n of them, `step` apart: the first attempts of all are independent of each other, and for primes just below a power of two nearly
// always the only ones (one after the other behind the loop's branch, eight of them were most of an encryption's last pass)
template <int n>
__device__ __forceinline__ void sample_uniform(const u64 key, const u64 i, const u64 step, const ModQ &m, u64 (&x)[n]) {
    const u64 first = sm64(key), mask = (1ull << m.k) - 1;
#pragma unroll
    for (int k = 0; k < n; k++) x[k] = draw(first, i + step * (u64)k) & mask;
#pragma unroll
    for (int k = 0; k < n; k++)
        if (x[k] >= m.q) x[k] = sample_uniform(key, i + step * (u64)k, m, 1);
}
__device__ __forceinline__ int sample_error(const u64 key, const u64 i) {
    const u64 x = draw(key, i), M21 = (1ull << 21) - 1;
    return __popcll(x & M21) - __popcll((x >> 21) & M21);
}
