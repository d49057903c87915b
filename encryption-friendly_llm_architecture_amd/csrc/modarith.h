// Device-side modular arithmetic for RNS primes below 2^61 on gfx950.
//
// gfx950 has no 64x64->128 multiplier: every 64-bit product below is assembled by the
// compiler from 32-bit v_mad_u64_u32 / v_mul_hi_u32 pieces, so the code is written to keep
// the number of wide products per modular multiplication minimal:
//   * constant multiplicands (NTT twiddles, 1/N, P^-1, q_l^-1, basis-conversion factors) carry a
//     precomputed Shoup quotient floor(w * 2^64 / q): one high product + two low products;
//   * data x data products are kept as 128-bit values, summed lazily, and reduced once with a
//     Barrett step sized to the prime's bit length.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

typedef unsigned long long u64;
typedef unsigned int u32;

struct u128_t {
    u64 lo, hi;
};

__device__ __forceinline__ u128_t mul64wide(u64 a, u64 b) {
    u128_t r;
    r.lo = a * b;
    r.hi = __umul64hi(a, b);
    return r;
}
__device__ __forceinline__ void add128(u128_t &acc, const u128_t &x) {
    u64 lo = acc.lo + x.lo;
    acc.hi += x.hi + (lo < acc.lo ? 1ull : 0ull);
    acc.lo = lo;
}

// Per-prime constants, passed to kernels by value or read from a small device table.
struct ModQ {
    u64 q;     // the prime
    u64 mu;    // floor(2^(2k) / q), k = bit length of q
    u32 k;     // bit length of q (q < 2^k, k <= 61)
    u32 mdot;  // floor(2^(k+31) / q) (dot_reduce_lazy)
    u64 mu3;   // floor(2^(k+63) / q) for k <= 60, else 0 (barrett_tight)
};

// x * w mod q for a constant w with ws = floor(w * 2^64 / q); result in [0, 2q).
__device__ __forceinline__ u64 mul_shoup_lazy(u64 x, u64 w, u64 ws, u64 q) {
    return x * w - __umul64hi(x, ws) * q;
}
__device__ __forceinline__ u64 mul_shoup(u64 x, u64 w, u64 ws, u64 q) {
    u64 r = mul_shoup_lazy(x, w, ws, q);
    return r >= q ? r - q : r;
}

// u + x * w - hi' * q with the quotient estimate hi' taken from three of the four 32-bit partial products of x * ws:
// hi' = xh wh + (xh wl >> 32) + (xl wh >> 32) is at most 2 below floor(x ws / 2^64), so that x * w - hi' * q lies in [0, 4q)
// instead of [0, 2q) for any 64-bit x.  One multiply-add and the carry chain of the exact high product are saved.
// x * w - hi' * q = x * w + hi' * (2^64 - q) mod 2^64 as 32-bit multiply-adds: the two low products accumulate on u (a carry
// out of bit 64 is dropped, as it should be), the four cross products, of which only the low word counts, in a register pair of their
// own.  That pair and the high word are hidden from the compiler, which otherwise makes low products and additions of the
// cross terms or takes some products twice: 31 vector instructions for an inverse butterfly where this is 17.
__device__ __forceinline__ u64 add_mul_shoup_lazy4(u64 u, u64 x, u64 w, u64 ws, u64 q) {
    const u32 xl = (u32)x, xh = (u32)(x >> 32), sl = (u32)ws, sh = (u32)(ws >> 32);
    const u64 hi = ((u64)xh * sh + __umulhi(xh, sl)) + __umulhi(xl, sh);
    const u64 nq = 0 - q;
    const u32 hl = (u32)hi, hh = (u32)(hi >> 32), wl = (u32)w, wh = (u32)(w >> 32), nl = (u32)nq, nh = (u32)(nq >> 32);
    const u64 t = (u64)hl * nl + ((u64)xl * wl + u);
    u64 cross = (u64)xl * wh + (u64)xh * wl + (u64)hl * nh + (u64)hh * nl;
    asm("" : "+v"(cross));
    u32 top = (u32)(t >> 32) + (u32)cross;
    asm("" : "+v"(top));
    return ((u64)top << 32) | (u32)t;
}
__device__ __forceinline__ u64 mul_shoup_lazy4(u64 x, u64 w, u64 ws, u64 q) { return add_mul_shoup_lazy4(0, x, w, ws, q); }
// v + e * (2^64 - q) for a quotient e of 32 bits
__device__ __forceinline__ u64 sub_multiple(u64 v, u32 e, u64 q) {
    const u64 nq = 0 - q, t = (u64)e * (u32)nq + v;
    u32 top = (u32)(t >> 32) + e * (u32)(nq >> 32);
    asm("" : "+v"(top));
    return ((u64)top << 32) | (u32)t;
}
// ---- primes just below 2^60: q = 2^60 - delta, delta < 2^27 ------------------------------------------------------------------
// What lies above bit 60 of a value counts delta times, so no quotient is estimated.  A constant w is kept with v = 2^32 w mod q, both cut at
// bit 29 (near60_cut in context.hip, Near60::cut), and y w for a 64-bit y is yl w + yh v: four multiply-adds into accumulators s0 and s1 of weights 1 and 2^29.
// 2^29 s1 is 2^29 times its low word plus 2^61 = 2 delta times its high word, two multiply-adds more; y is never cut into pieces.
#define NEAR60_DELTA (1ull << 27)
__host__ __device__ __forceinline__ bool near_2_60(const u64 q) { return q < (1ull << 60) && (1ull << 60) - q < NEAR60_DELTA; }
// u + y w, the product below 6.9q for y < 15.1q (5.8q for y < 8.1q): s0 < 2^29 (2^32 + yh), 2^29 sl < 2^61, 2 delta sh < 2^28 (2^31 + yh / 2)
__device__ __forceinline__ u64 near60_add_mul(const u64 u, const u64 y, const u64 w, const u64 v, const u32 two_delta, const u32 two_29) {
    const u32 yl = (u32)y, yh = (u32)(y >> 32);
    const u64 s1 = (u64)yh * (u32)(v >> 32) + (u64)yl * (u32)(w >> 32);
    u64 s0 = (u64)yl * (u32)w + u;
    s0 += (u64)yh * (u32)v;
    s0 += (u64)(u32)s1 * two_29;
    return s0 + (u64)(u32)(s1 >> 32) * two_delta;
}
// any v to below q + 2^32: the four bits above 2^60 are taken off and count delta each
__device__ __forceinline__ u64 near60_fold(const u64 v, const u32 delta) {
    const u32 h = (u32)(v >> 32);
    return (((u64)(h & 0x0fffffffu) << 32) | (u32)v) + (u64)(h >> 28) * delta;
}
struct Cut {   // a constant and 2^32 times it, cut
    u64 w, v;
};
// v < 32q (q < 2^59) to [0, q)
__device__ __forceinline__ u64 reduce_below_32q(u64 v, const u64 q) {
#pragma unroll
    for (int m = 16; m >= 1; m >>= 1)
        if (v >= (u64)m * q) v -= (u64)m * q;
    return v;
}
// Barrett reduction of a 128-bit value T to [0, q): T < 6 * 2^(2k) for primes below 2^60, T < 4 * 2^(2k) for those of 61 bits, where
// T / 2^(k-1) fills 64 bits.
__device__ __forceinline__ u64 barrett128(u128_t t, const ModQ &m) {
    const u32 k = m.k;
    u64 t1 = (t.hi << (65 - k)) | (t.lo >> (k - 1));
    u128_t p = mul64wide(t1, m.mu);
    u64 qhat = (p.hi << (63 - k)) | (p.lo >> (k + 1));
    u64 r = t.lo - qhat * m.q;
    const u64 q = m.q;
    if (r >= 4 * q) r -= 4 * q;
    if (r >= 2 * q) r -= 2 * q;
    if (r >= q) r -= q;
    return r;
}
// Barrett reduction of T < 3 * 2^(2k) to [0, q) for primes below 2^60 (m.mu3 != 0) with a constant of 64 bits:
// qhat = floor(floor(T / 2^(k-2)) * mu3 / 2^65) misses floor(T / q) by less than
// T / 2^(2k+3) + 2^(k-2) / q + 1 < 3/8 + 1/2 + 1, i.e. by at most 1: only the high half of one product and a single
// correction, against a full product and three corrections in barrett128.
__device__ __forceinline__ u64 barrett_tight(u128_t t, const ModQ &m) {
    const u32 k = m.k;
    const u64 t1 = (t.hi << (66 - k)) | (t.lo >> (k - 2));
    const u64 qhat = __umul64hi(t1, m.mu3) >> 1;
    const u64 r = t.lo - qhat * m.q;
    return r >= m.q ? r - m.q : r;
}
// any T: a sum of as many products of residues as 128 bits hold.  Multiples of 2^(k+1) q are taken off first, in front of the reduction and not
// in the loop that sums the products: there it costs every kernel registers, whatever number of digits it is run for.
__device__ __forceinline__ u128_t cut_sum(u128_t t, const ModQ &m) {   // to below 2 * 2^(2k)
    const u64 hi = m.q >> (63 - m.k), lo = m.q << (m.k + 1);
    while (t.hi > hi || (t.hi == hi && t.lo >= lo)) {
        t.hi -= hi + (t.lo < lo ? 1 : 0);
        t.lo -= lo;
    }
    return t;
}
// T < 3 * 2^(2k)
__device__ __forceinline__ u64 barrett3(u128_t t, const ModQ &m) {
    return m.mu3 != 0 ? barrett_tight(t, m) : barrett128(t, m);
}
__device__ __forceinline__ u64 mulmod(u64 a, u64 b, const ModQ &m) {
    return barrett3(mul64wide(a, b), m);
}
// reduce an arbitrary 64-bit value
__device__ __forceinline__ u64 reduce64(u64 a, const ModQ &m) {
    u128_t t;
    t.lo = a;
    t.hi = 0;
    return barrett128(t, m);
}
// Lazy dot product sum_i v_i * h_i of up to 8 residues v_i < 2^60 with constants h_i < 2^60 (a target residue of a fast basis
// conversion).  With v = v0 + 2^30 v1 and g = 2^30 h mod q kept beside h, the term is v0 h + v1 g: products of 30-bit
// pieces of v with 30-bit pieces of h and g, four multiply-adds into two 64-bit accumulators of weights 1 and 2^30 that 16
// products below 2^60 cannot overflow -- no carries, and a sum 34 bits longer than q instead of 64 to reduce.
struct Pieces {
    u32 lo, hi;
};
__device__ __forceinline__ Pieces pieces(const u64 v) { return Pieces{(u32)v & 0x3fffffffu, (u32)(v >> 30)}; }
struct DotCst {
    u32 h0, h1, g0, g1;
};
__device__ __forceinline__ DotCst dot_cst(const u64 h, const u64 g) {
    return DotCst{(u32)h & 0x3fffffffu, (u32)(h >> 30), (u32)g & 0x3fffffffu, (u32)(g >> 30)};
}
struct Dot2 {
    u64 s0, s1;
};
__device__ __forceinline__ void dot_clear(Dot2 &d) { d.s0 = d.s1 = 0; }
__device__ __forceinline__ void dot_add(Dot2 &d, const u64 v, const DotCst &c) {
    const u32 v0 = (u32)v & 0x3fffffffu, v1 = (u32)(v >> 30);
    d.s0 += (u64)v0 * c.h0;
    d.s0 += (u64)v1 * c.g0;
    d.s1 += (u64)v0 * c.h1;
    d.s1 += (u64)v1 * c.g1;
}
// the same of a residue that is kept in pieces
__device__ __forceinline__ void dot_add(Dot2 &d, const Pieces v, const DotCst &c) {
    d.s0 += (u64)v.lo * c.h0;
    d.s0 += (u64)v.hi * c.g0;
    d.s1 += (u64)v.lo * c.h1;
    d.s1 += (u64)v.hi * c.g1;
}
// the sum as a 128-bit value, below 2^(k + 34) for constants below 2^k
__device__ __forceinline__ u128_t dot_value(const Dot2 &d) {
    u128_t t;
    t.lo = d.s0 + (d.s1 << 30);
    t.hi = (d.s1 >> 34) + (t.lo < d.s0 ? 1ull : 0ull);
    return t;
}
// ... reduced to [0, q): k >= 32 (primes of 2^31 and more), so it lies below 6 * 2^(2k)
__device__ __forceinline__ u64 dot_reduce(const Dot2 &d, const ModQ &m) { return barrett3(dot_value(d), m); }
// ... to [0, 13q), for butterflies that take values below 16q (q < 2^60).  The sum is below 16 * 2^30 q, so that t = sum / 2^(k+2)
// fits 32 bits and t * (2^(k+31) / q) / 2^29 misses the quotient by less than 2^(k+2) / q for the cut of the sum, t / 2^29 for the
// cut of the constant and 1: 4 + 8 + 1 for q near 2^k, 8 + 4 + 1 for q near 2^(k-1).
__device__ __forceinline__ u64 dot_reduce_lazy(const Dot2 &d, const ModQ &m) {
    const u32 t = (u32)((d.s1 + (d.s0 >> 30)) >> (m.k - 28));
    const u64 qhat = ((u64)t * m.mdot) >> 29, nq = 0 - m.q;
    const u32 hl = (u32)qhat, hh = (u32)(qhat >> 32), nl = (u32)nq, nh = (u32)(nq >> 32);
    const u64 r = (u64)hl * nl + (d.s0 + (d.s1 << 30));
    return r + ((u64)(hl * nh + hh * nl) << 32);
}
__device__ __forceinline__ u64 addmod(u64 a, u64 b, u64 q) {
    u64 s = a + b;
    return s >= q ? s - q : s;
}
__device__ __forceinline__ u64 submod(u64 a, u64 b, u64 q) { return a >= b ? a - b : a + q - b; }

// ---- the same reductions for a modulus that is uniform over the wavefront (the prime of a workgroup's limb) ----------
// A 64-bit subtraction is a borrow chain of two instructions with a wait state between them on gfx950, an addition is one
// instruction: a value is reduced by ADDING 2^64 - m, kept in scalar registers where the compiler cannot see through it
// and turn the sum back into a subtraction, and selecting.  Same values as the forms above.
__device__ __forceinline__ u64 neg_uniform(u64 m) {
    u64 n = 0 - m;
    asm("" : "+s"(n));
    return n;
}
// u >= m ? u - m : u
__device__ __forceinline__ u64 cond_sub_u(u64 u, const u64 m) {
    u64 t = u + neg_uniform(m);
    asm("" : "+v"(t));
    return u >= m ? t : u;
}
__device__ __forceinline__ u64 mul_shoup_lazy_u(u64 x, u64 w, u64 ws, u64 q) {
    return x * w + __umul64hi(x, ws) * neg_uniform(q);
}
__device__ __forceinline__ u64 mul_shoup_u(u64 x, u64 w, u64 ws, u64 q) {
    return cond_sub_u(mul_shoup_lazy_u(x, w, ws, q), q);
}
__device__ __forceinline__ u64 barrett128_u(u128_t t, const ModQ &m) {
    const u32 k = m.k;
    const u64 t1 = (t.hi << (65 - k)) | (t.lo >> (k - 1));
    const u128_t p = mul64wide(t1, m.mu);
    const u64 qhat = (p.hi << (63 - k)) | (p.lo >> (k + 1));
    const u64 q = m.q;
    const u64 r = t.lo + qhat * neg_uniform(q);
    return cond_sub_u(cond_sub_u(cond_sub_u(r, 4 * q), 2 * q), q);
}
__device__ __forceinline__ u64 barrett_tight_u(u128_t t, const ModQ &m) {
    const u32 k = m.k;
    const u64 t1 = (t.hi << (66 - k)) | (t.lo >> (k - 2));
    const u64 qhat = __umul64hi(t1, m.mu3) >> 1;
    return cond_sub_u(t.lo + qhat * neg_uniform(m.q), m.q);
}
__device__ __forceinline__ u64 barrett3_u(u128_t t, const ModQ &m) {
    return m.mu3 != 0 ? barrett_tight_u(t, m) : barrett128_u(t, m);
}
__device__ __forceinline__ u64 mulmod_u(u64 a, u64 b, const ModQ &m) { return barrett3_u(mul64wide(a, b), m); }
__device__ __forceinline__ u64 addmod_u(u64 a, u64 b, u64 q) { return cond_sub_u(a + b, q); }
__device__ __forceinline__ u64 negmod(u64 a, u64 q) { return a ? q - a : 0; }

// ---- sums of products of residues below 2^60 in pieces of 30 bits -----------------------------------------------------------
// A 128-bit product summed as such is 17 instructions (the compiler makes its two halves apart, and carries them).  Cut at bit 30
// it is four multiply-adds into accumulators of weights 1, 2^30 and 2^60 that nothing is carried out of.
struct Acc3 {
    u64 s0, s1, s2;
};
// x < 2^62, y < 2^60: the hi pieces below 2^32 and 2^30, so s1 grows by less than 5 * 2^60 and s2 by less than 2^62
__device__ __forceinline__ void acc_mul(Acc3 &a, const Pieces x, const Pieces y) {
    a.s0 += (u64)x.lo * y.lo;
    a.s1 += (u64)x.lo * y.hi;
    a.s1 += (u64)x.hi * y.lo;
    a.s2 += (u64)x.hi * y.hi;
}
// T = s0 + 2^30 s1 + 2^60 s2 < 4 * 2^(2k) modulo a prime of 32 <= k <= 60 bits, to [0, 3q).  The quotient is barrett_tight's, from the
// accumulators' own parts above 2^(k-2) (which miss the carries between them: 2 at most) instead of T's: it misses
// floor(T / q) by less than T / 2^(2k+3) + (2 + 1) 2^(k-2) / q + 1 < 1/2 + 3/2 + 1, i.e. by at most 2.
__device__ __forceinline__ u64 acc_reduce(const Acc3 &a, const ModQ &m) {
    const u32 k = m.k;
    const u64 t1 = (a.s2 << (62 - k)) + (a.s1 >> (k - 32)) + (a.s0 >> (k - 2));
    const u64 qhat = __umul64hi(t1, m.mu3) >> 1;
    return (a.s0 + (a.s1 << 30) + (a.s2 << 60)) + qhat * neg_uniform(m.q);
}

// The arithmetic of a prime just below 2^60 that is uniform over the wavefront
struct Near60 {
    u64 q;
    u32 delta, delta2, delta4, two_29;
    __device__ __forceinline__ explicit Near60(const u64 prime) : q(prime), delta(0u - (u32)prime), delta2(2 * delta), delta4(4 * delta), two_29(1u << 29) {
        asm("" : "+s"(two_29));   // multiplied by, not shifted by in three instructions
    }
    // a constant with its Shoup quotient, whose upper half is the quotient of 2^32 times the constant
    __device__ __forceinline__ Cut cut(const u64 w, const u64 ws) const {
        const u64 v = (w << 32) - (ws >> 32) * q;
        return Cut{(w >> 29 << 32) | (w & 0x1fffffffu), (v >> 29 << 32) | (v & 0x1fffffffu)};
    }
    __device__ __forceinline__ u64 fold(const u64 v) const { return near60_fold(v, delta); }
    // u + y c; the product is below 6.9q for y < 15.1q, 4.9q for y < 2q
    __device__ __forceinline__ u64 add_mul(const u64 u, const u64 y, const Cut c) const { return near60_add_mul(u, y, c.w, c.v, delta2, two_29); }
    // s0 + 2^30 s1 for any two sums, below 7.1q
    __device__ __forceinline__ u64 reduce(const u64 s0, const u64 s1) const {
        return fold(s0) + (u64)(u32)s1 * (2 * two_29) + (u64)(u32)(s1 >> 32) * delta4;
    }
    // s0 + 2^30 s1 + 2^60 s2 for s0 < 2^62, s1 < 14 * 2^60, s2 < 2^63 (three products of values below 2q): 2^60 counts delta, 2^92 2^30 times
    // 4 delta.  Below 10.4q, 8.4q for three products of canonical values: multiply-adds alone where a Barrett step (acc_reduce) is 22 instructions.
    __device__ __forceinline__ u64 reduce(const Acc3 &a) const {
        const u64 s1 = a.s1 + (u64)(u32)(a.s2 >> 32) * delta4;
        u64 s0 = a.s0 + (u64)(u32)a.s2 * delta;
        s0 += (u64)(u32)s1 * (2 * two_29);
        return s0 + (u64)(u32)(s1 >> 32) * delta4;
    }
    // v < 2q to [0, q)
    __device__ __forceinline__ u64 canonical(const u64 v) const { return cond_sub_u(v, q); }
};
