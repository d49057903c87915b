// Device-side pieces shared by the transform kernels: butterflies, the two arithmetic back ends, register blocks of up
// to four stages, and the row pass.
#pragma once
#include "hemm_internal.hpp"
#include "sampling.h"

// a twiddle and its Shoup quotient; of primes just below 2^60 the twiddle and 2^32 times it, both cut (modarith.h, near60_add_mul)
struct __align__(16) Tw {
    u64 w, ws;
};
// what a pass does at its far end (see TAIL_*, LOAD_* below)
struct NttEpilogue {
    const u64 *minuend;
    u64 *out;
    const Tw *cst;  // per limb: constant and Shoup quotient
    size_t minuend_stride, out_stride;
    u32 galois;
    const u64 *second_in;   // strides as minuend / out
    u64 *second_out;
    const u64 *sk;          // [prime][N]
    u64 a_base;             // the stream of prime i has key sm64(sm64(a_base + i))
    __device__ __forceinline__ u64 *result(const int poly) const { return out + (size_t)poly * out_stride; }
};
// the same with the results where a list says, the launch's first polynomial being number `first` of it: a type of its own, since
// the list in the arguments of every launch made single key switches 0.4 % slower
struct NttEpilogueList : NttEpilogue {
    u32 first;
    ResultList list;
    __device__ __forceinline__ u64 *result(const int poly) const {
        const u32 p = first + (u32)poly;
        return list.at[p >> 1] + (p & 1 ? out_stride : 0);
    }
};

namespace {
typedef u32 u32x2 __attribute__((ext_vector_type(2)));
// Column passes address a limb through a buffer resource: the limb's base sits in scalar registers, the slab row
// (a step of 2 KiB or 32 KiB) goes into the scalar offset of each access and a thread supplies one 32-bit byte offset
// for all of its 16 accesses -- with 64-bit addresses in vector registers every access costs an add with carry.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t limb_rsrc(const void *p) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)p, 0, -1, 0x00020000);   // raw, no range limit, 32-bit format
}
template <class E>
__device__ __forceinline__ E buf_load(const __amdgpu_buffer_rsrc_t r, const u32 voff, const u32 soff) {
    const u32x2 w = __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0);
    const u64 u = ((u64)w.y << 32) | w.x;
    E v;
    __builtin_memcpy(&v, &u, 8);
    return v;
}
template <class E>
__device__ __forceinline__ void buf_store(const __amdgpu_buffer_rsrc_t r, const u32 voff, const u32 soff, const E v) {
    u64 u;
    __builtin_memcpy(&u, &v, 8);
    u32x2 w;
    w.x = (u32)u;
    w.y = (u32)(u >> 32);
    __builtin_amdgcn_raw_buffer_store_b64(w, r, voff, soff, 0);
}


// Lazy butterflies (q < 2^61, so 8q < 2^64): forward values stay in [0, 8q), inverse values in [0, 4q); q4 = 4q.
// u -= 4q when u >= 4q, written as an addition of -4q and a select: no borrow chain
__device__ __forceinline__ u64 csub(u64 u, const u64 m, const u64 neg_m) {
    u64 t = u + neg_m;
    asm("" : "+v"(t));          // keeps the compiler from turning this back into a subtraction of a selected 0 / m
    return u >= m ? t : u;
}
// 2^64 - m as a value the compiler cannot see through (it would turn x + (2^64 - m) back into a subtraction)
__device__ __forceinline__ u64 opaque_neg(u64 m) {
    u64 n = 0 - m;
    asm("" : "+s"(n));
    return n;
}
__device__ __forceinline__ void ct_bfly(u64 &x, u64 &y, const Tw tw, const u64 q, const u64 q4, const u64 nq4) {
    const u64 u = csub(x, q4, nq4);                        // < 4q
    x = add_mul_shoup_lazy4(u, y, tw.w, tw.ws, q);         // u + v, v < 4q
    y = (2 * u + q4) - x;                                  // u - v + 4q
}
__device__ __forceinline__ void gs_bfly(u64 &x, u64 &y, const Tw tw, const u64 q, const u64 q4, const u64 nq4) {
    const u64 u = x, v = y;                                // < 4q each
    x = csub(u + v, q4, nq4);
    y = mul_shoup_lazy4(u - v + q4, tw.w, tw.ws, q);
}

// Three arithmetic back ends share the kernels below.
//
// IntField: 64-bit Shoup butterflies with values kept in [0, 4q) (Harvey), for primes up to 2^61.
//
// Near60Field: primes just below 2^60, whose products need no quotient (beside it below).  A kernel that holds all three is larger: with 50-bit primes, rotation
// at level 9 of 12 + 4 primes 80.5 -> 81.5 us, its conversion pass of 512 workgroups 13.8 -> 14.3, a tensor product of ten limbs 7.1 -> 7.5.
//
// FpField: primes below 2^44 in double precision.  gfx950 issues one FP64 FMA per lane per clock but
// has to assemble every 64-bit integer product from 32-bit pieces, so for residues that fit a double
// exactly the floating-point butterfly is about a third of the instructions.  A product y*w mod q is
//     h = fl(y*w);  l = fma(y, w, -h)  [exact low part];  c = rint(h * (1/q));  r = fma(-c, q, h) + l
// Both h - c*q and the final sum are integers far below 2^53, so r is an exact residue of y*w, whatever c is.  The
// quotient comes from the rounded product, h * fl(1/q), which is off by at most |y| * 1.5 * 2^-52, so
// |r| <= (0.5 + |y| * 1.5 * 2^-52) q -- 0.57 q for |y| < 2^47.5, 0.8 q for |y| < 2^49.7.  Values stay signed and
// unreduced through the forward stages (growth 0.57 q per stage: below 11 q < 2^48 after all 16); the inverse
// stages double the sums, so a radix-16 block first reduces its inputs.
// The last pass maps to [0, q), which makes the stored result identical to the integer path's.
// Between the two launches of one transform the buffer holds the raw doubles.
#pragma clang fp contract(off)

// LAZY16 (primes below 2^60, so 16q < 2^64): forward values stay in [0, 16q) and only every other stage corrects its first
// operand -- by 8q, which takes values below 16q to below 8q; the stage after it adds up to 4q twice without a correction.
// Inverse values lie below 4q in front of a stage of even number in its block, whose sums are left below 8q; the stage after it reduces
// its sums, below 16q, by a quotient from their high word to below 3q.  One correction per two butterflies instead of one per butterfly.
// 32 x 24 limbs of 60 bits, forward 343 -> 329 us (with the sum u + v on the product's accumulator), inverse 395 -> 382; rotation on 2^13
// points 35.3 -> 34.1, product at level 9 111.9 -> 109.6, projection of a 768-wide layer 10157 -> 10015.
template <bool LAZY16>
struct IntFieldT {
    typedef u64 E;
    typedef Tw W;
    u64 q, q2, q4, nq8, nq4, nq2, nq1, ni, nis;
    u32 k, mdot;   // LAZY16: bit length of q, floor(2^(k+31) / q)
    __device__ __forceinline__ IntFieldT(const ModQ *modq, const u64 *ninv, const u64 *ninv_s, const double *, int prime) {
        q = modq[prime].q;
        k = modq[prime].k;
        mdot = modq[prime].mdot;
        q2 = 2 * q;
        q4 = 4 * q;
        nq8 = opaque_neg(2 * q4);
        nq4 = opaque_neg(q4);
        nq2 = opaque_neg(q2);
        nq1 = opaque_neg(q);
        // a pass that does not end an inverse transform has no use for them and brings no table
        ni = ninv != nullptr ? ninv[prime] : 0;
        nis = ninv_s != nullptr ? ninv_s[prime] : 0;
    }
    __device__ __forceinline__ void set_scale(const Tw c) {
        ni = c.w;
        nis = c.ws;
    }
    // v < 16q, 2^44 < q < 2^60, to below 3q: v / q exceeds (v >> 32) floor(2^64 / q) / 2^32 by less than v / 2^64 + 2^32 / q < 1 + 2^-12, and
    // the product's high word by less than 1 more
    __device__ __forceinline__ u64 reduce_3q(u64 v) const { return sub_multiple(v, __umulhi((u32)(v >> 32), mdot >> (k - 33)), q); }
    // ... to below 1.001 q: with floor(2^(k+31) / q) the first of the two errors is below 2^-27
    __device__ __forceinline__ u64 reduce_q(u64 v) const { return sub_multiple(v, __umulhi((u32)(v >> 32), mdot) >> (k - 33), q); }
    __device__ __forceinline__ E from_canonical(u64 v) const { return v; }
    // < 13q: primes below 2^60 only, whose butterflies take inputs below 16q
    __device__ __forceinline__ E from_dot(const Dot2 &d, const ModQ &m) const { return dot_reduce_lazy(d, m); }
    // odd: the stage's index within its radix-16 block is odd
    __device__ __forceinline__ void ct(E &x, E &y, const W tw, const bool odd) const {
        if (!LAZY16) {
            ct_bfly(x, y, tw, q, q4, nq4);
            return;
        }
        const u64 u = odd ? x : csub(x, 2 * q4, nq8);   // < 12q on odd stages, < 8q on even ones
        x = add_mul_shoup_lazy4(u, y, tw.w, tw.ws, q);  // u + v, v < 4q
        y = (2 * u + q4) - x;                           // u - v + 4q
    }
    // odd: as above; last: the stage is the last of its block
    __device__ __forceinline__ void gs(E &x, E &y, const W tw, const bool odd, const bool last) const {
        if (!LAZY16) {
            gs_bfly(x, y, tw, q, q4, nq4);
            return;
        }
        const u64 u = x, v = y;   // < 8q on odd stages, < 4q on even ones
        x = odd || last ? reduce_3q(u + v) : u + v;
        y = mul_shoup_lazy4((u + (odd ? 2 * q4 : q4)) - v, tw.w, tw.ws, q);
    }
    template <int T, int P>
    __device__ __forceinline__ void after_inverse_block(E (&)[P]) const {}
    __device__ __forceinline__ u64 to_canonical(E v) const {   // v < 8q (16q with LAZY16)
        if (LAZY16) return csub(reduce_q(v), q, nq1);
        return csub(csub(csub(v, q4, nq4), q2, nq2), q, nq1);
    }
    __device__ __forceinline__ u64 scale_to_canonical(E v) const {
        return csub(mul_shoup_lazy(v, ni, nis, q), q, nq1);
    }
    // a signed integer as an input of a forward transform, where it is as small as from_signed takes it: below 2q
    __device__ __forceinline__ bool takes_signed(long long v) const { return (u64)v + q < q2; }
    __device__ __forceinline__ E from_signed(long long v) const { return (u64)v + q; }
    // v - a s, canonical, for canonical a and s
    __device__ __forceinline__ u64 minus_product(E v, u64 a, u64 s, const ModQ &m) const { return submod(to_canonical(v), mulmod(a, s, m), q); }
    // (y - v) * cst mod q for a transformed value v and a canonical minuend y
    __device__ __forceinline__ u64 sub_scale(E v, u64 y, const Tw cst) const {
        const u64 c = to_canonical(v);
        const u64 d = y >= c ? y - c : y + q - c;
        return csub(mul_shoup_lazy(d, cst.w, cst.ws, q), q, nq1);
    }
};

typedef IntFieldT<false> IntField;

// Primes just below 2^60 (near_2_60: what a chain of 60-bit primes is made of, and the special primes).  Forward values stay below 15.1q: a
// stage of even number in its block folds its first operand to q and a little, sums and differences are then below 8.1q, and after the
// odd stage behind it below 15.1q.  Inverse values lie below 6.9q in front of every stage, whose sums are folded.  A butterfly is 10.5
// vector instructions forward and 13 inverse where LAZY16 takes 16.5 and 17 (a column pass of 16 points per thread 733 and 1140
// instructions in all, 1088 and 1501).  Such passes were bound by these instructions: 32 x 24 limbs forward 337 -> 309 us (the trips
// through memory take 303), rotation on 24 + 4 primes of 60 bits, level 20 125.8 -> 115.4, product of two encrypted 32 x 32 tiles
// 432 -> 404, projection of a 768-wide layer 9770 -> 9587.  The line: a product stays below 6.9q as long as 2^28 (2^31 + yh / 2) is
// below 0.97 * 2^60; the first 55 primes of rings of 2^16 points lie above 2^60 - 2^27, of smaller rings
// more.
struct Near60Field : Near60 {
    typedef u64 E;
    typedef Tw W;
    u64 q2, q7, nq1;
    Cut scale;   // what an inverse transform ends with
    __device__ __forceinline__ Near60Field(const ModQ *modq, const u64 *ninv, const u64 *ninv_s, const double *, int prime) : Near60(modq[prime].q) {
        q2 = 2 * q;
        q7 = 7 * q;
        asm("" : "+s"(q7));   // added, not made of q by a multiply-add
        nq1 = opaque_neg(q);
        if (ninv != nullptr) set_scale(Tw{ninv[prime], ninv_s[prime]});
    }
    // v c, canonical
    __device__ __forceinline__ u64 times(const u64 v, const Cut c) const { return csub(fold(add_mul(0, v, c)), q, nq1); }
    __device__ __forceinline__ void set_scale(const Tw c) { scale = cut(c.w, c.ws); }
    __device__ __forceinline__ E from_canonical(u64 v) const { return v; }
    // up to 8 sources: either half of the sum may fill 64 bits; below 7.1q
    __device__ __forceinline__ E from_dot(const Dot2 &d, const ModQ &) const { return reduce(d.s0, d.s1); }
    __device__ __forceinline__ void ct(E &x, E &y, const W tw, const bool odd) const {
        const u64 u = odd ? x : fold(x);
        x = add_mul(u, y, Cut{tw.w, tw.ws});
        y = (2 * u + q7) - x;
    }
    __device__ __forceinline__ void gs(E &x, E &y, const W tw, const bool, const bool) const {
        const u64 u = x, v = y;
        x = fold(u + v);
        y = add_mul(0, (u + q7) - v, Cut{tw.w, tw.ws});
    }
    template <int T, int P>
    __device__ __forceinline__ void after_inverse_block(E (&)[P]) const {}
    __device__ __forceinline__ u64 to_canonical(E v) const { return csub(fold(v), q, nq1); }
    __device__ __forceinline__ u64 scale_to_canonical(E v) const { return times(v, scale); }
    __device__ __forceinline__ bool takes_signed(long long v) const { return (u64)v + q < q2; }
    __device__ __forceinline__ E from_signed(long long v) const { return (u64)v + q; }
    __device__ __forceinline__ u64 minus_product(E v, u64 a, u64 s, const ModQ &m) const { return submod(to_canonical(v), mulmod(a, s, m), q); }
    __device__ __forceinline__ u64 sub_scale(E v, u64 y, const Tw cst) const { return times((y + q2) - fold(v), cut(cst.w, cst.ws)); }
};
// fn with the arithmetic of an integer prime below 2^60, resp. of any integer prime
template <class FN>
__device__ __forceinline__ void with_field_60(const ModQ *modq, const u64 *ninv, const u64 *ninv_s, const double *fp, const int prime, const FN fn) {
    if (near_2_60(modq[prime].q))
        fn(Near60Field(modq, ninv, ninv_s, fp, prime));
    else
        fn(IntFieldT<true>(modq, ninv, ninv_s, fp, prime));
}
template <class FN>
__device__ __forceinline__ void with_int_field(const ModQ *modq, const u64 *ninv, const u64 *ninv_s, const double *fp, const int prime, const FN fn) {
    if ((modq[prime].q >> 60) != 0)
        fn(IntField(modq, ninv, ninv_s, fp, prime));
    else
        with_field_60(modq, ninv, ninv_s, fp, prime, fn);
}

struct FpField {
    typedef double E;
    // (The quotient as y * (w * (1/q)) is as exact and takes an instruction more per twiddle: encoding 35.6 -> 34.6 us, inverse transform of
    // 5 x 7 limbs of 2^14 points 12.05 -> 11.9, product at level 9 96.6 -> 95.8, projection of a 768-wide layer 9280 -> 9200.)
    typedef double W;   // the twiddle as a double
    double q, qinv, ni;
    __device__ __forceinline__ FpField(const ModQ *, const u64 *, const u64 *, const double *fp, int prime) {
        q = fp[4 * prime];
        qinv = fp[4 * prime + 1];
        ni = fp[4 * prime + 2];
    }
    __device__ __forceinline__ void set_scale(const Tw c) { ni = (double)c.w; }
    __device__ __forceinline__ E mul(E y, E w) const {
        const double h = y * w;
        const double l = __builtin_fma(y, w, -h);
        const double c = __builtin_rint(h * qinv);
        return __builtin_fma(-c, q, h) + l;
    }
    __device__ __forceinline__ E reduce(E x) const { return __builtin_fma(-__builtin_rint(x * qinv), q, x); }
    __device__ __forceinline__ E from_canonical(u64 v) const {
        return __longlong_as_double((long long)(v | 0x4330000000000000ull)) - 4503599627370496.0;
    }
    // A lazy dot product as a residue of magnitude below 1.3 q: regrouped into pieces of weights 1 and 2^30, below 2^30 and 2^49
    // (constants below 2^44), both exact in a double; the upper one is multiplied by 2^30 (below q, as every prime is).  No
    // integer reduction and no conversion from canonical form; a forward transform then ends below 11 q as from canonical residues.
    __device__ __forceinline__ E from_dot(const Dot2 &d, const ModQ &) const {
        const u64 p1 = (d.s0 >> 30) + d.s1;
        return (double)((u32)d.s0 & 0x3fffffffu) + mul(from_canonical(p1), 1073741824.0);
    }
    __device__ __forceinline__ void ct(E &x, E &y, const W tw, const bool) const {
        const double v = mul(y, tw);
        const double u = x;
        x = u + v;
        y = u - v;
    }
    __device__ __forceinline__ void gs(E &x, E &y, const W tw, const bool, const bool) const {
        const double u = x, v = y;
        x = u + v;
        y = mul(u - v, tw);
    }
    // A Gentleman-Sande block of T stages doubles the sums: from inputs bounded by B, element 0 of a sub-block of 2^T is
    // bounded by 2^T B, element 1 by 2^(T-1) r, elements 2 and 3 by 2^(T-2) r, ... with r the bound of a product, and the
    // largest value it multiplies is 2^T B.  With element 0 of every sub-block (and element 1 where T = 4) reduced after
    // each block every block starts from B <= 4 r: r <= 0.8 q gives B <= 3.2 q and 16 B <= 51 q < 2^49.7 (q < 2^44), for
    // which r <= 0.8 q holds again; products of values below 2^50 are still exact.
    // (Eight registers per thread: the upper half of a block of four stages has its elements 4 and 5 reduced as well.  Four: register 0
    // of a block of four stages holds its elements 0 .. 3, registers 0 and 2 of two sub-blocks of three theirs.)
    template <int T, int P>
    __device__ __forceinline__ void after_inverse_block(E (&x)[P]) const {
        constexpr int step = P == 4 ? (T == 4 || T == 2 ? 4 : 2) : 1 << T;
#pragma unroll
        for (int k = 0; k < P; k += step) x[k] = reduce(x[k]);
        if (T == 4 && P > 4) x[1] = reduce(x[1]);
    }
    __device__ __forceinline__ u64 centred_to_canonical(E r) const {
        r += r < 0.0 ? q : 0.0;
        return (u64)__double_as_longlong(r + 4503599627370496.0) & 0x000fffffffffffffull;
    }
    __device__ __forceinline__ u64 to_canonical(E v) const { return centred_to_canonical(reduce(v)); }
    __device__ __forceinline__ u64 scale_to_canonical(E v) const { return centred_to_canonical(mul(v, ni)); }
    // integers of magnitude below 2^51 are exact, and so is what is left of them below q / 2
    __device__ __forceinline__ bool takes_signed(long long v) const { return (u64)v + (1ull << 51) < 1ull << 52; }
    __device__ __forceinline__ E from_signed(long long v) const {
        return reduce(__longlong_as_double(v + 0x4338000000000000ll) - 6755399441055744.0);
    }
    __device__ __forceinline__ u64 minus_product(E v, u64 a, u64 s, const ModQ &) const {
        return to_canonical(v - mul(from_canonical(a), from_canonical(s)));
    }
    __device__ __forceinline__ u64 sub_scale(E v, u64 y, const Tw cst) const {
        return centred_to_canonical(mul(from_canonical(y) - v, (double)cst.w));
    }
};

// How a block of up to four stages on 16 points lies in registers.  P = 16: one thread holds the block.  P = 8: two lanes of a
// wavefront 32 apart hold eight points each, h = 0 and 1; P = 4: four lanes 16 apart hold four each, h = 0 .. 3; the threads that
// share a block are otherwise numbered as with P = 16 (t).  Two layouts: `whole`, lane h holds points P h .. P h + P - 1, in which every
// stage of a distance below P is local, and `split`, in which the wider ones are: with P = 8 lane h holds points 4h .. 4h + 3 and
// 8 + 4h .. 8 + 4h + 3, with P = 4 points h, h + 4, h + 8 and h + 12.  v_permlane32_swap_b32 and, P = 4, v_permlane16_swap_b32 between
// registers turn one into the other.  Blocks without a wide stage only ever use `whole`.
// A thread of 16 points is one wavefront per SIMD in a launch of up to 256 workgroups, and then its load latencies and the
// dependences of 64-bit products are what the launch takes; eight and four points per thread put two and four wavefronts there with a half
// and a quarter of the instructions each.  The arithmetic of every point, and with it the residues, is the same.
template <int P>
struct Lanes {
    static constexpr int SHARE = 64 * P / 16;   // lanes of a wavefront with blocks of their own
    static __device__ __forceinline__ u32 t() { return P == 16 ? threadIdx.x : (threadIdx.x & (SHARE - 1u)) | ((threadIdx.x >> 6) * SHARE); }
    static __device__ __forceinline__ u32 h() { return P == 16 ? 0u : (threadIdx.x & 63u) / SHARE; }
    template <int T>
    static __device__ __forceinline__ constexpr bool wide() { return (1 << T) > P; }   // whether T stages begin in `split`
    // point of register k: a constant and the lane's part
    template <int T>
    static __device__ __forceinline__ constexpr int split(const int k) { return !wide<T>() ? k : P == 4 ? 4 * k : (k & 3) + 8 * (k >> 2); }
    template <int T>
    static __device__ __forceinline__ u32 h_split() { return !wide<T>() ? P * h() : P == 4 ? h() : 4u * h(); }
    static __device__ __forceinline__ u32 h_whole() { return P * h(); }
};
// split <-> whole: register k and lane h change places
template <int DISTANCE>
__device__ __forceinline__ void swap_lanes(u64 &a, u64 &b) {
    const u32x2 lo = DISTANCE == 32 ? __builtin_amdgcn_permlane32_swap((u32)a, (u32)b, false, false)
                                    : __builtin_amdgcn_permlane16_swap((u32)a, (u32)b, false, false);
    const u32x2 hi = DISTANCE == 32 ? __builtin_amdgcn_permlane32_swap((u32)(a >> 32), (u32)(b >> 32), false, false)
                                    : __builtin_amdgcn_permlane16_swap((u32)(a >> 32), (u32)(b >> 32), false, false);
    a = ((u64)hi.x << 32) | lo.x;
    b = ((u64)hi.y << 32) | lo.y;
}
template <int DISTANCE, class E>
__device__ __forceinline__ void swap_values(E &x, E &y) {
    u64 a, b;
    __builtin_memcpy(&a, &x, 8);
    __builtin_memcpy(&b, &y, 8);
    swap_lanes<DISTANCE>(a, b);
    __builtin_memcpy(&x, &a, 8);
    __builtin_memcpy(&y, &b, 8);
}
template <class E>
__device__ __forceinline__ void swap_layout(E (&x)[4]) {
    swap_values<32>(x[0], x[2]);
    swap_values<32>(x[1], x[3]);
    swap_values<16>(x[0], x[1]);
    swap_values<16>(x[2], x[3]);
}
template <class E>
__device__ __forceinline__ void swap_layout(E (&x)[8]) {
#pragma unroll
    for (int k = 0; k < 4; k++) swap_values<32>(x[k], x[k + 4]);
}
template <class E>
__device__ __forceinline__ void swap_layout(E (&)[16]) {}

// The pairs of a stage of distance d in a lane's registers: blocks of 2 dist, one twiddle group each, the first number first_group
template <int P>
struct StagePairs {
    int dist;            // of a pair's registers
    u32 first_group;
    __device__ __forceinline__ constexpr StagePairs(const int d, const bool split, const u32 h)
        : dist(!split ? d : P == 4 ? d / 4 : 4), first_group(!split ? h * (u32)(P / 2 / d) : 0u) {}
};
// The lane of a block of stages.  KeptLane: a number that the caller has; the stages are then simplified before its bits are known.  OwnLane: made
// where the stages begin.  Inverse transforms take the second, 72 registers and 484 instructions instead of 78 and 452 in the row pass of 2^16 points
// (even) and 64 registers instead of 72 where a limb is one launch (32 x 24 limbs of 2^13 points 28.3 -> 25.3 us, of 60 bits 34.5 -> 31.5), and so do conversions, of which eight sources on
// 2^15 points spill 20 registers with the first.  The other forward transforms take the first (the same limbs 24.0 -> 23.1).
struct KeptLane {
    u32 h;
    __device__ __forceinline__ u32 operator()() const { return h; }
};
template <int P>
struct OwnLane {
    __device__ __forceinline__ u32 operator()() const { return Lanes<P>::h(); }
};
// T Cooley-Tukey stages on 16 points that are 16 >> T sub-blocks of 2^T consecutive ones; stage s, group g uses twiddle
// tw(s, g).  Points come in as `split` and leave as `whole`.
template <int T, int P, class F, class TW, class LANE = KeptLane>
__device__ __forceinline__ void stages_fwd(const F &f, typename F::E (&x)[P], const TW tw, const LANE lane = LANE{Lanes<P>::h()}) {
    const u32 h = lane();
#pragma unroll
    for (int s = 0; s < T; s++) {
        const int d = 1 << (T - 1 - s);
        const bool split = d >= P;
        const StagePairs<P> p(d, split, h);
#pragma unroll
        for (int g = 0; g < P / 2 / p.dist; g++) {
            const typename F::W w = tw(s, p.first_group + (u32)g);
#pragma unroll
            for (int j = 0; j < p.dist; j++) f.ct(x[g * 2 * p.dist + j], x[g * 2 * p.dist + j + p.dist], w, (s & 1) != 0);
        }
        if (split && d / 2 < P) swap_layout(x);
    }
}
// T Gentleman-Sande stages, the other way round: `whole` in, `split` out; stage s has distance 1 << s.
template <int T, int P, class F, class TW, class LANE = OwnLane<P>>
__device__ __forceinline__ void stages_inv(const F &f, typename F::E (&x)[P], const TW tw, const LANE lane = LANE()) {
    const u32 h = lane();
#pragma unroll
    for (int s = 0; s < T; s++) {
        const int d = 1 << s;
        const bool split = d >= P;
        if (split && d / 2 < P) swap_layout(x);
        const StagePairs<P> p(d, split, h);
#pragma unroll
        for (int g = 0; g < P / 2 / p.dist; g++) {
            const typename F::W w = tw(s, p.first_group + (u32)g);
#pragma unroll
            for (int j = 0; j < p.dist; j++) f.gs(x[g * 2 * p.dist + j], x[g * 2 * p.dist + j + p.dist], w, (s & 1) != 0, s == T - 1);
        }
    }
}
// Blocks on the stage-ordered table: forward stage s, group g: entry (X << s) + g; inverse: (X << (T - 1 - s)) + g.  SAME: the
// sub-blocks are different columns of one block and share its twiddles.
template <int T, bool SAME = false, int P, class F, class LANE = KeptLane>
__device__ __forceinline__ void radix_fwd(const F &f, typename F::E (&x)[P], const typename F::W *__restrict__ tw,
                                          const u32 X, const LANE lane = LANE{Lanes<P>::h()}) {
    stages_fwd<T>(f, x, [&](const int s, const u32 g) { return tw[(X << s) + (SAME ? g & ((1u << s) - 1u) : g)]; }, lane);
}
template <int T, bool SAME = false, int P, class F, class LANE = OwnLane<P>>
__device__ __forceinline__ void radix_inv(const F &f, typename F::E (&x)[P], const typename F::W *__restrict__ tw,
                                          const u32 X, const LANE lane = LANE()) {
    stages_inv<T>(f, x, [&](const int s, const u32 g) {
        return tw[(X << (T - 1 - s)) + (SAME ? g & ((1u << (T - 1 - s)) - 1u) : g)];
    }, lane);
}

// The inner radix-16 block of a row pass (X = 16 (R + r) + c: a different X for every thread) reads its 15 twiddles
// from a table laid out for it: entry ((r * 15 + slot) * 16 + c), slot = 2^l - 1 + g for twiddle (X << l) + g, so that
// the 16 threads of a row read 16 consecutive entries per (l, g) -- from the stage-ordered table they would read 16
// entries 2^l apart, up to 64 cache lines per load instruction of a wavefront instead of 8.
template <int P, class F>
__device__ __forceinline__ void radix16_fwd_rows(const F &f, typename F::E (&x)[P], const typename F::W *__restrict__ rt) {
    stages_fwd<4>(f, x, [&](const int s, const u32 g) { return rt[((1u << s) - 1u + g) * 16u]; });
}
template <int P, class F>
__device__ __forceinline__ void radix16_inv_rows(const F &f, typename F::E (&x)[P], const typename F::W *__restrict__ rt) {
    stages_inv<4>(f, x, [&](const int s, const u32 g) { return rt[((8u >> s) - 1u + g) * 16u]; });
}

#define ROWPAD 272  // 256 residues of a row + one pad word per 16, so a 16-lane column read
                    // (stride 17 words) hits 16 distinct bank pairs
__device__ __forceinline__ int padc(int c) { return c + (c >> 4); }

__device__ __forceinline__ int swz_row(int r) { return r ^ ((r >> 4) & 1); }

// A signed coefficient of an encoding, plus an error coefficient where one is drawn, as a residue
__device__ __forceinline__ u64 lift_residue(const long long v, const ModQ &m) {
    const u64 r = reduce64((u64)(v < 0 ? -v : v), m), n = m.q - r;
    return (v < 0) & (r != 0) ? n : r;
}
__device__ __forceinline__ u64 lifted(const LiftSource &ls, const long long *__restrict__ coef, const u32 n, const ModQ &m) {
    const u64 r = lift_residue(coef[n], m);
    if (!ls.with_error) return r;
    const int e = sample_error(ls.error_key, n);
    return addmod(r, e >= 0 ? (u64)e : m.q - (u64)(-e), m.q);
}
// The coefficients of a thread, number k of them at index(k), as inputs of a forward transform.  Nearly always they are small enough to be taken as
// they are, in two instructions for primes of 44 bits and more and five for the others; a Barrett reduction of each (and a modular
// addition of the error) is 45.
template <int P, class F, class INDEX>
__device__ __forceinline__ void lifted_inputs(const F &f, typename F::E (&x)[P], const LiftSource &ls, const long long *__restrict__ coef,
                                              const ModQ &m, const INDEX index) {
    long long v[P];
    bool small = true;
#pragma unroll
    for (int k = 0; k < P; k++) v[k] = coef[index(k)];
#pragma unroll
    for (int k = 0; k < P; k++) {
        if (ls.with_error) v[k] = (long long)((u64)v[k] + (u64)(long long)sample_error(ls.error_key, index(k)));
        small = small && f.takes_signed(v[k]);
    }
    if (small) {
#pragma unroll
        for (int k = 0; k < P; k++) x[k] = f.from_signed(v[k]);
    } else {
#pragma unroll
        for (int k = 0; k < P; k++) x[k] = f.from_canonical(lifted(ls, coef, index(k), m));
    }
}
// The P coefficients of a thread as a basis conversion computed on the fly: coefficient k is sum_i v_i * hat_i mod q over
// the n_src <= NS source limbs (pre-scaled, the same sums as the stand-alone conversion kernels), read at voff + off(k) inside a
// limb; so[i]: byte offset of source limb i.
// The loads of the next coefficients, about CONV_LOADS residues, are in flight while the present one's products are taken: one
// wait for the first of them instead of one per source limb behind a branch of its own.  More in flight cost wavefronts: ModDown
// of 64 / 16 polynomials of 7 + 4 limbs 389 / 108 us with 20 residues and six waves per SIMD, 400 / 110 with 40 and four.
#define CONV_LOADS 20
template <int N_SRC, int NS, int P, class F, class OFF>
__device__ __forceinline__ void converted_exact(const F &f, typename F::E (&x)[P], const __amdgpu_buffer_rsrc_t src, const u32 voff,
                                                const u32 (&so)[NS], const DotCst (&h)[NS], const ModQ m, const OFF off) {
    constexpr int AHEAD = CONV_LOADS / N_SRC < P ? CONV_LOADS / N_SRC : P;   // coefficients whose sources are in flight together
    u32x2 v[P][N_SRC];
    auto load = [&](const int k) {
#pragma unroll
        for (int i = 0; i < N_SRC; i++) v[k][i] = __builtin_amdgcn_raw_buffer_load_b64(src, voff, so[i] + off(k), 0);
    };
#pragma unroll
    for (int k = 0; k < AHEAD; k++) load(k);
#pragma unroll
    for (int k = 0; k < P; k++) {
        Dot2 d;
        dot_clear(d);
#pragma unroll
        for (int i = 0; i < N_SRC; i++) dot_add(d, ((u64)v[k][i].y << 32) | v[k][i].x, h[i]);
        if (k + AHEAD < P) load(k + AHEAD);
        x[k] = f.from_dot(d, m);
    }
}
template <int K, int NS, int P, class F, class OFF>
__device__ __forceinline__ void converted_inputs(const F &f, typename F::E (&x)[P], const __amdgpu_buffer_rsrc_t src,
                                                 const u32 voff, const u32 (&so)[NS], const DotCst (&h)[NS], const int n_src,
                                                 const ModQ m, const OFF off) {
    if constexpr (K > 1)
        if (n_src < K) return converted_inputs<K - 1>(f, x, src, voff, so, h, n_src, m, off);
    converted_exact<K>(f, x, src, voff, so, h, m, off);
}

// A row's 16 threads (32 with eight points each, 64 with four) sit in one wavefront, so the LDS exchanges of
// the row kernel never cross a wavefront: ordering them needs no workgroup barrier, only a fence that
// keeps the compiler from moving LDS accesses across it.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Optional tail of a forward transform (TAIL), on the values v that the last pass already holds in registers, instead of
// storing them in place:
//   TAIL_SUB_SCALE: (minuend - v) * cst[limb] to `out` -- the last step of ModDown / rescale (saves one read and one write of
//                   every limb and a launch);
//   TAIL_ENCRYPT:   v is an encoded message plus an error: a sampled from a stream of the limb's prime to `second_out`,
//                   v - a s to `out`.
// Optional origin of an inverse transform's input (LOAD): `data` itself or `minuend` (same slot numbering, own polynomial
// stride; nullptr: data), LOAD_ROTATED: `minuend` through the automorphism `galois`, LOAD_DECRYPT: minuend + second_in * s.
//   TAIL_SUB_SCALE_LIST: TAIL_SUB_SCALE with results where a list says (a kernel's choice of NttEpilogueList; not of rows_body).
enum { TAIL_NONE = 0, TAIL_SUB_SCALE = 1, TAIL_ENCRYPT = 2, TAIL_SUB_SCALE_LIST = 3 };
constexpr int tail_of(const int tail) { return tail == TAIL_SUB_SCALE_LIST ? (int)TAIL_SUB_SCALE : tail; }
template <int TAIL>
struct EpilogueOf {
    typedef NttEpilogue T;
};
template <>
struct EpilogueOf<TAIL_SUB_SCALE_LIST> {
    typedef NttEpilogueList T;
};
enum { LOAD_PLAIN = 0, LOAD_ROTATED = 1, LOAD_DECRYPT = 2 };
// what TAIL_ENCRYPT and LOAD_DECRYPT need for one row
struct RowSecond {
    const u64 *in;
    u64 *out;
    const u64 *sk;
    u64 key;
    ModQ m;
};

// forward pass 2 / inverse pass 1 work on 16 whole rows (16 x 256 contiguous residues); r: the row of 2^log_r.
// LOAD_ROTATED: ld is the base of the source limb and residue k of the input is ld[galois_index(k)] -- an aligned
// group of 16 residues stays an aligned group under the automorphism, so the loads touch the same number of lines
// IN_LDS: the row pass follows (forward) or precedes (inverse) a column pass over the same limb in the same workgroup: the
// row is taken from, resp. left in, its padded LDS row instead of memory.
template <int P, bool INV, int TAIL, int LOAD, bool IN_LDS, class F>
__device__ __forceinline__ void rows_body(u64 *__restrict__ row, const Tw *__restrict__ tw_int,
                                          const Tw *__restrict__ rtw_int, const F f, u64 *lds_raw, const int log_r, const u32 r,
                                          const u64 *__restrict__ mn, u64 *__restrict__ o, const Tw cst,
                                          const u64 *__restrict__ ld, const u32 gal, const RowSecond &sec) {
    typedef typename F::E E;
    typedef Lanes<P> L;
    const typename F::W *tw = (const typename F::W *)tw_int;
    const int c = L::t() & 15, rr = L::t() >> 4;
    const typename F::W *rt = (const typename F::W *)rtw_int + (r * 15u * 16u + (u32)c);
    E *l = (E *)lds_raw + rr * ROWPAD;
    u64 *lc = lds_raw + rr * ROWPAD;
    E *mem = (E *)row;
    // residues of a thread: c + 16 e for the points e of the outer block, 16 c + e for the inner one, and from and to
    // memory in canonical form c + 16 e with the lanes of a pair side by side (e = 2 k + h)
    const int cs = c + 16 * (int)L::template h_split<4>(), cw = c + 16 * (int)L::h_whole();
    const int is = 16 * c + (int)L::template h_split<4>(), iw = 16 * c + (int)L::h_whole();
    const int cm = c + 16 * (int)L::h();
    constexpr int step = 256 / P;
    E x[P];
    if (!INV) {
#pragma unroll
        for (int k = 0; k < P; k++) {
            const int e = cs + 16 * L::template split<4>(k);
            x[k] = IN_LDS ? l[padc(e)] : mem[e];
        }
        radix_fwd<4>(f, x, tw, (1u << log_r) + r);
        if (IN_LDS && P < 16) wave_sync();   // both lanes of a pair have read before either writes
#pragma unroll
        for (int k = 0; k < P; k++) l[padc(cw + 16 * k)] = x[k];
        wave_sync();
#pragma unroll
        for (int k = 0; k < P; k++) x[k] = l[padc(is + L::template split<4>(k))];
        // the minuend of the fused tail is fetched under the second radix-16 block instead of after it
        u64 mv[TAIL == TAIL_SUB_SCALE ? P : 1];
        if (TAIL == TAIL_SUB_SCALE) {
#pragma unroll
            for (int k = 0; k < P; k++) mv[k] = __builtin_nontemporal_load(mn + cm + step * k);
        }
        radix16_fwd_rows(f, x, rt);
        wave_sync();
#pragma unroll
        for (int k = 0; k < P; k++) l[padc(iw + k)] = x[k];
        wave_sync();
        if (TAIL == TAIL_SUB_SCALE) {
#pragma unroll
            for (int k = 0; k < P; k++) o[cm + step * k] = f.sub_scale(l[padc(cm + step * k)], mv[k], cst);
        } else if (TAIL == TAIL_ENCRYPT) {
            u64 s[P], a[P];
#pragma unroll
            for (int k = 0; k < P; k++) s[k] = sec.sk[cm + step * k];
            sample_uniform(sec.key, (u64)((r << 8) + (u32)cm), (u64)step, sec.m, a);
#pragma unroll
            for (int k = 0; k < P; k++) {
                const int e = cm + step * k;
                o[e] = f.minus_product(l[padc(e)], a[k], s[k], sec.m);
                sec.out[e] = a[k];
            }
        } else {
#pragma unroll
            for (int k = 0; k < P; k++) row[cm + step * k] = f.to_canonical(l[padc(cm + step * k)]);
        }
    } else {
        if (LOAD == LOAD_DECRYPT) {
#pragma unroll
            for (int k = 0; k < P; k++) {
                const int e = cm + step * k;
                lc[padc(e)] = addmod(ld[e], mulmod(sec.in[e], sec.sk[e], sec.m), sec.m.q);
            }
        } else if (LOAD == LOAD_ROTATED) {
#pragma unroll
            for (int k = 0; k < P; k++) lc[padc(cm + step * k)] = ld[galois_index((r << 8) + (u32)(cm + step * k), gal, 8 + log_r)];
        } else {
#pragma unroll
            for (int k = 0; k < P; k++) lc[padc(cm + step * k)] = ld[cm + step * k];
        }
        wave_sync();
#pragma unroll
        for (int k = 0; k < P; k++) x[k] = f.from_canonical(lc[padc(iw + k)]);
        radix16_inv_rows(f, x, rt);
        f.template after_inverse_block<4>(x);
        wave_sync();
#pragma unroll
        for (int k = 0; k < P; k++) l[padc(is + L::template split<4>(k))] = x[k];
        wave_sync();
#pragma unroll
        for (int k = 0; k < P; k++) x[k] = l[padc(cw + 16 * k)];
        radix_inv<4>(f, x, tw, (1u << log_r) + r);
        f.template after_inverse_block<4>(x);
        if (IN_LDS && P < 16) wave_sync();
#pragma unroll
        for (int k = 0; k < P; k++) {   // IN_LDS: the places this thread, or the other one of its pair, has just read
            const int e = cs + 16 * L::template split<4>(k);
            if (IN_LDS) l[padc(e)] = x[k];
            else mem[e] = x[k];
        }
    }
}

}  // namespace
