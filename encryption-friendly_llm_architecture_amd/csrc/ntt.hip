// Batched negacyclic NTT / INTT over RNS primes < 2^61 for gfx950.
//
// Forward: merged-twiddle Cooley-Tukey, natural order in, bit-reversed order out
//   out[k] = sum_j a[j] psi^{(2 bitrev(k)+1) j};  inverse: Gentleman-Sande with the 1/N factor.
// Twiddle table per prime: tw[i] = (psi^bitrev(i), floor(that * 2^64 / q)) as one 16-byte entry.
//
// Rings of 2^13 points and more take two launches over the R x 256 view  index = r * 256 + c, R = N / 256 (a limb of 2^16
// points, 512 KiB, does not fit a CU's LDS, and a smaller one spread over R / 16 workgroups keeps more CUs busy):
//   forward pass 1: stages 0 .. log2 R - 1  act down columns  (butterfly distance >= 256)
//   forward pass 2: the last eight stages   act inside rows   (distance <= 128)
// and mirrored for the inverse.  Each workgroup owns 4096 points, R rows of 4096 / R columns (or 16 rows, 8 or 4 with eight or four
// points per thread); a thread keeps 16 residues in registers, or two or four lanes of a wavefront 8 or 4 each, runs a block of up to four
// stages on them, swaps through LDS once and runs the second block.  All global accesses
// are segments of at least 128 bytes shared by adjacent lanes, 64 in the half slabs of 2^16 points.
//
// Rings of 2^10 .. 2^12 points, and large batches of 2^13 and 2^14, take one launch (ntt_limb.hip), the smallest rings
// (2^6 .. 2^9, small-parameter tests) a plain LDS kernel; the butterfly network is the same for all, so residues are identical for every N.
#include <algorithm>
#include <cstring>

#include "ntt_device.h"

namespace {
// ------------------------------------------------------------------------------------------
// rings below 2^10 points: a workgroup transforms one limb in LDS, stage by stage
// ------------------------------------------------------------------------------------------
template <bool INV>
__global__ __launch_bounds__(256) void ntt_small_kernel(u64 *__restrict__ data, const Tw *__restrict__ tw_all,
                                                        const ModQ *__restrict__ modq,
                                                        const u64 *__restrict__ ninv, const u64 *__restrict__ ninv_s,
                                                        LimbList ll, LimbList sl, int n_limbs, size_t poly_stride,
                                                        int logN) {
    __shared__ u64 lds[512];
    const int N = 1 << logN;
    const int limb = blockIdx.y % n_limbs, poly = blockIdx.y / n_limbs;
    const int prime = (int)table_byte(ll.idx, limb);
    const Tw *tw = tw_all + (size_t)prime * N;
    const u64 q = modq[prime].q, q2 = 2 * q, q4 = 4 * q, nq4 = opaque_neg(q4);
    u64 *base = data + (size_t)poly * poly_stride + (size_t)table_byte(sl.idx, limb) * N;
    for (int e = threadIdx.x; e < N; e += blockDim.x) lds[e] = base[e];
    __syncthreads();
    for (int step = 0; step < logN; step++) {
        const int s = INV ? logN - 1 - step : step, t = N >> (s + 1);
        for (int b = threadIdx.x; b < N / 2; b += blockDim.x) {
            const int i = (b / t) * 2 * t + b % t, j = i + t;
            const Tw w = tw[(1 << s) + b / t];
            u64 x = lds[i], y = lds[j];
            if (INV)
                gs_bfly(x, y, w, q, q4, nq4);
            else
                ct_bfly(x, y, w, q, q4, nq4);
            lds[i] = x;
            lds[j] = y;
        }
        __syncthreads();
    }
    const u64 ni = ninv[prime], nis = ninv_s[prime];
    for (int e = threadIdx.x; e < N; e += blockDim.x) {
        u64 v = lds[e];
        if (INV) {
            v = mul_shoup_lazy(v, ni, nis, q);
        } else {
            if (v >= q4) v -= q4;
            if (v >= q2) v -= q2;
        }
        if (v >= q) v -= q;
        base[e] = v;
    }
}

// ------------------------------------------------------------------------------------------
// two-launch kernels (N = 2^13 .. 2^16)
// ------------------------------------------------------------------------------------------
// Column passes work on a slab of R = 2^LR rows and CW = 4096 / R columns (R = 256: 16 columns), or of CW >> H in small launches
// (narrower_slabs): the 16 residues of a thread or lane pair
// are rows rh + (R / 16) k for the block of the four widest stages and rows 16 rh + k for the LR - 4 others.
template <int LR, int P, int H = 0>
struct Slab {
    typedef Lanes<P> L;
    static constexpr int R = 1 << LR, Q = R / 16, CW = (4096 >> H) / R, T = LR - 4, WORDS = 4096 >> H;
    static __device__ __forceinline__ u32 cc() { return L::t() & (CW - 1); }
    static __device__ __forceinline__ u32 rh() { return L::t() >> (12 - LR - H); }
    // Slabs of eight columns: the two that share lines of 128 bytes lie on one XCD (workgroups go round the eight by their number),
    // whose L2 then fetches a line once and writes it whole
    static __device__ __forceinline__ u32 slab() {
        return CW >= 16 ? blockIdx.x : ((blockIdx.x & 7u) << 1) + ((blockIdx.x >> 4) << 4) + ((blockIdx.x >> 3) & 1u);
    }
    static __device__ __forceinline__ u32 col() { return slab() * CW + cc(); }
    // twiddle group of the second block: 16 / Q sub-blocks per thread
    static __device__ __forceinline__ u32 group() { return 16u + rh() * (16 / Q); }
    // place of (row r, column cc) in the exchange buffer.  At 16 columns a wavefront reads rows 16 apart together: row r is
    // kept at row r ^ (bit 4 of r), so that they alternate between the two halves of the 64 LDS banks instead of sharing one
    // (forward only: an inverse pass, which writes those rows, loses more to the xor in each address than to the
    // conflicts: 9.7 against 8.8 us for 10 limbs of 42-bit primes)
    template <bool INV>
    static __device__ __forceinline__ int at(const int r) {
        if (P == 4 && CW == 8)
            return (r ^ ((((r >> 6) ^ (r >> 4)) & 1) << 1)) * CW + (int)cc();
        if (P == 4)   // its lanes 16 apart hold rows a whole or the fourth part of a block apart, in both passes: one bit of either goes in
            return (r ^ (((LR >= 7 ? 0 : r >> 2) ^ (r >> (LR - 2))) & 1)) * CW + (int)cc();
        return (CW == 16 && !INV ? swz_row(r) : r) * CW + (int)cc();
    }
    // rows of a thread's register k: of the four widest stages (split, whole), of the others (split, whole)
    static __device__ __forceinline__ int r_outer_s(const int k) { return (int)(rh() + Q * L::template h_split<4>()) + Q * L::template split<4>(k); }
    static __device__ __forceinline__ int r_outer_w(const int k) { return (int)(rh() + Q * L::h_whole()) + Q * k; }
    static __device__ __forceinline__ int r_inner_s(const int k) { return (int)(16 * rh() + L::template h_split<T>()) + L::template split<T>(k); }
    static __device__ __forceinline__ int r_inner_w(const int k) { return (int)(16 * rh() + L::h_whole()) + k; }
    // byte offsets inside a limb of the widest stages' points (split) and of the others' (whole): a thread's part, and the
    // step to register k, which goes into the scalar offset
    static __device__ __forceinline__ u32 v_outer() { return (col() + ((u32)r_outer_s(0) << 8)) * 8u; }
    static __device__ __forceinline__ u32 v_inner() { return (col() + ((u32)r_inner_w(0) << 8)) * 8u; }
    static __device__ __forceinline__ constexpr u32 outer(const int k) { return (u32)L::template split<4>(k) * (Q << 11); }
    static __device__ __forceinline__ constexpr u32 inner(const int k) { return (u32)k << 11; }
};
// the exchange and the second block of a forward column pass, results to memory
template <int LR, int H = 0, int P, class F, class LANE = KeptLane>
__device__ __forceinline__ void cols_forward(const __amdgpu_buffer_rsrc_t limb, const typename F::W *__restrict__ tw,
                                             const F f, typename F::E (&x)[P], typename F::E *lds, const LANE lane = LANE{Lanes<P>::h()}) {
    typedef typename F::E E;
    typedef Slab<LR, P, H> S;
    radix_fwd<4>(f, x, tw, 1u, lane);
#pragma unroll
    for (int k = 0; k < P; k++) lds[S::template at<false>(S::r_outer_w(k))] = x[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < P; k++) x[k] = lds[S::template at<false>(S::r_inner_s(k))];
    radix_fwd<S::T>(f, x, tw, S::group(), lane);
#pragma unroll
    for (int k = 0; k < P; k++) buf_store<E>(limb, S::v_inner(), S::inner(k), x[k]);
}
template <int LR, int P, int H, bool INV, class F>
__device__ __forceinline__ void cols_body(const __amdgpu_buffer_rsrc_t limb, const Tw *__restrict__ tw_int, const F f,
                                          u64 *lds_raw) {
    typedef typename F::E E;
    typedef Slab<LR, P, H> S;
    const typename F::W *tw = (const typename F::W *)tw_int;
    E *lds = (E *)lds_raw;
    E x[P];
    if (!INV) {
#pragma unroll
        for (int k = 0; k < P; k++) x[k] = f.from_canonical(buf_load<u64>(limb, S::v_outer(), S::outer(k)));
        cols_forward<LR, H>(limb, tw, f, x, lds);
    } else {
#pragma unroll
        for (int k = 0; k < P; k++) x[k] = buf_load<E>(limb, S::v_inner(), S::inner(k));
        radix_inv<S::T>(f, x, tw, S::group());
        f.template after_inverse_block<S::T>(x);
#pragma unroll
        for (int k = 0; k < P; k++) lds[S::template at<true>(S::r_inner_s(k))] = x[k];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < P; k++) x[k] = lds[S::template at<true>(S::r_outer_w(k))];
        radix_inv<4>(f, x, tw, 1u);
#pragma unroll
        for (int k = 0; k < P; k++) buf_store<u64>(limb, S::v_outer(), S::outer(k), f.scale_to_canonical(x[k]));
    }
}

template <int LR, int P, int H, bool INV>
__global__ __launch_bounds__((4096 >> H) / P) void ntt16_cols_kernel(u64 *__restrict__ data, const Tw *__restrict__ tw_all,
                                                         const ModQ *__restrict__ modq,
                                                         const u64 *__restrict__ ninv, const u64 *__restrict__ ninv_s,
                                                         const double *__restrict__ fp, LimbList ll, LimbList sl,
                                                         int n_limbs, size_t poly_stride, const Tw *__restrict__ final_scale) {
    __shared__ u64 lds[4096 >> H];
    const int limb = blockIdx.y % n_limbs, poly = blockIdx.y / n_limbs;
    const int prime = (int)table_byte(ll.idx, limb);
    const Tw *tw = tw_all + ((size_t)prime << (8 + LR));
    const __amdgpu_buffer_rsrc_t base = limb_rsrc(
        data + (size_t)poly * poly_stride + ((size_t)table_byte(sl.idx, limb) << (8 + LR)));
    // final_scale (inverse transforms only): limb i ends with the constant final_scale[i] in place of 1/N -- a basis
    // conversion folds its (S/q_i)^-1 factor in here (the caller supplies (1/N)(S/q_i)^-1), at no cost
    if (fp[4 * prime] != 0.0) {
        FpField f(modq, ninv, ninv_s, fp, prime);
        if (INV && final_scale != nullptr) f.set_scale(final_scale[limb]);
        cols_body<LR, P, H, INV>(base, tw, f, lds);
    } else {
        with_int_field(modq, ninv, ninv_s, fp, prime, [&](auto f) {
            if (INV && final_scale != nullptr) f.set_scale(final_scale[limb]);
            cols_body<LR, P, H, INV>(base, tw, f, lds);
        });
    }
}

// Forward pass 1 over a slab whose input is a basis conversion computed on the fly.  The workgroups
// of the target limbs that share a (polynomial, slab) pair have consecutive blockIdx.y and the same blockIdx.x, so
// they sit on one XCD at about the same time and all but the first find the source slabs in its L2.
template <int LR, int P, int H, int NS, class F>
__device__ __forceinline__ void cols_converted_body(const __amdgpu_buffer_rsrc_t limb, const Tw *__restrict__ tw_int,
                                                    const F f, u64 *lds_raw, const __amdgpu_buffer_rsrc_t src,
                                                    const u32 (&so)[NS], const DotCst (&h)[NS], const int n_src, const ModQ m) {
    typedef Slab<LR, P, H> S;
    typename F::E x[P];
    // the row step goes into the scalar offset
    converted_inputs<NS>(f, x, src, S::v_outer(), so, h, n_src, m, [](const int k) { return S::outer(k); });
    cols_forward<LR, H>(limb, (const typename F::W *)tw_int, f, x, (typename F::E *)lds_raw, OwnLane<P>{});
}

// What bounds it is the work of a column pass and the trips to memory in front of it.  Eight points per thread and 20 source
// residues in flight fit 80 registers, six waves per SIMD (sixteen points: 154 - 166 registers, three waves; 40 residues: four).  1536
// workgroups (16 polynomials x 6 limbs, 5 sources) 42 -> 37 us alone, 1002 -> 789 vector instructions per wave, with sums that carry
// nothing (modarith.h, DotCst) and loads that wait once; rotation at 24 primes of 60 bits, level 20 161 -> 154 us, projection of a
// 768-wide layer 2.5 % less.
template <int LR, int P, int H, int NS>
__global__ __launch_bounds__((4096 >> H) / P) __attribute__((amdgpu_waves_per_eu(P == 4 ? 4 : 6, P == 4 ? 8 : 6))) void ntt16_cols_converted_kernel(
    u64 *__restrict__ data, const Tw *__restrict__ tw_all, const ModQ *__restrict__ modq, const u64 *__restrict__ ninv,
    const u64 *__restrict__ ninv_s, const double *__restrict__ fp, LimbList ll, LimbList sl, int n_limbs,
    size_t poly_stride, ConvSources cs) {
    __shared__ u64 lds[4096 >> H];
    const int per_poly = n_limbs + cs.n_copy;
    const int limb = blockIdx.y % per_poly, poly = blockIdx.y / per_poly;
    typedef Slab<LR, P, H> S;
    if (limb >= n_limbs) {   // a limb that is only copied into its slot
        const u64 *from = cs.copy_src + (size_t)poly * cs.copy_src_stride +
                          ((size_t)table_byte(cs.copy_src_slot, limb - n_limbs) << (8 + LR));
        u64 *base = data + (size_t)poly * poly_stride + ((size_t)table_byte(cs.copy_dst_slot, limb - n_limbs) << (8 + LR)) + S::col();
        u64 t[P];
        if (cs.copy_galois != 0) {   // the copy of the source's automorphism
#pragma unroll
            for (int k = 0; k < P; k++)
                t[k] = from[galois_index(((u32)S::r_outer_w(k) << 8) + S::col(), cs.copy_galois, 8 + LR)];
        } else {
#pragma unroll
            for (int k = 0; k < P; k++) t[k] = from[((u32)S::r_outer_w(k) << 8) + S::col()];
        }
#pragma unroll
        for (int k = 0; k < P; k++) base[(u32)S::r_outer_w(k) << 8] = t[k];
        return;
    }
    const __amdgpu_buffer_rsrc_t base = limb_rsrc(
        data + (size_t)poly * poly_stride + ((size_t)table_byte(sl.idx, limb) << (8 + LR)));
    const int prime = (int)table_byte(ll.idx, limb);
    const Tw *tw = tw_all + ((size_t)prime << (8 + LR));
    const int dg = (int)table_byte(cs.digit_of, limb), n_src = cs.d[dg].n_src;
    // The sources are read through a buffer resource: base (the polynomial's source limbs; far below 4 GiB), source slot
    // and slab row sit in scalar registers, a thread supplies one 32-bit offset for all of its P n_src loads.
    const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(cs.d[dg].src + (size_t)poly * cs.d[dg].src_poly_stride), 0, -1, 0x00020000);
    const Cst *hat = cs.d[dg].hat + prime;
    const ModQ m = modq[prime];
    u32 so[NS];
    DotCst h[NS];
#pragma unroll
    for (int i = 0; i < NS; i++) {
        const int ii = i < n_src ? i : 0;
        so[i] = table_byte(cs.d[dg].src_slot, ii) << (11 + LR);
        const Cst hg = hat[(size_t)ii * cs.hat_ld];
        h[i] = dot_cst(hg.w, hg.ws);
    }
    if (fp[4 * prime] != 0.0)
        cols_converted_body<LR, P, H, NS>(base, tw, FpField(modq, ninv, ninv_s, fp, prime), lds, src, so, h, n_src, m);
    else   // (the sums take primes below 2^60)
        with_field_60(modq, ninv, ninv_s, fp, prime, [&](const auto f) { cols_converted_body<LR, P, H, NS>(base, tw, f, lds, src, so, h, n_src, m); });
}

// Forward pass 1 whose input is the rounded coefficients of an encoding, the same for every limb of a polynomial: reduced
// as they are loaded instead of being written limb by limb and read back.
template <int LR, int P, int H, class F>
__device__ __forceinline__ void cols_lifted_body(const __amdgpu_buffer_rsrc_t limb, const Tw *__restrict__ tw_int, const F f,
                                                 u64 *lds_raw, const LiftSource &ls, const long long *__restrict__ coef,
                                                 const ModQ m) {
    typedef Slab<LR, P, H> S;
    typename F::E x[P];
    lifted_inputs(f, x, ls, coef, m, [](const int k) { return ((u32)S::r_outer_s(k) << 8) + S::col(); });
    cols_forward<LR, H>(limb, (const typename F::W *)tw_int, f, x, (typename F::E *)lds_raw);
}
template <int LR, int P, int H>
__global__ __launch_bounds__((4096 >> H) / P) void ntt16_cols_lifted_kernel(u64 *__restrict__ data, const Tw *__restrict__ tw_all,
                                                                const ModQ *__restrict__ modq, const double *__restrict__ fp,
                                                                LimbList ll, LimbList sl, int n_limbs, size_t poly_stride,
                                                                LiftSource ls) {
    __shared__ u64 lds[4096 >> H];
    const int limb = blockIdx.y % n_limbs, poly = blockIdx.y / n_limbs;
    const int prime = (int)table_byte(ll.idx, limb);
    const Tw *tw = tw_all + ((size_t)prime << (8 + LR));
    const __amdgpu_buffer_rsrc_t base = limb_rsrc(
        data + (size_t)poly * poly_stride + ((size_t)table_byte(sl.idx, limb) << (8 + LR)));
    const long long *coef = ls.coef + (size_t)poly * ls.stride;
    const ModQ m = modq[prime];
    if (fp[4 * prime] != 0.0)
        cols_lifted_body<LR, P, H>(base, tw, FpField(modq, nullptr, nullptr, fp, prime), lds, ls, coef, m);
    else
        with_int_field(modq, nullptr, nullptr, fp, prime, [&](const auto f) { cols_lifted_body<LR, P, H>(base, tw, f, lds, ls, coef, m); });
}
// ------------------------------------------------------------------------------------------
// Column-slab kernel of a ModDown: for one (polynomial, half slab of eight columns) a workgroup runs the second pass of the inverse
// transform of every source limb, keeps the canonical coefficients in registers and then, target limb by target limb, takes the basis
// conversion as lazy dot products and runs the first pass of the forward transform.  The inverse result is never written and
// the sources are never read back: the three steps are local to the slab, only the row passes on either side need the other half
// of the 256 x 256 view.  Arithmetic, order of operations and stored values are those of ntt16_cols_kernel<true> followed by
// ntt16_cols_converted_kernel.
// Four points per thread: five sources are 40 registers (122 in all, four waves per SIMD, two workgroups on a CU), kept in the pieces that the
// dot products take; a source's loads are in flight under the one before it.  Bound by issue: 3610 vector instructions per wave, VALUBusy 74 %,
// 43.5 us for 16 polynomials of 5 sources and 6 targets where the two kernels take 16 + 37.  (Sixteen points per thread, 256 registers and
// two waves per SIMD, was slower than the two kernels at any size.)
// ------------------------------------------------------------------------------------------
#define SLAB_MAX_SOURCES 5
struct SlabSources {
    const u64 *src;            // first-pass output of the inverse transform (raw field values), [n_polys][.][N]
    size_t src_poly_stride;
    const Cst *hat;            // [n_src][hat_ld]  (S/q_i) mod prime and 2^30 times that, indexed by prime
    const Tw *final_scale;     // [n_src]  (1/N)(S/q_i)^-1 mod q_i
    int hat_ld, n_dst;         // targets: chain primes 0 .. n_dst - 1, in the slots of these numbers
    uint8_t src_slot[8], src_prime[8];   // SLAB_MAX_SOURCES of them, whole words (table_byte)
};

// Half slabs of 2^16 points, four points per thread.  What a thread keeps through all limbs: its place in the exchange buffer (rows 4 h + k
// of the widest stages' block, k even and odd, and rows h + 4 k of the others': Slab::at written out) and the offset of its column.  The
// rest of its place is made anew for every limb: kept as well, the offsets of the twelve twiddles of either arithmetic spill.
struct SlabPlace {
    typedef Slab<8, 4, 1> S;
    u32 outer_even, outer_odd, inner, v_inner;
    __device__ __forceinline__ SlabPlace() {
        const u32 h = Lanes<4>::h(), rh = S::rh(), cc = S::cc(), flip = ((rh >> 2) ^ rh) & 1u;
        outer_even = ((rh ^ ((h & 1u) << 1)) + 64u * h) * 8u + cc;
        outer_odd = outer_even ^ 16u;
        inner = (16u * rh + (h ^ (flip << 1))) * 8u + cc;
        v_inner = S::v_inner();
    }
    __device__ __forceinline__ u32 outer(const int k) const { return (k & 1 ? outer_odd : outer_even) + 128u * (u32)k; }
    __device__ __forceinline__ u32 within(const int k) const { return inner + 32u * (u32)k; }
};
struct SlabLane {   // lane of a block, twiddle group of the second block
    u32 h, group;
    __device__ __forceinline__ SlabLane() {
        u32 t = threadIdx.x;
        asm volatile("" : "+v"(t));
        h = (t & 63u) >> 4;
        group = 16u + (((t & 15u) | ((t >> 6) << 4)) >> 3);
    }
};

// second pass of an inverse transform: x as loaded, r canonical coefficients in the layout a forward transform begins with
template <class F>
__device__ __forceinline__ void slab_inverse(const u64 (&raw)[4], const Tw *__restrict__ tw_int, const F f, u64 *lds_raw,
                                             const SlabPlace &at, Pieces (&r)[4]) {
    typedef typename F::E E;
    const typename F::W *tw = (const typename F::W *)tw_int;
    E *lds = (E *)lds_raw;
    const SlabLane lane;
    E x[4];
#pragma unroll
    for (int k = 0; k < 4; k++) __builtin_memcpy(&x[k], &raw[k], 8);
    radix_inv<4>(f, x, tw, lane.group, KeptLane{lane.h});
    f.template after_inverse_block<4>(x);
#pragma unroll
    for (int k = 0; k < 4; k++) lds[at.within(k)] = x[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; k++) x[k] = lds[at.outer(k)];
    radix_inv<4>(f, x, tw, 1u, KeptLane{lane.h});
#pragma unroll
    for (int k = 0; k < 4; k++) {
        r[k] = pieces(f.scale_to_canonical(x[k]));
        asm("" : "+v"(r[k].lo), "+v"(r[k].hi));   // kept as pieces, not as a residue that is cut again for every target
    }
}

template <int NS, class F>
__device__ __forceinline__ void slab_forward(const __amdgpu_buffer_rsrc_t limb, const Tw *__restrict__ tw_int, const F f, u64 *lds_raw,
                                             const SlabPlace &at, const Pieces (&c)[NS][4], const DotCst (&h)[NS], const ModQ m) {
    typedef typename F::E E;
    const typename F::W *tw = (const typename F::W *)tw_int;
    E *lds = (E *)lds_raw;
    const SlabLane lane;
    E x[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        Dot2 d;
        dot_clear(d);
#pragma unroll
        for (int i = 0; i < NS; i++) dot_add(d, c[i][k], h[i]);
        x[k] = f.from_dot(d, m);
    }
    radix_fwd<4>(f, x, tw, 1u, KeptLane{lane.h});
#pragma unroll
    for (int k = 0; k < 4; k++) lds[at.outer(k)] = x[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; k++) x[k] = lds[at.within(k)];
    radix_fwd<4>(f, x, tw, lane.group, KeptLane{lane.h});
#pragma unroll
    for (int k = 0; k < 4; k++) buf_store<E>(limb, at.v_inner, (u32)k << 11, x[k]);
}

__device__ __forceinline__ void slab_load(const u64 *__restrict__ src, const SlabSources &ss, const SlabPlace &at, const int i, u64 (&next)[4]) {
    const __amdgpu_buffer_rsrc_t limb = limb_rsrc(src + ((size_t)table_byte(ss.src_slot, i) << 16));
#pragma unroll
    for (int k = 0; k < 4; k++) next[k] = buf_load<u64>(limb, at.v_inner, (u32)k << 11);
}
// sources I, I + 1, ... of NS; the next one's loads are in flight under a source's butterflies
template <int I, int NS>
__device__ __forceinline__ void slab_sources(const u64 *__restrict__ src, const SlabSources &ss, const Tw *__restrict__ itw_all,
                                             const ModQ *__restrict__ modq, const u64 *__restrict__ ninv, const u64 *__restrict__ ninv_s,
                                             const double *__restrict__ fp, u64 (&lds)[2][2048], const SlabPlace &at, u64 (&next)[4],
                                             Pieces (&c)[NS][4]) {
    if constexpr (I < NS) {
        const int prime = (int)table_byte(ss.src_prime, I);
        const Tw *tw = itw_all + ((size_t)prime << 16);
        const Tw fs = ss.final_scale[I];
        u64 raw[4];
#pragma unroll
        for (int k = 0; k < 4; k++) raw[k] = next[k];
        if (I + 1 < NS) slab_load(src, ss, at, I + 1, next);
        if (fp[4 * prime] != 0.0) {
            FpField f(modq, ninv, ninv_s, fp, prime);
            f.set_scale(fs);
            slab_inverse(raw, tw, f, lds[I & 1], at, c[I]);
        } else {
            with_field_60(modq, ninv, ninv_s, fp, prime, [&](auto f) {
                f.set_scale(fs);
                slab_inverse(raw, tw, f, lds[I & 1], at, c[I]);
            });
        }
        slab_sources<I + 1>(src, ss, itw_all, modq, ninv, ninv_s, fp, lds, at, next, c);
    }
}

template <int NS>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4, 8))) void ntt16_slab_convert_kernel(
    u64 *__restrict__ data, const size_t poly_stride, const Tw *__restrict__ tw_all, const Tw *__restrict__ itw_all,
    const ModQ *__restrict__ modq, const u64 *__restrict__ ninv, const u64 *__restrict__ ninv_s,
    const double *__restrict__ fp, const SlabSources ss) {
    // Two exchange buffers in turn: a limb's exchange needs one barrier, since the one before the last is behind it for every wave
    __shared__ u64 lds[2][2048];
    const SlabPlace at;
    const int poly = blockIdx.y;
    const u64 *src = ss.src + (size_t)poly * ss.src_poly_stride;
    Pieces c[NS][4];
    u64 next[4];
    slab_load(src, ss, at, 0, next);
    slab_sources<0>(src, ss, itw_all, modq, ninv, ninv_s, fp, lds, at, next, c);
#pragma unroll 1
    for (int t = 0; t < ss.n_dst; t++) {
        const __amdgpu_buffer_rsrc_t limb = limb_rsrc(data + (size_t)poly * poly_stride + ((size_t)t << 16));
        const Tw *tw = tw_all + ((size_t)t << 16);
        const ModQ m = modq[t];
        const Cst *hat = ss.hat + t;
        DotCst h[NS];
#pragma unroll
        for (int i = 0; i < NS; i++) {
            const Cst hg = hat[(size_t)i * ss.hat_ld];
            h[i] = dot_cst(hg.w, hg.ws);
        }
        u64 *buffer = lds[(NS + t) & 1];
        if (fp[4 * t] != 0.0)
            slab_forward<NS>(limb, tw, FpField(modq, nullptr, nullptr, fp, t), buffer, at, c, h, m);
        else
            with_field_60(modq, nullptr, nullptr, fp, t, [&](const auto f) { slab_forward<NS>(limb, tw, f, buffer, at, c, h, m); });
    }
}

// LR: log2 of the rows of a limb, or 0: taken from the argument (the address arithmetic of N = 2^16 folds into constants:
// 1 - 1.5 % of a single rotation or ciphertext product)
template <int LR, int P, bool INV, int KTAIL, int LOAD>
__global__ __launch_bounds__(256) void ntt16_rows_kernel(u64 *__restrict__ data, const Tw *__restrict__ tw_all,
                                                         const Tw *__restrict__ rtw_all,
                                                         const ModQ *__restrict__ modq, const double *__restrict__ fp,
                                                         LimbList ll, LimbList sl, int n_limbs, size_t poly_stride,
                                                         typename EpilogueOf<KTAIL>::T ep, const int log_r_arg) {
    constexpr int TAIL = tail_of(KTAIL);
    constexpr int RB = P == 16 ? 4 : P == 8 ? 3 : 2;   // log2 of the rows of a workgroup
    __shared__ u64 lds[ROWPAD << RB];
    const int log_r = LR != 0 ? LR : log_r_arg;
    // The second radix-16 block of a row pass walks 1/16 of the prime's twiddle table per 16-row slab (as
    // many bytes as the slab's data), identical for every polynomial of the batch.  Workgroups are dealt
    // round-robin to the 8 XCDs, so the polynomials of one (limb, slab) pair are placed back to back on
    // one XCD and share those twiddles through its L2 instead of fetching them from HBM once each.
    const u32 groups = (u32)n_limbs << (log_r - RB), n_polys = gridDim.x / groups;
    u32 poly, group;
    if ((groups & 7u) == 0) {
        const u32 xcd = blockIdx.x & 7u, slot = blockIdx.x >> 3;
        poly = slot % n_polys;
        group = (slot / n_polys) * 8u + xcd;
    } else {   // small rings: a prime's whole table is a few dozen KiB
        poly = blockIdx.x % n_polys;
        group = blockIdx.x / n_polys;
    }
    const int limb = (int)(group >> (log_r - RB));
    const u32 slab = group & ((1u << (log_r - RB)) - 1u);
    const int log_n = 8 + log_r;
    const int prime = (int)table_byte(ll.idx, limb);
    const Tw *tw = tw_all + ((size_t)prime << log_n), *rtw = rtw_all + ((size_t)prime << log_n);
    const u32 r = (slab << RB) + (Lanes<P>::t() >> 4);  // global row
    u64 *row = data + (size_t)poly * poly_stride + ((size_t)table_byte(sl.idx, limb) << log_n) + ((size_t)r << 8);
    const u64 *mn = nullptr;
    u64 *o = nullptr;
    Tw cst{0, 0};
    RowSecond sec{};
    if (TAIL != TAIL_NONE) {
        const size_t off = ((size_t)limb << log_n) + ((size_t)r << 8);
        o = ep.result((int)poly) + off;
        if (TAIL == TAIL_SUB_SCALE) {
            mn = ep.minuend + (size_t)poly * ep.minuend_stride + off;
            cst = ep.cst[limb];
        } else {
            sec.out = ep.second_out + (size_t)poly * ep.out_stride + off;
            sec.key = sm64(sm64(ep.a_base + (u64)prime));
        }
    }
    const u64 *ld = row;
    if (INV && ep.minuend != nullptr)
        ld = ep.minuend + (size_t)poly * ep.minuend_stride + ((size_t)table_byte(sl.idx, limb) << log_n) + (LOAD == LOAD_ROTATED ? 0 : (size_t)r << 8);
    if (LOAD == LOAD_DECRYPT)
        sec.in = ep.second_in + (size_t)poly * ep.minuend_stride + ((size_t)table_byte(sl.idx, limb) << log_n) + ((size_t)r << 8);
    if (TAIL == TAIL_ENCRYPT || LOAD == LOAD_DECRYPT) {
        sec.sk = ep.sk + ((size_t)prime << log_n) + ((size_t)r << 8);
        sec.m = modq[prime];
    }
    const u32 gal = LOAD == LOAD_ROTATED ? ep.galois : 0u;
    if (fp[4 * prime] != 0.0)
        rows_body<P, INV, TAIL, LOAD, false>(row, tw, rtw, FpField(modq, nullptr, nullptr, fp, prime), lds, log_r, r, mn, o, cst, ld, gal,
                                            sec);
    else
        with_int_field(modq, nullptr, nullptr, fp, prime, [&](const auto f) {
            rows_body<P, INV, TAIL, LOAD, false>(row, tw, rtw, f, lds, log_r, r, mn, o, cst, ld, gal, sec);
        });
}

}  // namespace

// one-launch forms (ntt_limb.hip)
void launch_limb_forward(const hemm_context *c, u64 *data, const LimbList &ll, const LimbList &sl, int n_limbs, int n_polys,
                         size_t poly_stride, hipStream_t s, const ConvSources *cs, const LiftSource *ls, const NttEpilogue &ep,
                         int tail, const ResultList *list = nullptr);
void launch_limb_inverse(const hemm_context *c, u64 *data, const LimbList &ll, const LimbList &sl, int n_limbs, int n_polys,
                         size_t poly_stride, hipStream_t s, const void *final_scale, const NttEpilogue &from, int load);

// ---- launches of single passes (rings of 2^13 points and more) -------------------------------------------------------
// Which passes give a thread four or eight points instead of sixteen (ntt_device.h, Lanes): few points only where the launch leaves the
// chip part empty, since in a full one the twiddles and addresses of each lane of a block are work for nothing.  All figures down to
// narrower_slabs but the one marked there: us of device time a call, calls queued, one build with its lines moved; 60 bits in the arithmetic
// of primes that are not just below 2^60 (those lie between these figures and the ones of 42 bits).
// Transforms of 2^16 points with sixteen / eight / four points in that pass (workgroups of 4096 points, columns on whole slabs):
//   workgroups                 64               128              256              384              512              768              1024
//   columns, forward, 60 bits  11.1/10.6/10.4   13.7/13.2/13.1   19.3/18.9/18.5   25.6/25.6/25.2   27.1/27.1/26.6   29.9/29.7/29.9   35.6/35.6/36.3
//                     42 bits   9.3/ 9.1/ 9.0   11.6/11.3/11.3   16.7/16.3/16.0   22.2/21.9/21.8   24.9/24.5/24.4   23.8/23.1/24.5   27.9/27.9/29.9
//            inverse, 60 bits  11.9/11.2/11.0   14.6/14.0/13.8   20.2/19.6/19.1   27.2/26.8/26.9   29.7/28.9/28.8   32.4/31.9/32.4   39.2/39.1/40.2
//                     42 bits   9.5/ 9.2/ 9.4   12.0/11.7/11.9   17.1/16.8/16.6   22.6/22.7/22.9   26.0/25.6/25.8   24.7/24.3/25.8   28.9/28.8/31.0
//   rows,    forward, 60 bits  11.9/10.7/ 9.5   13.8/12.6/12.3   19.2/19.0/18.6   25.3/24.9/24.5   27.6/27.5/26.7   30.1/29.7/29.5   35.9/36.1/36.2
//                     42 bits  10.0/ 9.1/ 8.3   11.8/10.9/10.7   17.9/16.3/16.1   22.4/21.3/21.4   25.2/24.5/24.5   23.9/23.6/24.0   28.0/27.5/28.5
//            inverse, 60 bits  12.3/10.8/ 9.7   14.3/12.7/12.5   19.9/19.4/19.3   26.5/25.8/25.6   30.7/30.0/28.9   33.6/32.4/32.8   39.8/39.6/38.7
//                     42 bits  10.2/ 9.3/ 8.5   12.0/11.0/11.1   17.0/16.7/16.5   22.8/22.1/21.9   26.6/26.2/25.7   25.2/24.7/25.0   29.0/29.1/29.5
static bool few_for_columns(const hemm_context *c, int limbs) { return (size_t)limbs * (c->N >> 12) <= 512; }
// Row passes: four points have eight wavefronts per SIMD, all resident up to 512 workgroups of 4096 points, and lead up to 640; eight points
// lead from there to about 1000 (figures below; further since the butterflies take fewer
// instructions, table after it).  Encodings of 2^14 points leave four at 512 and eight, for sixteen, at 640.  us with sixteen / eight /
// four points, the second figure of each pair 42 bits:
//   workgroups                        544                              640                              768                              896
//   forward, 2^16 points   33.3/32.8/31.5 28.5/28.1/27.2  28.5/27.3/27.0 24.4/23.2/23.5  30.1/29.7/29.5 23.9/23.6/24.0  34.5/33.6/33.6 26.8/25.5/26.7
//            2^15          32.5/31.6/30.6 28.4/27.2/26.8  29.5/28.0/27.7 25.7/24.6/24.6  28.8/28.6/28.7 23.5/23.2/23.8  33.3/32.3/33.0 25.9/25.0/26.1
//   inverse, 2^16          37.0/35.3/34.1 29.7/29.5/28.5  32.6/31.5/30.7 26.1/25.2/24.9  33.6/32.4/32.8 25.2/24.7/25.0  38.4/36.7/36.6 27.9/26.8/27.3
//            2^15          37.4/34.3/33.2 31.0/28.6/28.2  34.0/30.9/31.2 27.3/25.6/26.1  32.5/30.9/31.8 25.0/24.1/25.0  36.6/35.2/35.9 27.1/26.5/27.5
//   rescale, 2^16          44.3/41.0/40.4 37.6/34.3/34.0  44.0/42.1/42.8 38.2/34.9/35.6  47.0/45.8/47.5 39.7/37.6/38.7
//            2^15          46.1/42.4/41.6 38.1/35.2/34.6  46.7/43.9/43.9 39.7/36.2/35.9  48.8/46.0/46.6 41.4/37.6/38.6
//   encodings of 2^14 points, m messages x limbs: 11x12 34.8/34.5/34.9, 23x6 37.9/36.6/37.6, 26x6 38.6/37.2/38.2, 32x5 37.6/37.3/38.7, 32x6 38.5/38.1/39.4,
//   64x3 39.9/39.9/41.1, 16x13 37.4/39.2/40.3; of 2^16 4x13 40.8/39.5/40.3, 9x6 42.4/41.3/42.2
// Forward passes beyond 900 workgroups, sixteen / eight points, with the present butterflies (60 bits: of primes just below 2^60):
//   2^16 points, workgroups           960        1280       1536       1792       3072 (runs)  | ModDowns, tails of 960 / 1536 / 3072 / 5120
//   60 bits                           29.9/28.8  37.7/35.9  42.1/41.0  46.3/46.1  293/297      | (42-bit chain) 70.4/68.5 88.3/86.6 167/164 301/301
//   42 bits                           26.3/25.8  33.3/32.5  37.4/36.6  41.3/40.4  269/269      | encodings of 72 / 117 / 208 limbs 45.0/44.0 57.3/55.5 84.1/82.5
//   2^15 points, 960 / 1280 / 1920 / 2560: 60 bits 30.0/29.1 38.5/38.2 53.0/51.4 63.2/63.2, 42 bits 25.8/25.3 34.0/33.4 46.3/45.3 57.8/56.0
//   2^14 points: ModDowns of 16 / 32 polynomials 39.0/39.4 53.4/54.0 (its line stays at 900)
//   other primes, 50 / 59 / 61 bits: 2^15 points, 1920 55.5/55.4 56.2/56.2 59.9/59.9, 2560 69.1/71.0 69.4/72.0 74.3/78.1; 2^16, 2400 69.0/68.8 70.1/70.5 76.5/77.5
// primes of 44 bits and more that are not just below 2^60 (IntFieldT), whose butterflies take the most instructions
static bool is_far(const u64 q) { return (q >> 44) != 0 && !near_2_60(q); }
static int points_for_rows(const hemm_context *c, const LimbList &ll, int n_limbs, int n_polys, bool inverse, int tail) {
    const size_t wgs = (size_t)n_limbs * n_polys * (c->N >> 12);
    const bool encoding = c->logN == 14 && !inverse && tail == TAIL_NONE;   // longer plain transforms of this ring are one launch
    if (wgs <= (encoding ? 512 : 640) || (tail == TAIL_ENCRYPT && c->logN < 16)) return 4;   // (an encryption's few limbs)
    if (inverse) return 8;
    if (c->logN >= 15) {
        if (tail != TAIL_NONE || wgs <= 1920) return 8;
        return wgs > 2560 || std::any_of(ll.idx, ll.idx + n_limbs, [&](const uint8_t i) { return is_far(c->primes[i]); }) ? 16 : 8;
    }
    return wgs <= (encoding ? 640 : 900) ? 8 : 16;
}

// Passes that begin in a basis conversion or a lift, on rings below 2^16 points: four points where every CU has one workgroup at most, eight
// otherwise (six waves per SIMD).  Rotations of 2^13 / 2^14 / 2^15 points at level 6 of 42 bits with eight / four points 33.6/32.2, 36.7/35.1,
// 45.9/45.6, at level 8 of 60 bits 37.8/36.0, 46.7/44.8, 61.8/61.2; encodings of nine messages of six limbs 17.0/16.7, 23.0/22.5, 31.6/31.7 (beyond
// the line).  At 2^16 points four points go with the half slabs of narrower_slabs, eight with whole ones.
static bool few_for_conversions(const hemm_context *c, int limbs) { return (size_t)limbs * (c->N >> 12) <= 256; }

// Column passes of few workgroups are bound by the instructions of the few CUs they are on: slabs of a half or a
// quarter of the columns (1, 2: as powers of two) put them on as many more CUs.  At 2^16 points a half slab is eight columns, segments of
// 64 bytes, and pays where both halves of a line are on one XCD (Slab::slab); on two of them rotations lost 3 %, and quarters gain nothing
// more.  Transforms of 2^16 points (forward, inverse) with whole / half slabs of four points, 60 and 42 bits:
//   workgroups   64                             128                             192                             256                             384                             448                             512
//   60 bits      10.4/ 9.5 11.0/ 9.7   13.0/12.3 13.8/12.6   15.6/15.9 16.3/16.5   18.2/18.3 19.0/18.9   25.0/24.1 26.6/25.3   26.2/26.4 28.0/28.3   26.5/26.6 28.6/28.9
//   42 bits       9.0/ 8.4  9.4/ 8.5   11.3/10.7 11.9/11.1   13.6/13.7 14.2/14.3   16.0/16.1 16.6/16.6   21.9/21.3 22.7/21.9   23.5/23.8 24.5/24.7   24.6/24.9 25.7/25.7
// Conversions take half slabs further, their whole ones being bound by the three workgroups that a CU holds in step.  Rotations and products of
// 2^16 points (whole calls with their host time, an earlier build), us, with none / up to 256 / 400 / 700 / 1000 workgroups of conversions on half slabs of four points:
//   42 bits, level  4 (160 and fewer)   54.6/50.0/50.0/50.0/50.0   85.2/ 79.5/ 79.5/ 79.5/ 79.5
//                   8 (up to 256, 288)  67.8/67.8/64.3/64.0/64.1  100.3/100.3/ 96.8/ 96.6/ 95.9
//                  10 (400, 528)        80.8/80.8/80.1/76.2/76.3  117.3/117.3/114.5/110.8/111.1
//   60 bits, level 10 (384)             82.2/80.6/75.2/75.2/75.4  124.4/120.7/113.9/114.1/113.9
//                  18 (608, 784)       117.3/117.3/117.0/114.9/113.9  170.3/170.3/170.4/168.2/167.4
//                  23 (768, 960)       130.2/130.2/130.2/130.6/131.6  191.2/191.2/191.5/191.6/192.7
// In the arithmetic of primes just below 2^60, lines at 768 / 1024: 60 bits, level 16 (736) 98.6/98.8, 18 (800) 105.3/104.2, 20 (864) 113.5/111.9,
// 22 (944) 117.8/118.8, 23 (976) 120.0/120.7; 24 + 6 primes of 42 bits, level 18 (800) 109.2/106.9.
// The products of matrices, whose large conversions run beside other chains, are 1 - 3 % slower with all of them on half slabs.
// Smaller rings, transforms of 42 bits (forward, inverse) with whole slabs of sixteen points / half slabs / quarter slabs of four:
//   limbs         1                             4                             16                            32                              48                                64
//   2^13 points   7.5/6.8/6.6  7.8/6.9/6.7   7.8/7.0/6.7  8.1/7.1/6.7   8.1/7.4/7.2  8.5/7.5/7.3    8.9/ 8.3/ 7.9  9.2/ 8.5/ 8.0   10.2/ 9.8/ 9.5 10.8/10.1/ 9.7   (one launch)
//   2^14          7.6/6.9/6.6  8.0/7.2/6.7   7.9/7.1/6.8  8.2/7.3/6.8   9.2/8.2/7.9  9.6/8.4/8.0   11.6/10.5/10.4 12.3/10.9/10.8   14.5/13.2/13.1 15.2/13.9/13.5   17.5/15.7/15.7 19.3/16.3/16.4
//   (35 / 80 limbs 12.6/11.7/11.5 13.2/12.3/12.0, 20.2/18.6/18.2 22.2/19.5/18.9: the line of quarter slabs, drawn with eight points, lies below its place
//   and has not been moved)
// Transforms of 2^15 points, whole slabs of sixteen / of four points / half slabs of four:
//   limbs      1                               16                                 32                                 40                                 48                                 64
//   42 bits    7.9/7.7/7.0   8.3/8.2/7.3   11.3/11.1/10.5 11.9/11.8/11.0   16.6/16.0/15.9 17.1/16.7/16.5   19.7/19.5/18.9 20.3/20.5/19.6   22.0/21.8/21.1 22.5/22.6/22.0   25.7/25.4/25.1 26.7/26.4/26.4
//   60 bits    9.5/9.0/8.1  10.5/9.7/8.4   13.2/12.8/12.0 14.5/13.7/12.4   18.8/18.2/18.2 20.1/18.9/18.8   22.6/22.4/21.6 24.4/24.1/22.8   24.9/24.9/24.0 26.8/26.4/25.0   28.0/27.8/27.9 30.5/29.9/29.6
// (plain forward passes of 2^15 points keep whole slabs above 128 workgroups: 24 limbs of 60 bits 15.4 against 15.7; from 40 limbs on half slabs
// would lead.)
static int narrower_slabs(const hemm_context *c, int limbs, bool plain = false, bool inverse = false) {
    const size_t wgs = (size_t)limbs * (c->N >> 12);
    if (c->logN == 16) return wgs <= (plain ? 384 : 880) ? 1 : 0;
    if (c->logN == 15 && plain && !inverse && wgs > 128) return 0;
    return c->logN <= 14 && wgs <= 128 ? 2 : wgs <= 512 ? 1 : 0;
}

static void cols_pass(const hemm_context *c, bool inverse, u64 *d, const LimbList &ll, const LimbList &sl, int n_limbs,
                      int n_polys, size_t poly_stride, hipStream_t s, const void *final_scale = nullptr) {
    const bool few = few_for_columns(c, n_limbs * n_polys);
    const int narrow = narrower_slabs(c, n_limbs * n_polys, true, inverse);
    const dim3 grid((unsigned)(c->N >> (12 - narrow)), (unsigned)(n_limbs * n_polys));
    const Tw *tw = (const Tw *)(inverse ? c->d_iw : c->d_w);
#define COLS_FORM(LR, P, H, INV)                                                                                          \
    hipLaunchKernelGGL((ntt16_cols_kernel<LR, P, H, INV>), grid, dim3((4096 >> H) / P), 0, s, d, tw, c->d_modq, c->d_ninv,          \
                       c->d_ninv_s, c->d_fp, ll, sl, n_limbs, poly_stride, (const Tw *)(INV ? final_scale : nullptr))
#define COLS_SLAB(LR, INV)                          \
    do {                                            \
        if (narrow == 1) COLS_FORM(LR, 4, 1, INV);  \
        else COLS_FORM(LR, 16, 0, INV);             \
    } while (0)
#define COLS(LR)                                    \
    do {                                            \
        if (inverse) COLS_SLAB(LR, true);           \
        else COLS_SLAB(LR, false);                  \
    } while (0)
#define COLS_SMALL(LR)                                      \
    do {                                                    \
        if (narrow == 2 && inverse) COLS_FORM(LR, 4, 2, true); \
        else if (narrow == 2) COLS_FORM(LR, 4, 2, false);   \
        else COLS(LR);                                      \
    } while (0)
    switch (c->logN) {
        case 13: COLS_SMALL(5); break;
        case 14: COLS_SMALL(6); break;
        case 15:   // (inverse whole slabs are never few)
            if (few && narrow == 0 && !inverse) COLS_FORM(7, 4, 0, false);
            else COLS(7);
            break;
        default:
            if (few && narrow == 0 && inverse) COLS_FORM(8, 4, 0, true);
            else if (few && narrow == 0) COLS_FORM(8, 4, 0, false);
            else COLS(8);
    }
#undef COLS_SMALL
#undef COLS_SLAB
#undef COLS
#undef COLS_FORM
}
static void rows_pass(const hemm_context *c, bool inverse, u64 *d, const LimbList &ll, const LimbList &sl, int n_limbs,
                      int n_polys, size_t poly_stride, hipStream_t s, const NttEpilogue &ep, int tail = TAIL_NONE,
                      int load = LOAD_PLAIN, const ResultList *list = nullptr, int first = 0) {
    const int points = points_for_rows(c, ll, n_limbs, n_polys, inverse, tail);
    const dim3 grid((unsigned)(c->N >> 8) / (unsigned)points * (unsigned)(n_limbs * n_polys)), block(256);
    const int log_r = c->logN - 8;
#define ROWS(LR, P, INV, TAIL, LOAD, EP)                                                                                      \
    hipLaunchKernelGGL((ntt16_rows_kernel<LR, P, INV, TAIL, LOAD>), grid, block, 0, s, d, (const Tw *)(INV ? c->d_iw : c->d_w), \
                       (const Tw *)(INV ? c->d_irw : c->d_rw), c->d_modq, c->d_fp, ll, sl, n_limbs, poly_stride, EP, log_r)
#define ROWS_RING(P, INV, TAIL, LOAD, EP)                  \
    do {                                                   \
        if (log_r == 8) ROWS(8, P, INV, TAIL, LOAD, EP);   \
        else ROWS(0, P, INV, TAIL, LOAD, EP);              \
    } while (0)
#define ROWS_INVERSE(LOAD)                                       \
    do {                                                         \
        if (points == 4) ROWS_RING(4, true, TAIL_NONE, LOAD, ep); \
        else ROWS_RING(8, true, TAIL_NONE, LOAD, ep);            \
    } while (0)
#define ROWS_FORWARD(TAIL, EP, ROWS_16)                          \
    do {                                                         \
        if (points == 4) ROWS_RING(4, false, TAIL, LOAD_PLAIN, EP); \
        else if (points == 8) ROWS_RING(8, false, TAIL, LOAD_PLAIN, EP); \
        else ROWS_16;                                            \
    } while (0)
    if (inverse && load == LOAD_ROTATED)
        ROWS_INVERSE(LOAD_ROTATED);
    else if (inverse && load == LOAD_DECRYPT)
        ROWS_RING(4, true, TAIL_NONE, LOAD_DECRYPT, ep);   // one or two limbs
    else if (inverse)
        ROWS_INVERSE(LOAD_PLAIN);
    else if (tail == TAIL_SUB_SCALE && list != nullptr) {
        const NttEpilogueList epl{ep, (u32)first, *list};
        ROWS_FORWARD(TAIL_SUB_SCALE_LIST, epl, ROWS(0, 16, false, TAIL_SUB_SCALE_LIST, LOAD_PLAIN, epl));
    } else if (tail == TAIL_SUB_SCALE)
        ROWS_FORWARD(TAIL_SUB_SCALE, ep, ROWS(0, 16, false, TAIL_SUB_SCALE, LOAD_PLAIN, ep));   // (2^14 points and fewer)
    else if (tail == TAIL_ENCRYPT && points == 4)   // 64 limbs at most: eight points at 2^16 alone
        ROWS_RING(4, false, TAIL_ENCRYPT, LOAD_PLAIN, ep);
    else if (tail == TAIL_ENCRYPT)
        ROWS(8, 8, false, TAIL_ENCRYPT, LOAD_PLAIN, ep);
    else
        ROWS_FORWARD(TAIL_NONE, ep, ROWS_RING(16, false, TAIL_NONE, LOAD_PLAIN, ep));
#undef ROWS_FORWARD
#undef ROWS_INVERSE
#undef ROWS_RING
#undef ROWS
}
static NttEpilogue sub_scale_tail(const u64 *minuend, size_t minuend_stride, u64 *out, size_t out_stride, const void *cst) {
    NttEpilogue ep{};
    ep.minuend = minuend;
    ep.minuend_stride = minuend_stride;
    ep.out = out;
    ep.out_stride = out_stride;
    ep.cst = (const Tw *)cst;
    return ep;
}

// A transform is two launches, and the second reads what the first wrote.  On a large batch the first launch has
// pushed its early output out of the 256 MB memory-side cache by the time the second one starts, so batches are cut
// into runs of whole polynomials of about this many limbs (of 0.5 MiB each) and the two launches alternate run by run.
// Measured on 32 x 24 limbs, one stream: forward transforms are fastest at 192 limbs per run (60-bit primes 0.52 ->
// 0.43 ms, primes below 2^44 0.41 -> 0.36 ms), inverse ones at 384 (0.48 -> 0.44 ms, 0.37 -> 0.34 ms).  A plain batch
// of several runs (launch_ntt_slots) deals them out over two streams, the caller's and the context's second one:
// a launch of one run fills the part-empty last round of workgroups of the other's.  Same box, runs of 192 limbs in
// both directions: forward 0.378 -> 0.350 ms (60-bit) and 0.309 -> 0.278 ms (42-bit), inverse 0.390 -> 0.383 and
// 0.285 -> 0.278 ms; runs of 96, 128 or 256 limbs on two streams are 1 - 8 % slower than that.  Smaller rings: as many
// limbs as make the same bytes.
static int polys_per_run(const hemm_context *c, int n_limbs, int n_polys, bool inverse, bool two_streams = false) {
    const int scale = 65536 / c->N;
    // batches of up to 448 limbs (224 MiB: what one chain of the matrix products transforms at once, whose input a
    // producer has just written) are fastest as one run: 480 us for the ModDown of 64 polynomials against 497 us cut
    if ((size_t)n_limbs * n_polys <= (size_t)448 * scale) return n_polys;
    const int limbs = (inverse && !two_streams ? 384 : 192) * scale;
    int p = limbs / n_limbs;
    if (p < 1) p = 1;
    return p < n_polys ? p : n_polys;
}

// Forward transform of data[n_polys][n_limbs][N] (limb j = chain prime j) whose result is consumed as
// out = (minuend - NTT(data)) * cst[j]; returns false when this ring size has no fused tail (the caller
// then runs the transform and the subtraction separately).
bool launch_ntt_sub_scale(const hemm_context *c, u64 *data, int n_limbs, int n_polys, const u64 *minuend,
                          size_t minuend_stride, u64 *out, size_t out_stride, const void *cst_dev, hipStream_t s,
                          const ResultList *list) {
    if (!ring_has_fused_forms(c)) return false;
    if (list != nullptr && n_polys > 2 * RESULT_PARTS) throw std::invalid_argument("too many results for one list");
    const bool one = one_launch(c, (size_t)n_limbs * n_polys, false);
    account(c, TR_NTT, (size_t)3 * n_limbs * n_polys * c->N * 8, one ? 1 : 2);   // limbs in, minuend in, result out
    LimbList ll, sl;
    for (int j = 0; j < HEMM_MAX_PRIMES; j++) ll.idx[j] = sl.idx[j] = (uint8_t)j;
    const size_t poly_stride = (size_t)n_limbs * c->N;
    if (one) {
        launch_limb_forward(c, data, ll, sl, n_limbs, n_polys, poly_stride, s, nullptr, nullptr,
                            sub_scale_tail(minuend, minuend_stride, out, out_stride, cst_dev), TAIL_SUB_SCALE, list);
        return true;
    }
    const int run = polys_per_run(c, n_limbs, n_polys, false);
    for (int p0 = 0; p0 < n_polys; p0 += run) {
        const int np = n_polys - p0 < run ? n_polys - p0 : run;
        u64 *d = data + (size_t)p0 * poly_stride;
        cols_pass(c, false, d, ll, sl, n_limbs, np, poly_stride, s);
        rows_pass(c, false, d, ll, sl, n_limbs, np, poly_stride, s,
                  sub_scale_tail(minuend + (size_t)p0 * minuend_stride, minuend_stride,
                                 list != nullptr ? nullptr : out + (size_t)p0 * out_stride, out_stride, cst_dev),
                  TAIL_SUB_SCALE, LOAD_PLAIN, list, p0);
    }
    return true;
}

bool launch_ntt_converted(const hemm_context *c, const ConvSources &cs, u64 *data, const LimbList &ll, const LimbList &sl,
                          int n_limbs, int n_polys, size_t poly_stride, hipStream_t s, const u64 *ep_minuend,
                          size_t ep_minuend_stride, u64 *ep_out, size_t ep_out_stride, const void *ep_cst_dev,
                          const ResultList *ep_list, bool cols_only) {
    if (!ring_has_fused_forms(c)) return false;
    if (n_limbs > HEMM_MAX_PRIMES || cs.n_copy < 0 || cs.n_copy > HEMM_MAX_PRIMES)
        throw std::invalid_argument("too many limbs in one converted transform");
    int widest = 0;
    for (int l = 0; l < n_limbs; l++) {
        if (cs.digit_of[l] >= CONV_MAX_DIGITS) throw std::invalid_argument("conversion digit out of range");
        widest = std::max(widest, cs.d[cs.digit_of[l]].n_src);
    }
    if (widest < 1 || widest > CONV_MAX_SOURCES) return false;
    if (n_limbs <= 0 || n_polys <= 0) return true;
    if (ep_list != nullptr && n_polys > 2 * RESULT_PARTS) throw std::invalid_argument("too many results for one list");
    const bool tail = ep_out != nullptr || ep_list != nullptr;
    // sources of every digit in use once, limbs out (through the tail: minuend in, result out)
    size_t src_limbs = 0;
    bool seen[CONV_MAX_DIGITS] = {false, false, false, false};
    for (int l = 0; l < n_limbs; l++)
        if (!seen[cs.digit_of[l]]) {
            seen[cs.digit_of[l]] = true;
            src_limbs += (size_t)cs.d[cs.digit_of[l]].n_src;
        }
    if ((size_t)(n_limbs + cs.n_copy) * (size_t)n_polys > 65535)
        return false;   // more workgroup rows than one launch holds: the caller converts and transforms separately
    account(c, TR_BCONV, (src_limbs + 2 * (size_t)cs.n_copy) * n_polys * c->N * 8, 0);
    const bool one = one_launch(c, (size_t)n_limbs * n_polys, false);
    if (one && cols_only) throw std::invalid_argument("a transform in one launch has no passes");
    account(c, TR_NTT, (size_t)(tail ? 2 : 1) * n_limbs * n_polys * c->N * 8, one || cols_only ? 1 : 2);
    if (one) {
        launch_limb_forward(c, data, ll, sl, n_limbs, n_polys, poly_stride, s, &cs, nullptr,
                            sub_scale_tail(ep_minuend, ep_minuend_stride, ep_out, ep_out_stride, ep_cst_dev),
                            tail ? TAIL_SUB_SCALE : TAIL_NONE, ep_list);
        return true;
    }
    const int narrow = narrower_slabs(c, (n_limbs + cs.n_copy) * n_polys);
    const dim3 grid((unsigned)(c->N >> (12 - narrow)), (n_limbs + cs.n_copy) * n_polys);
    const bool few = few_for_conversions(c, (n_limbs + cs.n_copy) * n_polys);
#define CONV_FORM(LR, P, H, K)                                                                                               \
    hipLaunchKernelGGL((ntt16_cols_converted_kernel<LR, P, H, K>), grid, dim3((4096 >> H) / P), 0, s, data, (const Tw *)c->d_w, c->d_modq, \
                       c->d_ninv, c->d_ninv_s, c->d_fp, ll, sl, n_limbs, poly_stride, cs)
#define CONV_RING(LR, P, H)                        \
    do {                                           \
        if (widest <= 2) CONV_FORM(LR, P, H, 2);   \
        else if (widest <= 5) CONV_FORM(LR, P, H, 5); \
        else CONV_FORM(LR, P, H, 8);               \
    } while (0)
#define CONV_SLAB(LR)                          \
    do {                                       \
        if (narrow == 0) CONV_RING(LR, 8, 0);  \
        else if (few) CONV_RING(LR, 4, 1);     \
        else CONV_RING(LR, 8, 1);              \
    } while (0)
#define CONV_SMALL(LR)                         \
    do {                                       \
        if (narrow == 2) CONV_RING(LR, 4, 2);  \
        else CONV_SLAB(LR);                    \
    } while (0)
    switch (c->logN) {
        case 13: CONV_SMALL(5); break;
        case 14: CONV_SMALL(6); break;
        case 15: CONV_SLAB(7); break;
        default:   // half slabs take four points whatever the line of the smaller rings says
            if (narrow == 1) CONV_RING(8, 4, 1);
            else CONV_RING(8, 8, 0);
    }
#undef CONV_SMALL
#undef CONV_SLAB
#undef CONV_RING
#undef CONV_FORM
    if (cols_only) return true;
    rows_pass(c, false, data, ll, sl, n_limbs, n_polys, poly_stride, s,
              sub_scale_tail(ep_minuend, ep_minuend_stride, ep_out, ep_out_stride, ep_cst_dev), tail ? TAIL_SUB_SCALE : TAIL_NONE,
              LOAD_PLAIN, ep_list);
    return true;
}

static bool has_far_primes(const hemm_context *c) {
    for (const u64 q : c->primes)
        if (is_far(q)) return true;
    return false;
}
// The polynomials of a ModDown that go through its launches together: as many as have limbs that the memory-side cache holds between the
// launches, as in polys_per_run, or the whole rounds of the slab kernel (sixteen polynomials) in that where the kernel has fewer rounds then.  48 polynomials
// of 5 -> 10 limbs, cut 44 + 4 / 32 + 16: 396/359 us of 42 bits, 468/428 of 50, 429/395 of 60.
static int slab_run(int n_src, int nq_out, int n_polys) {
    const int fit = std::max(1, 448 / std::max(n_src, nq_out)), whole = fit - fit % 16;
    auto rounds = [&](int run) { return n_polys / run * ((run + 15) / 16) + (n_polys % run + 15) / 16; };
    if (n_polys <= fit) return n_polys;
    return whole != 0 && rounds(whole) < rounds(fit) ? whole : fit;
}
// The slab kernel saves two trips of every source limb and a launch, and keeps few workgroups, 32 per polynomial of which 512 are
// resident, busy for as long as there are targets: it leads by 2 - 10 % where its last round of sixteen polynomials is full, three quarters full or half
// full (a workgroup on every CU), and loses where that round has few more than none or than half.  Whole ModDowns in four launches / with it, us, one build
// with the line moved (sources -> targets; 42 bits in the chain; 50; 60):
//   polynomials            8              10              12              18              20              24              40              64             100
//   2->5  42 bits   41.1/ 38.8      47.8/ 46.7      52.4/ 48.8      70.6/ 64.9      76.0/ 68.4      84.3/ 75.5       127/119         211/201         334/330
//   3->6  42 bits   49.3/ 45.9      58.4/ 57.1      67.4/ 61.8      85.3/ 83.3      90.7/ 86.9       104/ 95         169/156         281/266         450/417
//         50 bits   60.3/ 59.9      71.0/ 74.2      83.8/ 79.3       105/105         114/111         129/120         207/196         330/320         520/501
//   4->7  42 bits   58.3/ 53.2      68.3/ 67.1      74.9/ 72.1       100/102         108/107         128/121         213/203         371/355         580/540
//         50 bits   69.9/ 67.8      82.9/ 85.7      91.9/ 92.3       124/133         133/138         156/152         255/248         417/407         648/637
//   5->8  42 bits   66.8/ 61.9      77.2/ 79.7      86.1/ 85.2       120/120         129/126         156/145         266/255         444/415         743/649
//         50 bits   80.7/ 80.0      94.6/101        106/108          143/154         157/161         185/181         309/302         493/488         804/753
//         60 bits   73.8/ 71.9      85.3/ 87.5      95.7/ 94.2       132/137         143/143         171/165         286/279         469/449         778/693
// and with more targets:
//   polynomials           13              14              16              20              28              32              48              64             128
//   2->12 50 bits    116/114         122/118         135/128
//   3->12 50 bits    125/125         133/130         145/140
//   4->12 50 bits    133/134         140/138         156/152
//   5->9  42 bits    100/ 95         104/ 98         118/105         144/138         198/193         231/221         358/336         482/446        1029/888
//   5->12 42 bits    118/112         123/116         139/127         174/175         246/245         287/280         439/410         599/549        1243/1103
//         50 bits    144/144         150/148         168/159         209/219         295/297         333/327         494/492         663/644        1354/1292
//         60 bits    129/126         136/131         153/143         190/196         270/272         306/299         465/454         628/598        1295/1196
//   polynomials           26              28              34              36              50              68
//   4->7  60 bits    151/150         162/159         197/201         209/210         295/300         398/415
//         50 bits    165/169         177/175         214/218         227/227         318/323         429/450
//   5->8  42 bits    164/165         177/175         218/218         234/231         332/332         468/448
//         60 bits    182/186         195/196         237/242         252/252         353/356         492/489
//         50 bits    196/206         212/216         256/265         272/275         378/384         518/528
// The line lies where nothing in these tables loses more than 3 %, but for 68 polynomials, which are cut 64 + 4 either way (calls of one process differ by as
// much from another's where neither form leads clearly, at 26 and 34 polynomials for instance).  uncut: never in runs.
bool takes_moddown_slab(const hemm_context *c, int n_src, int nq_out, int n_polys, bool uncut) {
    if (c->logN != 16 || n_src < 2 || n_src > SLAB_MAX_SOURCES || n_polys < 8) return false;
    const bool far = has_far_primes(c);
    const int run = uncut ? n_polys : slab_run(n_src, nq_out, n_polys), last = n_polys % 16;   // polynomials of the last round, 0: a full one
    if (nq_out <= n_src + 3) {
        if (n_src == 2) return n_polys != 9;
        if (n_src == 3) return n_polys == 8 || n_polys >= 12 || !far;
        if (last == 0 || last == 8 || last >= 13 || n_polys > 96 || (run == n_polys && n_polys >= 48)) return true;
        return !far && (n_polys == 12 || n_polys >= 20 || (n_src == 4 && n_polys <= 11 && n_polys >= 10));
    }
    if (nq_out > 12) return false;
    if (n_polys <= 16) return n_polys >= 13;
    if (n_src != 5 || n_polys < 28) return false;
    if (far) return last == 0 || last >= 14 || (run == n_polys && (last == 8 || (last >= 12 && n_polys > 32)));
    const int rest = (n_polys - 1) % run + 1;   // the last of the runs
    return rest % 16 == 0 || rest % 16 >= 12 || (rest > 16 && rest % 16 == 8);
}

bool launch_moddown_slab(const hemm_context *c, u64 *y, size_t y_stride, const uint8_t *src_slot, const uint8_t *src_prime,
                         int n_src, const void *final_scale_dev, const void *hat_dev, int hat_ld, u64 *conv, int nq_out,
                         int n_polys, u64 *out, size_t out_stride, const void *cst_dev, hipStream_t s, const ResultList *list,
                         bool rows_done, bool cols_only) {
    if (c->logN != 16 || n_src < 2 || n_src > SLAB_MAX_SOURCES || nq_out < 1 || nq_out > c->nQ || n_polys > 65535) return false;
    if (n_polys <= 0) return true;
    if (list != nullptr && n_polys > 2 * RESULT_PARTS) throw std::invalid_argument("too many results for one list");
    SlabSources ss;
    memset(&ss, 0, sizeof(ss));
    LimbList sp, ssl, ident;
    memset(&sp, 0, sizeof(sp));
    memset(&ssl, 0, sizeof(ssl));
    for (int j = 0; j < HEMM_MAX_PRIMES; j++) ident.idx[j] = (uint8_t)j;
    for (int i = 0; i < n_src; i++) {
        ss.src_slot[i] = ssl.idx[i] = src_slot[i];
        ss.src_prime[i] = sp.idx[i] = src_prime[i];
    }
    ss.src_poly_stride = y_stride;
    ss.hat = (const Cst *)hat_dev;
    ss.final_scale = (const Tw *)final_scale_dev;
    ss.hat_ld = hat_ld;
    ss.n_dst = nq_out;
    // same algorithmic bytes as the separate launches: the dropped limbs in and out of the inverse transform, the
    // conversion's sources, the minuend in and the result out of the forward transform
    account(c, TR_NTT, (size_t)2 * n_src * n_polys * c->N * 8, rows_done ? 1 : 2);
    account(c, TR_BCONV, (size_t)n_src * n_polys * c->N * 8, 0);
    account(c, TR_NTT, (size_t)(cols_only ? 1 : 2) * nq_out * n_polys * c->N * 8, cols_only ? 0 : 1);
    const size_t conv_stride = (size_t)nq_out << 16;
    const int run = rows_done && cols_only ? n_polys : slab_run(n_src, nq_out, n_polys);
    for (int p0 = 0; p0 < n_polys; p0 += run) {
        const int np = std::min(run, n_polys - p0);
        u64 *yp = y + (size_t)p0 * y_stride, *cp = conv + (size_t)p0 * conv_stride;
        ss.src = yp;
        if (!rows_done) rows_pass(c, true, yp, sp, ssl, n_src, np, y_stride, s, NttEpilogue{});
        const dim3 grid(32, (unsigned)np), block(512);
#define SLAB_CASE(NS)                                                                                                         \
    hipLaunchKernelGGL((ntt16_slab_convert_kernel<NS>), grid, block, 0, s, cp, conv_stride, (const Tw *)c->d_w,      \
                       (const Tw *)c->d_iw, c->d_modq, c->d_ninv, c->d_ninv_s, c->d_fp, ss)
        switch (n_src) {
            case 2: SLAB_CASE(2); break;
            case 3: SLAB_CASE(3); break;
            case 4: SLAB_CASE(4); break;
            default: SLAB_CASE(5);
        }
#undef SLAB_CASE
        if (cols_only) continue;
        rows_pass(c, false, cp, ident, ident, nq_out, np, conv_stride, s,
                  sub_scale_tail(yp, y_stride, list != nullptr ? nullptr : out + (size_t)p0 * out_stride, out_stride, cst_dev),
                  TAIL_SUB_SCALE, LOAD_PLAIN, list, p0);
    }
    return true;
}

bool launch_intt_from(const hemm_context *c, const u64 *src, size_t src_poly_stride, u64 *data, const LimbList &ll,
                      const LimbList &sl, int n_limbs, int n_polys, size_t poly_stride, hipStream_t s,
                      const void *final_scale, u32 galois) {
    if (!ring_has_fused_forms(c)) {
        if (galois != 0) throw std::invalid_argument("a transform reads through an automorphism at N >= 2^10 only");
        return false;
    }
    if (n_limbs <= 0 || n_polys <= 0) return true;
    // (through an automorphism: the input of a single key switch, less than the 64 limbs of the line of 2^13 points)
    const bool one = galois == 0 ? one_launch(c, (size_t)n_limbs * n_polys, true) : c->logN <= 12;
    account(c, TR_NTT, (size_t)2 * n_limbs * n_polys * c->N * 8, one ? 1 : 2);
    if (one) {
        NttEpilogue from{};
        from.minuend = src;
        from.minuend_stride = src_poly_stride;
        from.galois = galois;
        launch_limb_inverse(c, data, ll, sl, n_limbs, n_polys, poly_stride, s, final_scale, from,
                            galois != 0 ? LOAD_ROTATED : LOAD_PLAIN);
        return true;
    }
    const int run = polys_per_run(c, n_limbs, n_polys, true);
    for (int p0 = 0; p0 < n_polys; p0 += run) {
        const int np = n_polys - p0 < run ? n_polys - p0 : run;
        u64 *d = data + (size_t)p0 * poly_stride;
        NttEpilogue from{};
        from.minuend = src + (size_t)p0 * src_poly_stride;
        from.minuend_stride = src_poly_stride;
        from.galois = galois;
        rows_pass(c, true, d, ll, sl, n_limbs, np, poly_stride, s, from, TAIL_NONE, galois != 0 ? LOAD_ROTATED : LOAD_PLAIN);
        cols_pass(c, true, d, ll, sl, n_limbs, np, poly_stride, s, final_scale);
    }
    return true;
}

bool launch_ntt_lifted(const hemm_context *c, const LiftSource &ls, u64 *data, const LimbList &ll, int n_limbs, int n_polys,
                       size_t poly_stride, hipStream_t s, const EncryptTail *enc) {
    if (!ring_has_fused_forms(c)) return false;
    LimbList sl;
    for (int j = 0; j < HEMM_MAX_PRIMES; j++) sl.idx[j] = (uint8_t)j;
    // (an encryption has a limb per chain prime, 64 at most: the line of 2^13 points is reached by one chain length, without
    // special primes, which is not worth a kernel)
    const bool one = one_launch(c, (size_t)n_limbs * n_polys, false) && (enc == nullptr || c->logN <= 12);
    account(c, TR_NTT, (size_t)(n_limbs + 1) * n_polys * c->N * 8 + (enc ? (size_t)2 * n_limbs * n_polys * c->N * 8 : 0), one ? 1 : 2);
    NttEpilogue ep{};
    if (enc != nullptr) {
        ep.out = enc->b;
        ep.second_out = enc->a;
        ep.out_stride = poly_stride;
        ep.sk = enc->sk;
        ep.a_base = enc->a_base;
    }
    const int tail = enc != nullptr ? TAIL_ENCRYPT : TAIL_NONE;
    if (one) {
        launch_limb_forward(c, data, ll, sl, n_limbs, n_polys, poly_stride, s, nullptr, &ls, ep, tail);
        return true;
    }
    const int run = polys_per_run(c, n_limbs, n_polys, false);
    for (int p0 = 0; p0 < n_polys; p0 += run) {
        const int np = n_polys - p0 < run ? n_polys - p0 : run;
        u64 *d = data + (size_t)p0 * poly_stride;
        LiftSource l = ls;
        l.coef += (size_t)p0 * ls.stride;
        // (2^16 points: the loads of a lift are few and shared by the limbs of a message, so that half slabs of four points pay longer than
        // in a conversion.  Encodings of 4 x 6 / 4 x 13 / 9 x 6 / 9 x 13 limbs, us: 28.8/39.3/41.5/56.2 -> 27.7/38.7/40.4/56.5)
        const bool half = c->logN == 16 ? n_limbs * np <= 64 : narrower_slabs(c, n_limbs * np) != 0;
        const dim3 grid((unsigned)(c->N >> (half ? 11 : 12)), (unsigned)(n_limbs * np));
        const bool few = few_for_conversions(c, n_limbs * np);
#define LIFTED_FORM(LR, P, H)                                                                                                       \
    hipLaunchKernelGGL((ntt16_cols_lifted_kernel<LR, P, H>), grid, dim3((4096 >> H) / P), 0, s, d, (const Tw *)c->d_w, c->d_modq, c->d_fp, ll, sl, \
                       n_limbs, poly_stride, l)
#define LIFTED(LR)                            \
    do {                                      \
        if (!half) LIFTED_FORM(LR, 8, 0);     \
        else if (few) LIFTED_FORM(LR, 4, 1);  \
        else LIFTED_FORM(LR, 8, 1);           \
    } while (0)
        switch (c->logN) {
            case 13: LIFTED(5); break;
            case 14: LIFTED(6); break;
            case 15: LIFTED(7); break;
            default:
                if (half) LIFTED_FORM(8, 4, 1);
                else LIFTED_FORM(8, 8, 0);
        }
#undef LIFTED
#undef LIFTED_FORM
        rows_pass(c, false, d, ll, sl, n_limbs, np, poly_stride, s, ep, tail);
        if (enc != nullptr) {
            ep.out += (size_t)np * poly_stride;
            ep.second_out += (size_t)np * poly_stride;
        }
    }
    return true;
}

bool launch_intt_decrypt(const hemm_context *c, const u64 *b, const u64 *a, const u64 *sk, u64 *data, int n_limbs, hipStream_t s) {
    if (!ring_has_fused_forms(c)) return false;
    LimbList ll;
    for (int j = 0; j < HEMM_MAX_PRIMES; j++) ll.idx[j] = (uint8_t)j;
    const bool one = c->logN <= 12;   // one or two limbs
    account(c, TR_NTT, (size_t)4 * n_limbs * c->N * 8, one ? 1 : 2);
    NttEpilogue from{};
    from.minuend = b;
    from.second_in = a;
    from.sk = sk;
    const size_t poly_stride = (size_t)n_limbs * c->N;
    if (one) {
        launch_limb_inverse(c, data, ll, ll, n_limbs, 1, poly_stride, s, nullptr, from, LOAD_DECRYPT);
        return true;
    }
    rows_pass(c, true, data, ll, ll, n_limbs, 1, poly_stride, s, from, TAIL_NONE, LOAD_DECRYPT);
    cols_pass(c, true, data, ll, ll, n_limbs, 1, poly_stride, s);
    return true;
}

void launch_ntt_slots(const hemm_context *c, u64 *data, const LimbList &ll, const LimbList &sl, int n_limbs,
                      int n_polys, size_t poly_stride, bool inverse, hipStream_t s, const void *final_scale) {
    if (n_limbs <= 0 || n_polys <= 0) return;
    if (final_scale != nullptr && (!inverse || !ring_has_fused_forms(c)))
        throw std::invalid_argument("a final constant is taken by the inverse transform of N >= 2^10 only");
    const bool one = one_launch(c, (size_t)n_limbs * n_polys, true) || !ring_has_fused_forms(c);
    account(c, TR_NTT, (size_t)2 * n_limbs * n_polys * c->N * 8, one ? 1 : 2);
    if (!ring_has_fused_forms(c)) {
        const dim3 grid(1, (unsigned)(n_limbs * n_polys)), block(256);
        if (inverse)
            hipLaunchKernelGGL(ntt_small_kernel<true>, grid, block, 0, s, data, (const Tw *)c->d_iw, c->d_modq, c->d_ninv,
                               c->d_ninv_s, ll, sl, n_limbs, poly_stride, c->logN);
        else
            hipLaunchKernelGGL(ntt_small_kernel<false>, grid, block, 0, s, data, (const Tw *)c->d_w, c->d_modq, c->d_ninv,
                               c->d_ninv_s, ll, sl, n_limbs, poly_stride, c->logN);
        return;
    }
    if (one) {
        if (inverse)
            launch_limb_inverse(c, data, ll, sl, n_limbs, n_polys, poly_stride, s, final_scale, NttEpilogue{}, LOAD_PLAIN);
        else
            launch_limb_forward(c, data, ll, sl, n_limbs, n_polys, poly_stride, s, nullptr, nullptr, NttEpilogue{}, TAIL_NONE);
        return;
    }
    const int run = polys_per_run(c, n_limbs, n_polys, inverse, true);
    // several runs: the odd ones on the context's second stream, which starts after what the caller's stream holds
    // so far and is waited for before the call returns to it
    const bool two = run < n_polys;
    const hipStream_t own = s;
    if (two && c->aux == nullptr) {
        hemm_context *m = const_cast<hemm_context *>(c);
        HEMM_HIP(hipStreamCreateWithFlags(&m->aux, hipStreamNonBlocking));
        HEMM_HIP(hipEventCreateWithFlags(&m->aux_fork, hipEventDisableTiming));
        HEMM_HIP(hipEventCreateWithFlags(&m->aux_join, hipEventDisableTiming));
    }
    if (two) {
        HEMM_HIP(hipEventRecord(c->aux_fork, own));
        HEMM_HIP(hipStreamWaitEvent(c->aux, c->aux_fork, 0));
    }
    int run_index = 0;
    for (int p0 = 0; p0 < n_polys; p0 += run, run_index++) {
        const int np = n_polys - p0 < run ? n_polys - p0 : run;
        u64 *d = data + (size_t)p0 * poly_stride;
        s = two && (run_index & 1) ? c->aux : own;
        if (!inverse) {
            cols_pass(c, false, d, ll, sl, n_limbs, np, poly_stride, s);
            rows_pass(c, false, d, ll, sl, n_limbs, np, poly_stride, s, NttEpilogue{});
        } else {
            rows_pass(c, true, d, ll, sl, n_limbs, np, poly_stride, s, NttEpilogue{});
            cols_pass(c, true, d, ll, sl, n_limbs, np, poly_stride, s, final_scale);
        }
    }
    if (two) {
        HEMM_HIP(hipEventRecord(c->aux_join, c->aux));
        HEMM_HIP(hipStreamWaitEvent(own, c->aux_join, 0));
    }
}

void launch_intt_cols(const hemm_context *c, u64 *data, const LimbList &ll, const LimbList &sl, int n_limbs, int n_polys,
                      size_t poly_stride, hipStream_t s, const void *final_scale) {
    account(c, TR_NTT, (size_t)2 * n_limbs * n_polys * c->N * 8, 1);
    const int run = std::min(n_polys, 65535 / n_limbs);   // rows of workgroups of a launch
    for (int p0 = 0; p0 < n_polys; p0 += run)
        cols_pass(c, true, data + (size_t)p0 * poly_stride, ll, sl, n_limbs, std::min(run, n_polys - p0), poly_stride, s, final_scale);
}

void launch_ntt(const hemm_context *c, u64 *data, const LimbList &ll, int n_limbs, int n_polys,
                size_t poly_stride, bool inverse, hipStream_t s) {
    LimbList sl;
    for (int j = 0; j < HEMM_MAX_PRIMES; j++) sl.idx[j] = (uint8_t)j;
    launch_ntt_slots(c, data, ll, sl, n_limbs, n_polys, poly_stride, inverse, s);
}
