// Transforms in one launch, a workgroup per limb: rings of 2^10 .. 2^12 points, and batches of many limbs of 2^13 and 2^14.
//
// Such a limb (8 .. 128 KiB) fits the LDS of one CU, so the column pass and the row pass of the R x 256 view
// (R = N / 256) meet in LDS instead of in memory, and a transform that the two-launch kernels would take as two dependent
// launches is one.  What bounds a call on the small rings is the number of dependent launches, a few microseconds each
// however little they do, not arithmetic or bytes: one transform of 2^12 points 7 us against 36 us with the butterflies
// of every stage read from and written to LDS one by one, which these kernels replace.  A thread holds four or eight residues (16 at 2^14 points, where
// eight would take 2048 threads; with eight a CU has two wavefronts per SIMD on a limb of 2^12 points instead of one: product
// of two encrypted 32 x 32 tiles 687 -> 595 us): the log2 R
// column stages in one block (R <= 16) or two, one exchange through LDS after each, then the row pass of the two-launch
// kernels (two radix-16 blocks).  The first stages can read their input from a
// basis conversion, the last ones can end in (minuend - v) * constant, and an inverse transform can read its input
// elsewhere and through an automorphism, as in the two-launch kernels: same arithmetic, same residues.
#include <algorithm>
#include <cstring>

#include "ntt_device.h"

namespace {

template <int LR, int P>
struct Limb {
    typedef Lanes<P> L;
    static constexpr int R = 1 << LR, NT = 16 << LR;   // rows, threads
    static constexpr int Q = LR > 4 ? R / 16 : 1;      // LR > 4: two column blocks, of four stages and of LR - 4
    static constexpr int T1 = LR > 4 ? 4 : LR, T2 = LR - T1;
    // R <= 16: element k of a thread is row k % R of column threadIdx.x + NT * (k / R); otherwise row rh + Q k of column
    // threadIdx.x % 256 in the first block and row 16 rh + k in the second, rh = threadIdx.x / 256
    static __device__ __forceinline__ u32 t() { return L::t(); }
    static __device__ __forceinline__ int rh() { return LR > 4 ? (int)(t() >> 8) : 0; }
    // row and column of point e of the first block
    static __device__ __forceinline__ int row(const int e) { return LR > 4 ? rh() + Q * e : e & (R - 1); }
    static __device__ __forceinline__ int col(const int e) { return LR > 4 ? (int)(t() & 255) : (int)t() + NT * (e / R); }
    // byte offset inside the limb of the first block's points (split): a thread's part and the step to register k
    static __device__ __forceinline__ constexpr u32 step(const u32 e) {
        return LR > 4 ? e * (u32)(Q * 2048) : (e & (R - 1)) * 2048u + (e / R) * (u32)(NT * 8);
    }
    static __device__ __forceinline__ u32 voff() {
        return ((LR > 4 ? t() & 255 : t()) + ((u32)rh() << 8)) * 8u + step(L::template h_split<T1>());
    }
    static __device__ __forceinline__ constexpr u32 off(const int k) { return step((u32)L::template split<T1>(k)); }
    // places in LDS of register k: of the first block (split, whole) and of the second, which has less than four stages
    static __device__ __forceinline__ int place(const int e) { return row(e) * ROWPAD + padc(col(e)); }
    static __device__ __forceinline__ int at_s(const int k) { return place((int)L::template h_split<T1>() + L::template split<T1>(k)); }
    static __device__ __forceinline__ int at_w(const int k) { return place((int)L::h_whole() + k); }
    static __device__ __forceinline__ int at2(const int k) { return (16 * rh() + (int)L::h_whole() + k) * ROWPAD + padc(col(0)); }
};

// NS > 0: the input is a conversion of up to NS sources, LIFTED: the coefficients of an encoding
enum { LIFTED = -1 };
template <int LR, int P, int NS, int TAIL, class F>
__device__ __forceinline__ void limb_forward(u64 *__restrict__ limb, const Tw *__restrict__ tw_int, const Tw *__restrict__ rtw,
                                             const F f, u64 *lds_raw, const __amdgpu_buffer_rsrc_t src,
                                             const u32 (&so)[NS > 0 ? NS : 1], const DotCst (&h)[NS > 0 ? NS : 1], const int n_src,
                                             const ModQ m, const LiftSource &ls, const long long *__restrict__ coef,
                                             const u64 *__restrict__ mn, u64 *__restrict__ o, const Tw cst, RowSecond sec) {
    typedef typename F::E E;
    typedef Limb<LR, P> S;
    E *lds = (E *)lds_raw;
    E x[P];
    if constexpr (NS > 0) {
        converted_inputs<NS>(f, x, src, S::voff(), so, h, n_src, m,
                             [](const int k) { return S::off(k); });
    } else if (NS == LIFTED) {
        lifted_inputs(f, x, ls, coef, m, [](const int k) { return (S::voff() + S::off(k)) >> 3; });
    } else {
#pragma unroll
        for (int k = 0; k < P; k++) x[k] = f.from_canonical(buf_load<u64>(src, S::voff(), S::off(k)));
    }
    radix_fwd<S::T1, true>(f, x, (const typename F::W *)tw_int, 1u);
#pragma unroll
    for (int k = 0; k < P; k++) lds[S::at_w(k)] = x[k];
    __syncthreads();
    if (S::T2 > 0) {
#pragma unroll
        for (int k = 0; k < P; k++) x[k] = lds[S::at2(k)];
        radix_fwd<S::T2>(f, x, (const typename F::W *)tw_int, 16u + (u32)S::rh() * (16 / S::Q));
#pragma unroll
        for (int k = 0; k < P; k++) lds[S::at2(k)] = x[k];   // the places this thread has just read
        __syncthreads();
    }
    const u32 r = Lanes<P>::t() >> 4;
    if (TAIL == TAIL_ENCRYPT) {
        sec.out += r << 8;
        sec.sk += r << 8;
    }
    rows_body<P, false, TAIL, LOAD_PLAIN, true>(limb + (r << 8), tw_int, rtw, f, lds_raw, LR, r,
                                             TAIL == TAIL_SUB_SCALE ? mn + (r << 8) : nullptr,
                                             TAIL != TAIL_NONE ? o + (r << 8) : nullptr, cst, nullptr, 0, sec);
}

// data[n_polys][.][N] (polynomial stride poly_stride), limb l in slot sl[l]; the plain copies of cs follow the limbs of a
// polynomial.
template <int LR, int P, int NS, int KTAIL>
__global__ __launch_bounds__((256 / P) << LR) void ntt_limb_forward_kernel(
    u64 *__restrict__ data, const Tw *__restrict__ tw_all, const Tw *__restrict__ rtw_all, const ModQ *__restrict__ modq,
    const double *__restrict__ fp, LimbList ll, LimbList sl, int n_limbs, size_t poly_stride, ConvSources cs,
    LiftSource ls, typename EpilogueOf<KTAIL>::T ep) {
    constexpr int TAIL = tail_of(KTAIL);
    __shared__ u64 lds[(ROWPAD << LR)];
    const int log_n = 8 + LR;
    const int per_poly = n_limbs + (NS > 0 ? cs.n_copy : 0);
    const int limb = blockIdx.x % per_poly, poly = blockIdx.x / per_poly;
    if (NS > 0 && limb >= n_limbs) {   // a limb that is only copied into its slot
        const u64 *from = cs.copy_src + (size_t)poly * cs.copy_src_stride + ((size_t)table_byte(cs.copy_src_slot, limb - n_limbs) << log_n);
        u64 *to = data + (size_t)poly * poly_stride + ((size_t)table_byte(cs.copy_dst_slot, limb - n_limbs) << log_n);
        u64 t[P];
#pragma unroll
        for (int k = 0; k < P; k++) {
            const u32 n = threadIdx.x + (u32)k * (u32)((256 / P) << LR);
            t[k] = from[cs.copy_galois != 0 ? galois_index(n, cs.copy_galois, log_n) : n];
        }
#pragma unroll
        for (int k = 0; k < P; k++) to[threadIdx.x + (u32)k * (u32)((256 / P) << LR)] = t[k];
        return;
    }
    const int prime = (int)table_byte(ll.idx, limb);
    u64 *base = data + (size_t)poly * poly_stride + ((size_t)table_byte(sl.idx, limb) << log_n);
    const Tw *tw = tw_all + ((size_t)prime << log_n), *rtw = rtw_all + ((size_t)prime << log_n);
    const ModQ m = modq[prime];
    __amdgpu_buffer_rsrc_t src = limb_rsrc(base);
    u32 so[NS > 0 ? NS : 1];
    DotCst h[NS > 0 ? NS : 1];
    int n_src = 0;
    if (NS > 0) {
        const int dg = (int)table_byte(cs.digit_of, limb);
        n_src = cs.d[dg].n_src;
        src = limb_rsrc(cs.d[dg].src + (size_t)poly * cs.d[dg].src_poly_stride);
        const Cst *hat = cs.d[dg].hat + prime;
#pragma unroll
        for (int i = 0; i < NS; i++) {
            const int ii = i < n_src ? i : 0;
            so[i] = table_byte(cs.d[dg].src_slot, ii) << (log_n + 3);
            const Cst hg = hat[(size_t)ii * cs.hat_ld];
            h[i] = dot_cst(hg.w, hg.ws);
        }
    }
    const u64 *mn = nullptr;
    u64 *o = nullptr;
    Tw cst{0, 0};
    RowSecond sec{};
    if (TAIL != TAIL_NONE) o = ep.result(poly) + ((size_t)limb << log_n);
    if (TAIL == TAIL_SUB_SCALE) {
        mn = ep.minuend + (size_t)poly * ep.minuend_stride + ((size_t)limb << log_n);
        cst = ep.cst[limb];
    } else if (TAIL == TAIL_ENCRYPT) {
        sec.out = ep.second_out + (size_t)poly * ep.out_stride + ((size_t)limb << log_n);
        sec.sk = ep.sk + ((size_t)prime << log_n);
        sec.key = sm64(sm64(ep.a_base + (u64)prime));
        sec.m = m;
    }
    const long long *coef = NS == LIFTED ? ls.coef + (size_t)poly * ls.stride : nullptr;
    if (fp[4 * prime] != 0.0)
        limb_forward<LR, P, NS, TAIL>(base, tw, rtw, FpField(modq, nullptr, nullptr, fp, prime), lds, src, so, h, n_src, m, ls,
                                   coef, mn, o, cst, sec);
    else {
        const auto transform = [&](const auto f) {
            limb_forward<LR, P, NS, TAIL>(base, tw, rtw, f, lds, src, so, h, n_src, m, ls, coef, mn, o, cst, sec);
        };
        if constexpr (NS <= 0)
            with_int_field(modq, nullptr, nullptr, fp, prime, transform);
        else   // (the sums of a conversion take primes below 2^60)
            with_field_60(modq, nullptr, nullptr, fp, prime, transform);
    }
}

template <int LR, int P, int LOAD, class F>
__device__ __forceinline__ void limb_inverse(u64 *__restrict__ limb, const Tw *__restrict__ tw_int, const Tw *__restrict__ rtw,
                                             const F f, u64 *lds_raw, const u64 *__restrict__ ld, const u32 gal, RowSecond sec) {
    typedef typename F::E E;
    typedef Limb<LR, P> S;
    E *lds = (E *)lds_raw;
    const u32 r = Lanes<P>::t() >> 4;
    if (LOAD == LOAD_DECRYPT) {
        sec.in += r << 8;
        sec.sk += r << 8;
    }
    rows_body<P, true, TAIL_NONE, LOAD, true>(limb, tw_int, rtw, f, lds_raw, LR, r, nullptr, nullptr, Tw{0, 0},
                                           LOAD == LOAD_ROTATED ? ld : ld + (r << 8), gal, sec);
    __syncthreads();
    E x[P];
#pragma unroll
    for (int k = 0; k < P; k++) x[k] = lds[S::T2 > 0 ? S::at2(k) : S::at_w(k)];
    if (S::T2 > 0) {
        radix_inv<S::T2>(f, x, (const typename F::W *)tw_int, 16u + (u32)S::rh() * (16 / S::Q));
        f.template after_inverse_block<S::T2>(x);
#pragma unroll
        for (int k = 0; k < P; k++) lds[S::at2(k)] = x[k];   // the places this thread has just read
        __syncthreads();
#pragma unroll
        for (int k = 0; k < P; k++) x[k] = lds[S::at_w(k)];
    }
    radix_inv<S::T1, true>(f, x, (const typename F::W *)tw_int, 1u);
    const __amdgpu_buffer_rsrc_t to = limb_rsrc(limb);
#pragma unroll
    for (int k = 0; k < P; k++) buf_store<u64>(to, S::voff(), S::off(k), f.scale_to_canonical(x[k]));
}

template <int LR, int P, int LOAD>
__global__ __launch_bounds__((256 / P) << LR) void ntt_limb_inverse_kernel(
    u64 *__restrict__ data, const Tw *__restrict__ tw_all, const Tw *__restrict__ rtw_all, const ModQ *__restrict__ modq,
    const u64 *__restrict__ ninv, const u64 *__restrict__ ninv_s, const double *__restrict__ fp, LimbList ll, LimbList sl,
    int n_limbs, size_t poly_stride, const Tw *__restrict__ final_scale, NttEpilogue from) {
    __shared__ u64 lds[(ROWPAD << LR)];
    const int log_n = 8 + LR;
    const int limb = blockIdx.x % n_limbs, poly = blockIdx.x / n_limbs;
    const int prime = (int)table_byte(ll.idx, limb);
    const size_t slot = (size_t)table_byte(sl.idx, limb) << log_n;
    u64 *base = data + (size_t)poly * poly_stride + slot;
    const u64 *ld = from.minuend != nullptr ? from.minuend + (size_t)poly * from.minuend_stride + slot : base;
    RowSecond sec{};
    if (LOAD == LOAD_DECRYPT) {
        sec.in = from.second_in + (size_t)poly * from.minuend_stride + slot;
        sec.sk = from.sk + ((size_t)prime << log_n);
        sec.m = modq[prime];
    }
    const Tw *tw = tw_all + ((size_t)prime << log_n), *rtw = rtw_all + ((size_t)prime << log_n);
    if (fp[4 * prime] != 0.0) {
        FpField f(modq, ninv, ninv_s, fp, prime);
        if (final_scale != nullptr) f.set_scale(final_scale[limb]);
        limb_inverse<LR, P, LOAD>(base, tw, rtw, f, lds, ld, from.galois, sec);
    } else {
        with_int_field(modq, ninv, ninv_s, fp, prime, [&](auto f) {
            if (final_scale != nullptr) f.set_scale(final_scale[limb]);
            limb_inverse<LR, P, LOAD>(base, tw, rtw, f, lds, ld, from.galois, sec);
        });
    }
}

// points per thread: of 2^12 points four where every CU has one limb at most (sixteen wavefronts on it), eight in larger launches, whose second
// twiddle and address cost more than that.  Transforms, us of device time with eight / four: 64 limbs of 60 bits 7.2/6.9, 256 8.6/8.3, 264 11.6/11.9,
// 1024 22.4/23.8, 4096 79.4/82.7; of 42 bits 5.5/5.6, 6.7/6.7, 8.7/9.2, 16.3/18.2, 56.5/61.1; rotations 42.2/41.1 (42 bits), 47.7/46.6 (60)
#define POINTS(LR) ((LR) <= 5 ? 8 : 16)
#define POINTS_FEW(LR) ((LR) == 4 ? 4 : POINTS(LR))
static bool few_limbs(const size_t limbs) { return limbs <= 256; }
}  // namespace

void launch_limb_forward(const hemm_context *c, u64 *data, const LimbList &ll, const LimbList &sl, int n_limbs, int n_polys,
                         size_t poly_stride, hipStream_t s, const ConvSources *cs, const LiftSource *ls, const NttEpilogue &ep,
                         int tail, const ResultList *list) {
    const int LR = c->logN - 8;
    int widest = 0;
    ConvSources conv;
    LiftSource lift{};
    memset(&conv, 0, sizeof(conv));
    if (cs != nullptr) {
        conv = *cs;
        for (int l = 0; l < n_limbs; l++) widest = std::max(widest, cs->d[cs->digit_of[l]].n_src);
    }
    if (ls != nullptr) lift = *ls;
    NttEpilogueList epl{ep, 0, {}};
    if (list != nullptr) epl.list = *list;
    const dim3 grid((unsigned)((n_limbs + conv.n_copy) * n_polys));
    const bool few = few_limbs(grid.x);
#define LIMB_FORWARD_POINTS(L, P, K, TAIL, EP)                                                                             \
    hipLaunchKernelGGL((ntt_limb_forward_kernel<L, P, K, TAIL>), grid, dim3((256 / (P)) << (L)), 0, s, data, (const Tw *)c->d_w,       \
                       (const Tw *)c->d_rw, c->d_modq, c->d_fp, ll, sl, n_limbs, poly_stride, conv, lift, EP)
#define LIMB_FORWARD(L, K, TAIL, EP)                                       \
    do {                                                                   \
        if (few) LIMB_FORWARD_POINTS(L, POINTS_FEW(L), K, TAIL, EP);       \
        else LIMB_FORWARD_POINTS(L, POINTS(L), K, TAIL, EP);               \
    } while (0)
#define LIMB_SOURCES(L, TAIL, EP)                          \
    do {                                                   \
        if (widest == 0) LIMB_FORWARD(L, 0, TAIL, EP);     \
        else if (widest <= 2) LIMB_FORWARD(L, 2, TAIL, EP); \
        else if (widest <= 5) LIMB_FORWARD(L, 5, TAIL, EP); \
        else LIMB_FORWARD(L, 8, TAIL, EP);                 \
    } while (0)
#define LIMB_RING(L)                                                       \
    do {                                                                   \
        if (ls != nullptr && tail == TAIL_ENCRYPT) LIMB_FORWARD_POINTS(L, POINTS_FEW(L), LIFTED, TAIL_ENCRYPT, ep); /* one message */ \
        else if (ls != nullptr) LIMB_FORWARD(L, LIFTED, TAIL_NONE, ep);    \
        else if (tail == TAIL_SUB_SCALE && list != nullptr) LIMB_SOURCES(L, TAIL_SUB_SCALE_LIST, epl); \
        else if (tail == TAIL_SUB_SCALE) LIMB_SOURCES(L, TAIL_SUB_SCALE, ep);  \
        else LIMB_SOURCES(L, TAIL_NONE, ep);                               \
    } while (0)
    switch (LR) {
        case 2: LIMB_RING(2); break;
        case 3: LIMB_RING(3); break;
        case 4: LIMB_RING(4); break;
        case 5:
            if (tail == TAIL_ENCRYPT) throw std::invalid_argument("no one-launch encryption for this ring size");
            if (ls != nullptr) LIMB_FORWARD(5, LIFTED, TAIL_NONE, ep);
            else if (tail == TAIL_SUB_SCALE && list != nullptr) LIMB_SOURCES(5, TAIL_SUB_SCALE_LIST, epl);
            else if (tail == TAIL_SUB_SCALE) LIMB_SOURCES(5, TAIL_SUB_SCALE, ep);
            else LIMB_SOURCES(5, TAIL_NONE, ep);
            break;
        case 6: LIMB_FORWARD(6, 0, TAIL_NONE, ep); break;
        default: throw std::invalid_argument("no one-launch transform for this ring size");
    }
#undef LIMB_RING
#undef LIMB_SOURCES
#undef LIMB_FORWARD
#undef LIMB_FORWARD_POINTS
}

void launch_limb_inverse(const hemm_context *c, u64 *data, const LimbList &ll, const LimbList &sl, int n_limbs, int n_polys,
                         size_t poly_stride, hipStream_t s, const void *final_scale, const NttEpilogue &from, int load) {
    const int LR = c->logN - 8;
    const dim3 grid((unsigned)(n_limbs * n_polys));
    const bool few = few_limbs(grid.x);
#define LIMB_INVERSE(L, LOAD)                                              \
    do {                                                                   \
        if (few) LIMB_INVERSE_POINTS(L, POINTS_FEW(L), LOAD);              \
        else LIMB_INVERSE_POINTS(L, POINTS(L), LOAD);                      \
    } while (0)
#define LIMB_INVERSE_POINTS(L, P, LOAD)                                                                               \
    hipLaunchKernelGGL((ntt_limb_inverse_kernel<L, P, LOAD>), grid, dim3((256 / (P)) << (L)), 0, s, data, (const Tw *)c->d_iw,              \
                       (const Tw *)c->d_irw, c->d_modq, c->d_ninv, c->d_ninv_s, c->d_fp, ll, sl, n_limbs, poly_stride, \
                       (const Tw *)final_scale, from)
#define LIMB_RING(L)                                                   \
    do {                                                               \
        if (load == LOAD_ROTATED) LIMB_INVERSE(L, LOAD_ROTATED);       \
        else if (load == LOAD_DECRYPT) LIMB_INVERSE_POINTS(L, POINTS_FEW(L), LOAD_DECRYPT); /* one or two limbs */ \
        else LIMB_INVERSE(L, LOAD_PLAIN);                              \
    } while (0)
    switch (LR) {
        case 2: LIMB_RING(2); break;
        case 3: LIMB_RING(3); break;
        case 4: LIMB_RING(4); break;
        case 5:
            if (load != LOAD_PLAIN) throw std::invalid_argument("no such one-launch transform for this ring size");
            LIMB_INVERSE(5, LOAD_PLAIN);
            break;
        case 6: LIMB_INVERSE(6, LOAD_PLAIN); break;
        default: throw std::invalid_argument("no one-launch transform for this ring size");
    }
#undef LIMB_RING
#undef LIMB_INVERSE
#undef LIMB_INVERSE_POINTS
}
