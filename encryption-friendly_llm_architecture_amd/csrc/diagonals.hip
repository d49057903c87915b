// A plaintext matrix applied to every row of an encrypted one as a sum over its diagonals, in baby and giant steps:
//   A B = sum_r rho^r(A) (.) P_r = sum_t rho^(g t)( sum_j rho^j(A) (.) Q_tj ),   Q_tj = rho^(-g t)(P_(g t + j)).
// P_r, 1 - k <= r < k, holds B[c + r][c] in column c of every row of a k x k tile (rows of w slots: w / k tiles side by side), zero
// where c + r lies outside: the same w values in every row.  Such a plaintext is a polynomial in X^(N / 2w), and its transform is constant
// over runs of N / 2w residues: 2w values per limb instead of N.  The two steps that are not key switches are here: the tables
// of all Q_tj, made once per weight, and the inner sums, from rotations that stay in the extended basis.
#include <cstring>

#include "hoisted.h"
#include "ntt_device.h"

#define DIAG_OUT 8        // inner sums of one workgroup
#define DIAG_MAX_W 512

namespace {
__device__ __forceinline__ long long rounded(const double x) { return (long long)__builtin_round(x); }

// The table entry of (limb e, run, t, j): the residue h and 2^30 h as a lazy dot product takes them (DotCst).  Outputs come in chunks of
// DIAG_OUT, the terms of a chunk back to back: [E][2w][chunks][g][DIAG_OUT].
template <class F>
__device__ __forceinline__ void transform_runs(const F f, u64 *buf, const Tw *__restrict__ tw_int, const u32 w, const int log2w) {
    typedef typename F::E E;
    const typename F::W *tw = (const typename F::W *)tw_int;
    E *x = (E *)buf;
    for (u32 i = threadIdx.x; i < 2 * w; i += 256) x[i] = f.from_canonical(buf[i]);
    __syncthreads();
    // the first stages of the transform of N points: the later ones find zeros at a distance and change nothing
    for (int s = 0; s < log2w; s++) {
        const u32 t = 2 * w >> (s + 1);
        for (u32 b = threadIdx.x; b < w; b += 256) {
            const u32 i = (b / t) * 2 * t + (b & (t - 1));
            f.ct(x[i], x[i + t], tw[(1u << s) + b / t], (s & 1) != 0);
        }
        __syncthreads();
    }
    for (u32 i = threadIdx.x; i < 2 * w; i += 256) buf[i] = f.to_canonical(x[i]);
    __syncthreads();
}
// One workgroup per (t, j) and limb.  The embedding of w points is the tail of the one of N / 2: before it every butterfly adds a value to
// itself or subtracts it from itself, both exactly.
__global__ __launch_bounds__(256) void diagonal_tables_kernel(const double2 *__restrict__ block, const double2 *__restrict__ roots,
                                                              const Tw *__restrict__ tw_all, const ModQ *__restrict__ modq,
                                                              const double *__restrict__ fp, const Cst *__restrict__ pmod, LimbList ll,
                                                              const int nq, const int logN, const u32 k, const u32 log_w, const u32 g,
                                                              const u32 giants, const u32 chunks, const double scale,
                                                              uint4 *__restrict__ tables) {
#pragma clang fp contract(off)
    __shared__ double2 z[DIAG_MAX_W];
    __shared__ u64 buf[2 * DIAG_MAX_W];
    const u32 w = 1u << log_w, t = blockIdx.x / g, j = blockIdx.x % g, e = blockIdx.y;
    const int amount = t < giants / 2 ? (int)(t * g) : ((int)t - (int)giants) * (int)g, r = amount + (int)j;
    const double inv_n = 1.0 / (double)(1u << (logN - 1));
    for (u32 c = threadIdx.x; c < w; c += 256) {
        const u32 from = (c - (u32)amount) & (w - 1);
        const int row = (int)(from & (k - 1)) + r;
        double2 v = make_double2(0.0, 0.0);
        if (t < giants && row >= 0 && row < (int)k) v = block[((size_t)row << log_w) + from];
        const double times = (double)(1u << (logN - 1 - (int)log_w));
        z[c] = make_double2(v.x * times, v.y * times);
    }
    __syncthreads();
    for (u32 h = w / 2; h >= 1; h >>= 1) {
        for (u32 b = threadIdx.x; b < w / 2; b += 256) {
            const u32 q = b & (h - 1), i = (b / h) * 2 * h + q;
            const double2 a = z[i], d = z[i + h], root = roots[h + q];
            const double2 s = make_double2(a.x - d.x, a.y - d.y);
            z[i] = make_double2(a.x + d.x, a.y + d.y);
            z[i + h] = make_double2(s.x * root.x - s.y * root.y, s.x * root.y + s.y * root.x);
        }
        __syncthreads();
    }
    const int prime = (int)table_byte(ll.idx, e);
    const ModQ m = modq[prime];
    for (u32 p = threadIdx.x; p < w; p += 256) {
        const u32 c = __brev(p) >> (32 - log_w);
        buf[c] = lift_residue(rounded(z[p].x * inv_n * scale), m);
        buf[w + c] = lift_residue(rounded(z[p].y * inv_n * scale), m);
    }
    __syncthreads();
    const Tw *tw = tw_all + ((size_t)prime << logN);
    if (fp[4 * prime] != 0.0)
        transform_runs(FpField(modq, nullptr, nullptr, fp, prime), buf, tw, w, (int)log_w + 1);
    else
        with_field_60(modq, nullptr, nullptr, fp, prime, [&](const auto f) { transform_runs(f, buf, tw, w, (int)log_w + 1); });
    // the rotation by nothing enters as P times the ciphertext, on the chain limbs: its diagonals carry the factor
    const bool own = j == 0, none = own && (int)e >= nq;
    for (u32 run = threadIdx.x; run < 2 * w; run += 256) {
        u64 h = none ? 0 : buf[run];
        if (own && !none) h = mulmod(h, pmod[e].w, m);
        const DotCst d = dot_cst(h, mulmod(h, (u64)1 << 30, m));
        tables[((((size_t)e * 2 * w + run) * chunks + t / DIAG_OUT) * g + j) * DIAG_OUT + t % DIAG_OUT] = make_uint4(d.h0, d.h1, d.g0, d.g1);
    }
}

// Residues (n, n + 1) of both polynomials of a rotation in the extended basis: what a hoisted sum of that one term makes of them, with the loads
// apart from the arithmetic.
template <bool FP, bool COMPACT>
struct KeyPair {
    ulonglong2 v;
    __device__ __forceinline__ void load(const RotTermDev &T, const __amdgpu_buffer_rsrc_t, const u32 limb, const u32 n) { v = key_pair_ptr(T, limb, n); }
    __device__ __forceinline__ D2 fp() const { return to_d2(v); }
};
template <>
struct KeyPair<true, true> {
    u32x3 v;
    __device__ __forceinline__ void load(const RotTermDev &, const __amdgpu_buffer_rsrc_t key, const u32 limb, const u32 n) { v = key_record(key, limb, n); }
    __device__ __forceinline__ D2 fp() const { return key_record_fp(v); }
};
template <bool FP, int B, bool COMPACT>
struct Rotation {
    ulonglong2 x[B], b;
    KeyPair<FP, COMPACT> kb[B], ka[B];
    bool swap;
    __device__ __forceinline__ void load(const RotTermDev &T, const KeyLimb kl, const u32 n, const u32 e, const int nq, const int E, const int logN) {
        const u32 np = galois_index(n, T.galois, logN);
        swap = (np & 1u) != 0;
        const size_t N = (size_t)1 << logN, from = (np & ~1u) + e * N;
        const __amdgpu_buffer_rsrc_t key = key_rsrc(T);
#pragma unroll
        for (int d = 0; d < B; d++) {
            x[d] = load2(T.ext + (size_t)d * E * N + from);
            kb[d].load(T, key, kl.of(d, 0), n);
            ka[d].load(T, key, kl.of(d, 1), n);
        }
        if ((int)e < nq) b = load2(T.b + from);
    }
    // to [0, q); NEAR: of a prime just below 2^60 (modarith.h, Near60)
    template <bool NEAR>
    __device__ __forceinline__ void finish(const ModQ &m, const FpMod f, const Cst pmod, const bool with_b, const int premultiplied, u64 (&rb)[2], u64 (&ra)[2]) {
        if (FP) {
            double sb0 = 0, sb1 = 0, sa0 = 0, sa1 = 0;
#pragma unroll
            for (int d = 0; d < B; d++) {
                swap_if(swap, x[d]);
                const D2 xd = to_d2(x[d]), b0 = kb[d].fp(), a0 = ka[d].fp();
                sb0 += f.mul(xd.x, b0.x);
                sb1 += f.mul(xd.y, b0.y);
                sa0 += f.mul(xd.x, a0.x);
                sa1 += f.mul(xd.y, a0.y);
            }
            if (with_b) {
                swap_if(swap, b);
                const D2 bd = to_d2(b);
                const double p = (double)pmod.w;
                sb0 += premultiplied ? bd.x : f.mul(bd.x, p);
                sb1 += premultiplied ? bd.y : f.mul(bd.y, p);
            }
            rb[0] = f.canonical(sb0);
            rb[1] = f.canonical(sb1);
            ra[0] = f.canonical(sa0);
            ra[1] = f.canonical(sa1);
        } else if constexpr (!FP) {
            const u64 q = m.q;
            Acc3 sb[2] = {{0, 0, 0}, {0, 0, 0}}, sa[2] = {{0, 0, 0}, {0, 0, 0}};
#pragma unroll
            for (int d = 0; d < B; d++) {
                swap_if(swap, x[d]);
                const Pieces px = pieces(x[d].x), py = pieces(x[d].y);
                acc_mul(sb[0], px, pieces(kb[d].v.x));
                acc_mul(sb[1], py, pieces(kb[d].v.y));
                acc_mul(sa[0], px, pieces(ka[d].v.x));
                acc_mul(sa[1], py, pieces(ka[d].v.y));
            }
            if (NEAR) {
                const Near60 near(q);
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    rb[h] = near.reduce(sb[h]);
                    ra[h] = near.canonical(near.fold(near.reduce(sa[h])));
                }
                if (with_b) {
                    swap_if(swap, b);
                    const Cut p = near.cut(pmod.w, pmod.ws);
                    rb[0] = premultiplied ? rb[0] + b.x : near.add_mul(rb[0], b.x, p);
                    rb[1] = premultiplied ? rb[1] + b.y : near.add_mul(rb[1], b.y, p);
                }
#pragma unroll
                for (int h = 0; h < 2; h++) rb[h] = near.canonical(near.fold(rb[h]));
                return;
            }
#pragma unroll
            for (int h = 0; h < 2; h++) {   // below 3q
                rb[h] = acc_reduce(sb[h], m);
                ra[h] = cond_sub_u(cond_sub_u(acc_reduce(sa[h], m), 2 * q), q);
            }
            if (with_b) {                   // below 5q
                swap_if(swap, b);
                rb[0] += premultiplied ? b.x : mul_shoup_lazy_u(b.x, pmod.w, pmod.ws, q);
                rb[1] += premultiplied ? b.y : mul_shoup_lazy_u(b.y, pmod.w, pmod.ws, q);
            }
#pragma unroll
            for (int h = 0; h < 2; h++) rb[h] = cond_sub_u(cond_sub_u(cond_sub_u(rb[h], 4 * q), 2 * q), q);
        }
    }
};

// What a workgroup has of the sums it makes
struct DiagonalTile {
    u32 n, e, half, at;
    const uint4 *tab;
    u64 *y;
    size_t pol;               // words between the polynomials of a sum
    int sums;                 // of this half of the workgroup, at most DIAG_OUT / 2
    ulonglong2 (*made)[2][2][128];   // [turn][rotation of the turn][polynomial]: residues n, n + 1
    u64 (*acc)[256];          // [DIAG_OUT / 2 * 4]: what the accumulators have been reduced to
};
template <bool FP, int B, bool COMPACT, bool NEAR>
__device__ __forceinline__ void diagonal_sums(const HoistedArgs &args, const DiagonalTile &w, const u64 *__restrict__ a, const size_t a_stride,
                                              const ModQ m, const FpMod f, const Cst pmod, const KeyLimb kl, const int nq, const int E,
                                              const int logN, const int premultiplied, const u32 g) {
    constexpr int OUT = DIAG_OUT / 2;
    const u64 q = m.q, n8 = opaque_neg(8 * q), n4 = opaque_neg(4 * q), n2 = opaque_neg(2 * q), n1 = opaque_neg(q);
    const Near60 near(q);
    const size_t N = (size_t)1 << logN;
    const bool chain = (int)w.e < nq;
    // what the accumulators hold, added to acc < 8q, to below 8q
    auto more = [&](const u64 acc, const Dot2 &s) {
        if (NEAR) return near.fold(acc + near.reduce(s.s0, s.s1));
        return csub(acc + csub(dot_reduce_lazy(s, m), 8 * q, n8), 8 * q, n8);   // 13q to 8q, and the sum of two to 8q
    };
    Dot2 d[OUT][4];
#pragma unroll
    for (int i = 0; i < OUT; i++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            w.acc[i * 4 + v][threadIdx.x] = 0;
            dot_clear(d[i][v]);
        }
    Rotation<FP, B, COMPACT> r;
    if (w.half != 0) r.load(args.t[0], kl, w.n, w.e, nq, E, logN);
    for (u32 j0 = 0; j0 < g; j0 += 2) {
        const u32 j = j0 + w.half, turn = (j0 >> 1) & 1u;
        u64 rb[2] = {0, 0}, ra[2] = {0, 0};
        if (j != 0) {
            r.template finish<NEAR>(m, f, pmod, chain, premultiplied, rb, ra);
        } else if (chain) {
            const ulonglong2 b0 = load2(a + w.e * N + w.n), a0 = load2(a + a_stride + w.e * N + w.n);
            rb[0] = b0.x;
            rb[1] = b0.y;
            ra[0] = a0.x;
            ra[1] = a0.y;
        }
        w.made[turn][w.half][0][w.at] = make_ulonglong2(rb[0], rb[1]);
        w.made[turn][w.half][1][w.at] = make_ulonglong2(ra[0], ra[1]);
        if (j0 + 2 < g) r.load(args.t[j + 1], kl, w.n, w.e, nq, E, logN);   // in flight under the products below
        __syncthreads();   // the other turn's buffer is written next: its readers have passed this barrier by then
#pragma unroll
        for (u32 jj = 0; jj < 2; jj++) {
            const ulonglong2 xb = w.made[turn][jj][0][w.at], xa = w.made[turn][jj][1][w.at];
            const u64 x[4] = {xb.x, xb.y, xa.x, xa.y};
#pragma unroll
            for (int i = 0; i < OUT; i++) {
                const uint4 c = w.tab[(j0 + jj) * DIAG_OUT + i];
                const DotCst h{c.x, c.y, c.z, c.w};
#pragma unroll
                for (int v = 0; v < 4; v++) dot_add(d[i][v], x[v], h);
            }
        }
        if ((j0 & 6u) == 6u && j0 + 2 < g) {   // eight products: what the accumulators hold
#pragma unroll
            for (int i = 0; i < OUT; i++)
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    u64 &acc = w.acc[i * 4 + v][threadIdx.x];
                    acc = more(acc, d[i][v]);
                    dot_clear(d[i][v]);
                }
        }
    }
#pragma unroll
    for (int i = 0; i < OUT; i++) {
        if (i >= w.sums) break;
        u64 s[4];
#pragma unroll
        for (int v = 0; v < 4; v++) {
            s[v] = more(w.acc[i * 4 + v][threadIdx.x], d[i][v]);
            s[v] = csub(NEAR ? s[v] : csub(csub(s[v], 4 * q, n4), 2 * q, n2), q, n1);
        }
        u64 *to = w.y + (size_t)i * 2 * w.pol;
        stream_store2(to, s[0], s[1]);
        stream_store2(to + w.pol, s[2], s[3]);
    }
}

// The inner sums y[t][pol][e] = sum_j x_j[pol][e] (.) Q_tj[e]; x_0 is the ciphertext `a`, x_j its rotation under the key of term j - 1.  The
// rotations are made here, as a hoisted sum would make them, and never written: of a workgroup's 256 threads one half makes the even
// ones of 256 residues and one the odd ones, they meet in LDS, and each half goes on to their products with half of a chunk's diagonals
// (all of them would be 128 registers of sums per thread).  A wavefront lies in one run (UNIFORM: runs of 128 residues and more): the
// table entries are scalars, and a product is four multiply-adds with nothing loaded for it.
// Bound by the keys' way from memory.  31 rotations of 10 limbs of 2^16 (two digits) into 8 sums: 733 MB fetched, 84 written; 294 us as a
// hoisted sum that writes the rotations and a kernel that reads them back, 271 in one, 194 with a rotation's loads in flight under the
// products of the two before it, 4.2 TB/s (168 registers, three waves per SIMD; what the accumulators are reduced to stays in LDS for
// that).  Product of 128 x 128 tiles, pair layout 621 -> 501 us, 64 x 64 tiles 237 -> 222.
template <bool COMPACT, bool UNIFORM>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void diagonal_sums_kernel(
    const HoistedArgs args, const u64 *__restrict__ a, const size_t a_stride, const uint4 *__restrict__ tables, u64 *__restrict__ y,
    const ModQ *__restrict__ modq, const double *__restrict__ fp, LimbList ll, const Cst *__restrict__ pmods, const int nq, const int E,
    const int beta, const int n_full, const int logN, const int premultiplied, const u32 *__restrict__ koff, const int log_run, const u32 g,
    const u32 giants, const u32 chunks, const u32 tiles) {
    __shared__ ulonglong2 made[2][2][2][128];
    __shared__ u64 acc[DIAG_OUT / 2 * 4][256];
    // the chunks of a tile of 256 residues run back to back on one XCD, which then has its keys in L2
    u32 chunk, tile;
    if ((tiles & 7u) == 0) {
        const u32 xcd = blockIdx.x & 7u, slot = blockIdx.x >> 3;
        chunk = slot % chunks;
        tile = (slot / chunks) * 8u + xcd;
    } else {
        chunk = blockIdx.x % chunks;
        tile = blockIdx.x / chunks;
    }
    chunk = __builtin_amdgcn_readfirstlane(chunk);
    tile = __builtin_amdgcn_readfirstlane(tile);
    const size_t N = (size_t)1 << logN;
    DiagonalTile w;
    w.at = threadIdx.x & 127u;
    w.half = (u32)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 7));
    w.e = tile >> (logN - 8);
    w.n = ((tile & ((1u << (logN - 8)) - 1)) << 8) + 2 * w.at;
    const u32 first = chunk * DIAG_OUT + w.half * (DIAG_OUT / 2);
    w.sums = (int)giants - (int)first;
    w.pol = (size_t)E * N;
    w.y = y + ((size_t)first * 2 * E + w.e) * N + w.n;
    w.made = made;
    w.acc = acc;
    const int prime = (int)table_byte(ll.idx, w.e);
    const ModQ m = modq[prime];
    const KeyLimb kl = key_limb<COMPACT>(koff, prime, logN, n_full);
    const u32 lane_run = w.n >> log_run, run = UNIFORM ? (u32)__builtin_amdgcn_readfirstlane((int)lane_run) : lane_run;
    w.tab = tables + ((((size_t)w.e << (logN - log_run)) + run) * chunks + chunk) * g * DIAG_OUT + w.half * (DIAG_OUT / 2);
    const Cst pmod = (int)w.e < nq ? pmods[w.e] : Cst{0, 0};
    const FpMod f{fp[4 * prime], fp[4 * prime + 1]};
#define SUMS(FP, B, NEAR) diagonal_sums<FP, B, COMPACT, NEAR>(args, w, a, a_stride, m, f, pmod, kl, nq, E, logN, premultiplied, g)
    if (f.q != 0.0) {
        if (beta == 1) SUMS(true, 1, false);
        else if (beta == 2) SUMS(true, 2, false);
        else SUMS(true, 3, false);
    } else if (near_2_60(m.q) && beta <= 2) {   // (with three digits it would spill more)
        if (beta == 1) SUMS(false, 1, true);
        else SUMS(false, 2, true);
    } else {
        if (beta == 1) SUMS(false, 1, false);
        else if (beta == 2) SUMS(false, 2, false);
        else SUMS(false, 3, false);
    }
#undef SUMS
}
}  // namespace

bool diagonals_ok(const hemm_context *c, u32 k, u32 w, u32 g, int nq) {
    auto pow2 = [](u32 v) { return v != 0 && (v & (v - 1)) == 0; };
    for (u64 q : c->primes)   // what the lazy dot products and their reduction take
        if ((q >> 60) != 0 || (q >> 32) == 0) return false;
    // 4w <= N: a thread's two residues lie in one run of N / 2w
    return ring_has_fused_forms(c) && c->nP >= 1 && nq <= 3 * c->alpha && pow2(k) && pow2(w) && pow2(g) && g >= 4 && g <= k && g <= HOISTED_ARG_TERMS &&
           k <= w && w <= DIAG_MAX_W && 4 * (size_t)w <= c->N;
}
static u32 diagonal_chunks(u32 k, u32 g) { return (2 * k / g + DIAG_OUT - 1) / DIAG_OUT; }
size_t diagonal_table_words(const hemm_context *c, u32 k, u32 w, u32 g, int nq) {
    return (size_t)(nq + c->nP) * 2 * w * diagonal_chunks(k, g) * g * DIAG_OUT * 2;
}
void launch_diagonal_tables(hemm_context *c, const double *block, u32 k, u32 w, u32 g, double scale, int nq, u64 *tables, hipStream_t s) {
    const u32 chunks = diagonal_chunks(k, g);
    u32 log_w = 0;
    while ((1u << log_w) < w) log_w++;
    account(c, TR_POINTWISE, (size_t)k * w * 16 + diagonal_table_words(c, k, w, g, nq) * 8);
    hipLaunchKernelGGL(diagonal_tables_kernel, dim3(chunks * DIAG_OUT * g, (unsigned)(nq + c->nP)), dim3(256), 0, s, (const double2 *)block,
                       (const double2 *)encode_roots(c), (const Tw *)c->d_w, c->d_modq, c->d_fp, pmod_table(c), limbs_default(c, nq, 1), nq,
                       c->logN, k, log_w, g, 2 * k / g, chunks, scale, (uint4 *)tables);
}
void launch_diagonal_sums(hemm_context *c, const HoistedList &l, const u64 *a, size_t a_stride, u32 k, u32 w, u32 g, int nq, bool b_premultiplied,
                          const u64 *tables, u64 *y, hipStream_t s) {
    const int E = nq + c->nP, beta = (nq + c->alpha - 1) / c->alpha, n_full = c->nQ + c->nP;
    const u32 chunks = diagonal_chunks(k, g), giants = 2 * k / g, tiles = (u32)E << (c->logN - 8);
    const bool compact = (((const RotTermDev *)l.terms)[0].flags & ROT_TERM_COMPACT_KEY) != 0;
    if ((size_t)c->dnum * 2 * n_full * c->N * 8 >= ((size_t)1 << 32)) throw std::invalid_argument("hoisted terms need keys below 4 GiB");
    int log_run = c->logN;
    for (u32 v = 2 * w; v > 1; v >>= 1) log_run--;
    HoistedArgs args;
    memset(&args, 0, sizeof(args));
    memcpy(args.t, l.terms, (size_t)(g - 1) * sizeof(RotTermDev));
    memcpy(args.off, l.offsets, (size_t)g * sizeof(u32));
    account(c, TR_KEYPROD, ((size_t)(g - 1) * 2 * beta * E + (size_t)beta * E + 3 * nq + (size_t)giants * 2 * E) * c->N * 8 + diagonal_table_words(c, k, w, g, nq) * 8);
    const dim3 grid(tiles * chunks), wg(256);
#define DIAGONAL_SUMS(C, U)                                                                                                               \
    hipLaunchKernelGGL((diagonal_sums_kernel<C, U>), grid, wg, 0, s, args, a, a_stride, (const uint4 *)tables, y, c->d_modq, c->d_fp,      \
                       limbs_default(c, nq, 1), pmod_table(c), nq, E, beta, n_full, c->logN, b_premultiplied ? 1 : 0, c->d_key_off, log_run, g,  \
                       giants, chunks, tiles)
    if (compact) {
        if (log_run >= 7) DIAGONAL_SUMS(true, true);
        else DIAGONAL_SUMS(true, false);
    } else {
        if (log_run >= 7) DIAGONAL_SUMS(false, true);
        else DIAGONAL_SUMS(false, false);
    }
#undef DIAGONAL_SUMS
}
