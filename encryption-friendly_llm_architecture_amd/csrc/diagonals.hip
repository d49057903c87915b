// A plaintext matrix applied to every row of an encrypted one as a sum over its diagonals, in baby and giant steps:
//   A B = sum_r rho^r(A) (.) P_r = sum_t rho^(g t)( sum_j rho^j(A) (.) Q_tj ),   Q_tj = rho^(-g t)(P_(g t + j)).
// P_r, 1 - k <= r < k, holds B[c + r][c] in column c of every row of a k x k tile (rows of w slots: w / k tiles side by side), zero
// where c + r lies outside: the same w values in every row.  Such a plaintext is a polynomial in X^(N / 2w), and its transform is constant
// over runs of N / 2w residues: 2w values per limb instead of N.  The two steps that are not key switches are here: the tables
// of all Q_tj, made once per weight, and the inner sums, from rotations that stay in the extended basis.
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
        transform_runs(IntFieldT<true>(modq, nullptr, nullptr, fp, prime), buf, tw, w, (int)log_w + 1);
    // the rotation by nothing enters as P times the ciphertext, on the chain limbs: its diagonals carry the factor
    const bool own = j == 0, none = own && (int)e >= nq;
    for (u32 run = threadIdx.x; run < 2 * w; run += 256) {
        u64 h = none ? 0 : buf[run];
        if (own && !none) h = mulmod(h, pmod[e].w, m);
        const DotCst d = dot_cst(h, mulmod(h, (u64)1 << 30, m));
        tables[((((size_t)e * 2 * w + run) * chunks + t / DIAG_OUT) * g + j) * DIAG_OUT + t % DIAG_OUT] = make_uint4(d.h0, d.h1, d.g0, d.g1);
    }
}

// The inner sums y[t][pol][e] = sum_j x_j[pol][e] (.) Q_tj[e]; x_0 is the ciphertext `a`, x_j its rotations.  A lane has one residue of both
// polynomials, a wavefront lies in one run (UNIFORM: runs of 64 residues and more), so the table entries are scalars and a product is four
// multiply-adds with nothing loaded for it.  124 registers, four waves per SIMD; 31 rotations of 10 limbs of 2^16 into 8 sums, 430 MB: 115 us.
template <bool UNIFORM>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(UNIFORM ? 4 : 2))) void diagonal_sums_kernel(
    const u64 *__restrict__ rotated, const u64 *__restrict__ a, const size_t a_stride, const uint4 *__restrict__ tables, u64 *__restrict__ y,
    const ModQ *__restrict__ modq, LimbList ll, const int nq, const int E, const int logN, const int log_run, const u32 g, const u32 giants,
    const u32 chunks, const u32 tiles) {
    // the chunks of a tile of 256 residues run back to back on one XCD, which then has its rotations in L2
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
    const u32 e = tile >> (logN - 8), n = ((tile & ((1u << (logN - 8)) - 1)) << 8) + threadIdx.x;
    const ModQ m = modq[__builtin_amdgcn_readfirstlane((int)table_byte(ll.idx, e))];
    const u64 q = m.q, n8 = opaque_neg(8 * q), n4 = opaque_neg(4 * q), n2 = opaque_neg(2 * q), n1 = opaque_neg(q);
    const u32 lane_run = n >> log_run, run = UNIFORM ? (u32)__builtin_amdgcn_readfirstlane((int)lane_run) : lane_run;
    const uint4 *__restrict__ tab = tables + ((((size_t)e << (logN - log_run)) + run) * chunks + chunk) * g * DIAG_OUT;
    const u64 *x0 = rotated + (size_t)e * N + n;
    u64 acc[DIAG_OUT][2];
    Dot2 d[DIAG_OUT][2];
#pragma unroll
    for (int i = 0; i < DIAG_OUT; i++) {
        acc[i][0] = acc[i][1] = 0;
        dot_clear(d[i][0]);
        dot_clear(d[i][1]);
    }
    for (u32 j0 = 0; j0 < g; j0 += 4) {
        u64 x[4][2];
#pragma unroll
        for (u32 jj = 0; jj < 4; jj++)
#pragma unroll
            for (u32 p = 0; p < 2; p++) {
                const u32 j = j0 + jj;
                if (j == 0)
                    x[jj][p] = (int)e < nq ? a[p * a_stride + (size_t)e * N + n] : 0;
                else
                    x[jj][p] = x0[((size_t)(j - 1) * 2 + p) * E * N];
            }
#pragma unroll
        for (u32 jj = 0; jj < 4; jj++) {
#pragma unroll
            for (int i = 0; i < DIAG_OUT; i++) {
                const uint4 c = tab[(j0 + jj) * DIAG_OUT + i];
                const DotCst h{c.x, c.y, c.z, c.w};
                dot_add(d[i][0], x[jj][0], h);
                dot_add(d[i][1], x[jj][1], h);
            }
        }
        if ((j0 & 4u) != 0 || j0 + 4 == g) {   // eight products: what the accumulators hold
#pragma unroll
            for (int i = 0; i < DIAG_OUT; i++)
#pragma unroll
                for (int p = 0; p < 2; p++) {   // 13q to 8q, and the sum of two to 8q
                    acc[i][p] = csub(acc[i][p] + csub(dot_reduce_lazy(d[i][p], m), 8 * q, n8), 8 * q, n8);
                    dot_clear(d[i][p]);
                }
        }
    }
#pragma unroll
    for (int i = 0; i < DIAG_OUT; i++) {
        const u32 t = chunk * DIAG_OUT + i;
        if (t >= giants) break;
#pragma unroll
        for (u32 p = 0; p < 2; p++)
            __builtin_nontemporal_store(csub(csub(csub(acc[i][p], 4 * q, n4), 2 * q, n2), q, n1),
                                        y + (((size_t)t * 2 + p) * E + e) * N + n);
    }
}
}  // namespace

bool diagonals_ok(const hemm_context *c, u32 k, u32 w, u32 g) {
    auto pow2 = [](u32 v) { return v != 0 && (v & (v - 1)) == 0; };
    for (u64 q : c->primes)   // what the lazy dot products and their reduction take
        if ((q >> 60) != 0 || (q >> 32) == 0) return false;
    return ring_has_fused_forms(c) && c->nP >= 1 && pow2(k) && pow2(w) && pow2(g) && g >= 4 && g <= k && k <= w && w <= DIAG_MAX_W && 2 * (size_t)w <= c->N;
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
void launch_diagonal_sums(hemm_context *c, const u64 *rotated, const u64 *a, size_t a_stride, u32 k, u32 w, u32 g, int nq, const u64 *tables,
                          u64 *y, hipStream_t s) {
    const int E = nq + c->nP;
    const u32 chunks = diagonal_chunks(k, g), giants = 2 * k / g, tiles = (u32)E << (c->logN - 8);
    int log_run = c->logN;
    for (u32 v = 2 * w; v > 1; v >>= 1) log_run--;
    account(c, TR_MASKED, ((size_t)(g - 1) * 2 * E + 2 * nq + (size_t)giants * 2 * E) * c->N * 8 + diagonal_table_words(c, k, w, g, nq) * 8);
    const dim3 grid(tiles * chunks), wg(256);
#define DIAGONAL_SUMS(U)                                                                                                                  \
    hipLaunchKernelGGL((diagonal_sums_kernel<U>), grid, wg, 0, s, rotated, a, a_stride, (const uint4 *)tables, y, c->d_modq,               \
                       limbs_default(c, nq, 1), nq, E, c->logN, log_run, g, giants, chunks, tiles)
    if (log_run >= 6)
        DIAGONAL_SUMS(true);
    else
        DIAGONAL_SUMS(false);
#undef DIAGONAL_SUMS
}
