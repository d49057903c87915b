// CKKS encode / decode on the device: the canonical embedding restricted to the orbit zeta^(5^j) and its inverse
// (HEaaN::EnDecoder::encode / decode, EnDecoder.hpp:51,66), in double precision, and the encryption and decryption around
// them.
//
//   encode: slots z[n] (n = N/2 complex numbers) -> n-point "special" inverse transform (decimation in frequency,
//           stages len = n, n/2, ..., 2, butterfly (a, b) -> (a + b, (a - b) * ksi[M - 5^j * M / 4 len])) -> bit reversal ->
//           coefficient i = round(Re z_i / n * scale), coefficient i + n = round(Im z_i / n * scale) -> residues modulo
//           every limb's prime -> forward NTT.
//   decode: inverse NTT of the first one or two limbs -> centred integer (CRT over two limbs) / scale -> bit reversal ->
//           stages len = 2, 4, ..., n, butterfly (a, b) -> (a + b ksi, a - b ksi), ksi = ksi[5^j * M / 4 len].
//
// Every floating-point operation is a single IEEE operation in a fixed order (no contraction into fused multiply-adds),
// and the root table holds the doubles cos / sin return on the host, so the result does not depend on where the
// transform runs: a host loop over the same butterflies gives the same bits.
//
// From N = 2^10 on the n points are viewed as R x 256 and take two launches, like the residue transforms: the stages with
// len > 256 down the columns, the others inside the rows.  What bounded this transform was latency, not work: a tile of
// 4096 points per workgroup left all but eight CUs idle, and every butterfly waited for two dependent table reads (5^j, then
// the root).  Here a tile has 512 or 1024 points (2048 where rows meet), a thread owns one butterfly of each stage and
// loads the roots of all its stages, laid out in stage order, before it starts.  The row pass of an encoding leaves rounded
// integers, in coefficient order, which the first pass of the NTT reduces modulo each prime as it loads them; the row
// pass of a decoding recovers them from the residues it reads.  One message at N = 2^16, level 12: 24 + 3 x 3.5 + 14 us for the
// embedding and the lift before, 4 + 5 us now.
#include <cmath>
#include <mutex>
#include <unordered_map>

#include "hemm_internal.hpp"

#pragma clang fp contract(off)

namespace {

struct EmbTables {
    double2 *enc = nullptr, *dec = nullptr;   // [n] each: root of butterfly j of the stage of half length h at h + j
};
std::mutex g_mu;
std::unordered_map<const hemm_context *, EmbTables> g_tabs;

const EmbTables &tables_of(const hemm_context *c) {
    std::lock_guard<std::mutex> lk(g_mu);
    auto it = g_tabs.find(c);
    if (it != g_tabs.end()) return it->second;
    const size_t n = (size_t)c->N / 2, M = 2 * (size_t)c->N;
    std::vector<double2> k(M + 1);   // exp(2 pi i k / M)
    // separate loops: a cos / sin pair on one value may be merged into one sincos call, which rounds differently
    for (size_t i = 0; i <= M; i++) k[i].x = cos(2.0 * M_PI * (double)i / (double)M);
    for (size_t i = 0; i <= M; i++) k[i].y = sin(2.0 * M_PI * (double)i / (double)M);
    std::vector<size_t> rot(n);      // 5^j mod M
    u64 g = 1;
    for (size_t j = 0; j < n; j++) {
        rot[j] = (size_t)g;
        g = g * 5 % M;
    }
    std::vector<double2> enc(n), dec(n);
    for (size_t h = 1; h < n; h <<= 1) {
        const size_t lenq = h << 3, gap = M / lenq;
        for (size_t j = 0; j < h; j++) {
            const size_t r = rot[j] & (lenq - 1);
            enc[h + j] = k[(lenq - r) * gap];
            dec[h + j] = k[r * gap];
        }
    }
    EmbTables t;
    HEMM_HIP(hipMalloc((void **)&t.enc, n * sizeof(double2)));
    HEMM_HIP(hipMalloc((void **)&t.dec, n * sizeof(double2)));
    HEMM_HIP(hipMemcpy(t.enc, enc.data(), n * sizeof(double2), hipMemcpyHostToDevice));
    HEMM_HIP(hipMemcpy(t.dec, dec.data(), n * sizeof(double2), hipMemcpyHostToDevice));
    return g_tabs.emplace(c, t).first->second;
}

__device__ __forceinline__ double2 cmul(const double2 v, const double2 k) {
    return make_double2(v.x * k.x - v.y * k.y, v.x * k.y + v.y * k.x);
}
template <bool DECODE>
__device__ __forceinline__ void butterfly(double2 &a, double2 &b, const double2 k) {
    if (!DECODE) {
        const double2 u = make_double2(a.x + b.x, a.y + b.y), v = make_double2(a.x - b.x, a.y - b.y);
        a = u;
        b = cmul(v, k);
    } else {
        const double2 t = cmul(b, k);
        const double2 u = a;
        a = make_double2(u.x + t.x, u.y + t.y);
        b = make_double2(u.x - t.x, u.y - t.y);
    }
}
__device__ __forceinline__ long long round_half_away(double x) { return (long long)__builtin_round(x); }
// the real value of a coefficient from its residues modulo the first prime, or the first two
struct CentreArgs {
    u64 q0, q1, q0inv;
    int two;
    double scale;
};
__device__ __forceinline__ double centred(const u64 l0, const u64 l1, const CentreArgs &c, const ModQ &m1) {
    if (!c.two) return (l0 > c.q0 / 2 ? -(double)(c.q0 - l0) : (double)l0) / c.scale;
    const u64 b = reduce64(l0, m1);
    const u64 k = mulmod(submod(l1, b, c.q1), c.q0inv, m1);
    const unsigned __int128 Q = (unsigned __int128)c.q0 * c.q1, x = (unsigned __int128)l0 + (unsigned __int128)c.q0 * k;
    double w;
    if (x > Q / 2) {
        const unsigned __int128 y = Q - x;
        w = -((double)(u64)(y >> 64) * 18446744073709551616.0 + (double)(u64)y);
    } else
        w = (double)(u64)(x >> 64) * 18446744073709551616.0 + (double)(u64)x;
    return w / c.scale;
}

// ---- two launches over the R x 256 view, R = 2^LR = n / 256 -----------------------------------------------------------
// Where an encoding's column pass finds its slots and a decoding's leaves them: complex numbers, or the real parts of the
// first `count` slots (the others are zero resp. not wanted), in memory the host sees as well.
struct Slots {
    double2 *z;        // [n_msgs][n]
    double *re;        // z == nullptr: [count]
    u32 count;
};
// The column stages.  A workgroup owns R rows of CW columns, a thread one butterfly of each stage: rows i and i + d.
// POINTS of a workgroup: 1024, or 2048 (2^16 points) where the slots are read from host memory: segments of 128 bytes are half the requests,
// 11.2 -> 8.8 us for 128 x 128 values.  Writing there gains nothing from them (5.9 / 6.5).
template <int LR, bool DECODE, int POINTS>
__global__ __launch_bounds__(POINTS / 2) void emb_cols_kernel(const Slots io, double2 *__restrict__ z, const double2 *__restrict__ roots) {
    constexpr int R = 1 << LR, CW = R >= 4 ? POINTS / R : 256;
    __shared__ double2 s[R * CW];
    const u32 cc = threadIdx.x % CW, q = threadIdx.x / CW, col = blockIdx.x * CW + cc, n = 256u << LR;
    double2 k[LR];
    u32 row[LR];   // the upper row of this thread's butterfly in stage t, half length 256 d
#pragma unroll
    for (int t = 0; t < LR; t++) {
        const u32 d = DECODE ? 1u << t : (u32)R >> (t + 1), j = q & (d - 1);
        k[t] = roots[((d + j) << 8) + col];
        row[t] = ((q - j) << 1) + j;
    }
    double2 *zm = z + (size_t)blockIdx.y * n + col;
    double2 a, b;
#pragma unroll
    for (int t = 0; t < LR; t++) {
        const u32 d = DECODE ? 1u << t : (u32)R >> (t + 1), ra = row[t], rb = row[t] + d;
        if (t == 0) {
            if (DECODE) {
                a = zm[ra << 8];
                b = zm[rb << 8];
            } else if (io.z != nullptr) {
                a = io.z[(size_t)blockIdx.y * n + (ra << 8) + col];
                b = io.z[(size_t)blockIdx.y * n + (rb << 8) + col];
            } else {
                const u32 ia = (ra << 8) + col, ib = (rb << 8) + col;
                a = make_double2(ia < io.count ? io.re[ia] : 0.0, 0.0);
                b = make_double2(ib < io.count ? io.re[ib] : 0.0, 0.0);
            }
        } else {
            a = s[ra * CW + cc];
            b = s[rb * CW + cc];
        }
        butterfly<DECODE>(a, b, k[t]);
        if (t < LR - 1) {
            // a thread writes where it has just read: the other threads' turn comes after the barrier
            s[ra * CW + cc] = a;
            s[rb * CW + cc] = b;
            __syncthreads();
        } else if (!DECODE) {
            zm[ra << 8] = a;
            zm[rb << 8] = b;
        } else if (io.z != nullptr) {
            io.z[(size_t)blockIdx.y * n + (ra << 8) + col] = a;
            io.z[(size_t)blockIdx.y * n + (rb << 8) + col] = b;
        } else {
            const u32 ia = (ra << 8) + col, ib = (rb << 8) + col;
            if (ia < io.count) io.re[ia] = a.x;
            if (ib < io.count) io.re[ib] = b.x;
        }
    }
}

// The row stages and the integers.  Coefficient i sits at point brev(i): i = brev8(column) R + brev(row).  A workgroup owns
// the W rows whose reversed index runs over W consecutive values, so that it touches the coefficients in runs of W.
// Encode: z -> coef (coefficient order); decode: residues co[limb][N] -> z.
// Eight rows, runs of 64 bytes; up to 256 rows of all messages together, which would leave most CUs without a workgroup (a decoding's
// integers and divisions are 4 us of instructions on sixteen), two rows, runs of 16.  From 2^15 points the four workgroups that touch
// the same 64 bytes then lie on one XCD; smaller rings have too few workgroups for that and gain from the rows all the same.
// Whole calls, us with eight / two rows; the line lies where both sides were measured, two rows still lead one message past it:
//   points                                   2^12        2^13        2^14        2^15        2^16
//   decode, two limbs                   18.5/15.4   19.5/16.6   20.1/17.3   21.5/18.1   22.2/19.0
//   encode, three limbs, one message    14.3/12.8   15.7/13.9   16.3/14.5   17.1/15.2   17.7/15.8
//           256 rows of messages        16.3/14.8   18.7/17.4   18.6/16.7   19.6/17.8   19.0/17.2
//           one message more            16.3/14.9               19.0/17.9               21.3/19.6
template <int LR, bool DECODE, int W>
__global__ __launch_bounds__(128 * W) void emb_rows_kernel(double2 *__restrict__ z, const double2 *__restrict__ roots,
                                                        long long *__restrict__ coef, const double scale,
                                                        const u64 *__restrict__ co, const CentreArgs ca,
                                                        const ModQ *__restrict__ modq) {
    constexpr int R = 1 << LR, LW = W == 8 ? 3 : 1, PITCH = 257, TH = 128 * W, SHARE = R < 8 ? 1 : 8 / W;
    __shared__ double2 s[W * PITCH];
    const u32 x = blockIdx.x, slot = R >= 64 ? ((x & 7u) + 8u * ((x >> 3) / SHARE)) * SHARE + (x >> 3) % SHARE : x;
    const u32 n = 256u << LR, w = threadIdx.x >> 7, q = threadIdx.x & 127u, i0 = slot * W;
    const u32 r = __brev(i0 + w) >> (32 - LR);   // the row in this slot
    double2 k[8];
#pragma unroll
    for (int t = 0; t < 8; t++) {
        const u32 d = DECODE ? 1u << t : 128u >> t;
        k[t] = roots[d + (q & (d - 1))];
    }
    double2 *zr = z + (size_t)blockIdx.y * n + ((size_t)r << 8);
    double2 *sr = s + w * PITCH;
    if (DECODE) {
        const ModQ m1 = modq[ca.two];
        const u64 *l1 = co + (ca.two ? 2 * (size_t)n : 0);
#pragma unroll
        for (u32 e = threadIdx.x; e < 256u * W; e += TH) {
            const u32 ww = e & (W - 1), cb = e >> LW, i = (cb << LR) + i0 + ww;
            s[ww * PITCH + (__brev(cb) >> 24)] =
                make_double2(centred(co[i], l1[i], ca, m1), centred(co[n + i], l1[n + i], ca, m1));
        }
        __syncthreads();
    }
    double2 a, b;
#pragma unroll
    for (int t = 0; t < 8; t++) {
        const u32 d = DECODE ? 1u << t : 128u >> t, j = q & (d - 1), ia = ((q - j) << 1) + j, ib = ia + d;
        if (!DECODE && t == 0) {
            a = zr[ia];
            b = zr[ib];
        } else {
            a = sr[ia];
            b = sr[ib];
        }
        butterfly<DECODE>(a, b, k[t]);
        if (DECODE && t == 7) {
            zr[ia] = a;
            zr[ib] = b;
        } else {
            sr[ia] = a;
            sr[ib] = b;
            __syncthreads();
        }
    }
    if (!DECODE) {
        const double inv_n = 1.0 / (double)n;   // a power of two: the same value a division by n gives
        long long *o = coef + (size_t)blockIdx.y * 2 * n;
#pragma unroll
        for (u32 e = threadIdx.x; e < 256u * W; e += TH) {
            const u32 ww = e & (W - 1), cb = e >> LW, i = (cb << LR) + i0 + ww;
            const double2 v = s[ww * PITCH + (__brev(cb) >> 24)];
            o[i] = round_half_away(v.x * inv_n * scale);
            o[n + i] = round_half_away(v.y * inv_n * scale);
        }
    }
}

// ---- rings below 2^10: one workgroup per message ----------------------------------------------------------------------
template <bool DECODE>
__global__ __launch_bounds__(128) void emb_tile_kernel(double2 *__restrict__ z, const u32 n, const double2 *__restrict__ roots) {
    __shared__ double2 s[256];
    double2 *p = z + (size_t)blockIdx.x * n;
    for (u32 e = threadIdx.x; e < n; e += blockDim.x) s[e] = p[e];
    __syncthreads();
    for (u32 step = 1; step < n; step <<= 1) {
        const u32 h = DECODE ? step : n / step / 2;
        for (u32 t = threadIdx.x; t < n / 2; t += blockDim.x) {
            const u32 j = t & (h - 1), i = (t / h) * 2 * h;
            butterfly<DECODE>(s[i + j], s[i + j + h], roots[h + j]);
        }
        __syncthreads();
    }
    for (u32 e = threadIdx.x; e < n; e += blockDim.x) p[e] = s[e];
}
// transformed slots -> residues of the rounded coefficients, limb by limb (coefficient form, ready for the NTT)
__global__ __launch_bounds__(256) void emb_lift_kernel(const double2 *__restrict__ z, const u32 n, const int log_n,
                                                       const double scale, const ModQ *__restrict__ modq, LimbList ll,
                                                       const int n_limbs, u64 *__restrict__ out) {
    const u32 i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const double2 v = z[(size_t)blockIdx.y * n + (__brev(i) >> (32 - log_n))];
    const double inv_n = 1.0 / (double)n;
    const long long c0 = round_half_away(v.x * inv_n * scale), c1 = round_half_away(v.y * inv_n * scale);
    u64 *o = out + (size_t)blockIdx.y * n_limbs * 2 * n;
    for (int j = 0; j < n_limbs; j++) {
        const ModQ m = modq[table_byte(ll.idx, j)];
        const u64 r0 = reduce64((u64)(c0 < 0 ? -c0 : c0), m), r1 = reduce64((u64)(c1 < 0 ? -c1 : c1), m);
        o[(size_t)j * 2 * n + i] = c0 < 0 && r0 ? m.q - r0 : r0;
        o[(size_t)j * 2 * n + n + i] = c1 < 0 && r1 ? m.q - r1 : r1;
    }
}
// coefficient form of the first limb (or the first two) -> centred value / scale, written in bit-reversed order
__global__ __launch_bounds__(256) void emb_centre_kernel(const u64 *__restrict__ co, const u32 n, const int log_n,
                                                         const CentreArgs ca, const ModQ *__restrict__ modq,
                                                         double2 *__restrict__ z) {
    const u32 i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const ModQ m1 = modq[ca.two];
    const u64 *l1 = co + (ca.two ? 2 * (size_t)n : 0);
    z[__brev(i) >> (32 - log_n)] = make_double2(centred(co[i], l1[i], ca, m1), centred(co[n + i], l1[n + i], ca, m1));
}

constexpr unsigned pow2(int e) { return e > 0 ? 1u << e : 1u; }
template <bool DECODE>
void cols_stages(const hemm_context *c, const Slots &io, double2 *z, int n_msgs, hipStream_t s) {
    const EmbTables &t = tables_of(c);
    const double2 *roots = DECODE ? t.dec : t.enc;
#define EMB_COLS(LR)                                                                                                       \
    hipLaunchKernelGGL((emb_cols_kernel<LR, DECODE, LR >= 2 ? 1024 : 512>), dim3(pow2(LR - 2), n_msgs), dim3(LR >= 2 ? 512 : 256), \
                       0, s, io, z, roots)
    switch (c->logN - 9) {
        case 1: EMB_COLS(1); break;
        case 2: EMB_COLS(2); break;
        case 3: EMB_COLS(3); break;
        case 4: EMB_COLS(4); break;
        case 5: EMB_COLS(5); break;
        case 6: EMB_COLS(6); break;
        default:
            if (!DECODE && io.z == nullptr)
                hipLaunchKernelGGL((emb_cols_kernel<7, false, 2048>), dim3(16, n_msgs), dim3(1024), 0, s, io, z, roots);
            else
                EMB_COLS(7);
    }
#undef EMB_COLS
}
template <bool DECODE>
void rows_stages(const hemm_context *c, double2 *z, long long *coef, double scale, const u64 *co, const CentreArgs &ca,
                 int n_msgs, hipStream_t s) {
    const EmbTables &t = tables_of(c);
    const double2 *roots = DECODE ? t.dec : t.enc;
#define EMB_ROWS_OF(LR, W)                                                                                            \
    hipLaunchKernelGGL((emb_rows_kernel<LR, DECODE, W>), dim3((1u << LR) / (W), n_msgs), dim3(128 * (W)), 0, s, z, roots, coef, scale, co, ca, \
                       c->d_modq)
#define EMB_ROWS(LR)                            \
    do {                                        \
        if constexpr (!DECODE && LR >= 3)       \
            if ((n_msgs << LR) > 256) {         \
                EMB_ROWS_OF(LR, 8);             \
                break;                          \
            }                                   \
        EMB_ROWS_OF(LR, 2);                     \
    } while (0)   // (a decoding is one message)
    switch (c->logN - 9) {
        case 1: EMB_ROWS(1); break;
        case 2: EMB_ROWS(2); break;
        case 3: EMB_ROWS(3); break;
        case 4: EMB_ROWS(4); break;
        case 5: EMB_ROWS(5); break;
        case 6: EMB_ROWS(6); break;
        default: EMB_ROWS(7); break;
    }
#undef EMB_ROWS
#undef EMB_ROWS_OF
}

CentreArgs centre_args(const hemm_context *c, int n_limbs, double scale) {
    CentreArgs a;
    a.two = n_limbs == 2 ? 1 : 0;
    a.q0 = c->primes[0];
    a.q1 = a.two ? c->primes[1] : 1;
    a.q0inv = a.two ? h_invmod(a.q0 % a.q1, a.q1) : 0;
    a.scale = scale;
    return a;
}
}  // namespace

const void *encode_roots(const hemm_context *c) { return tables_of(c).enc; }

void hemm_embedding_tables_free(const hemm_context *c) {
    std::lock_guard<std::mutex> lk(g_mu);
    auto it = g_tabs.find(c);
    if (it == g_tabs.end()) return;
    (void)hipFree(it->second.enc);
    (void)hipFree(it->second.dec);
    g_tabs.erase(it);
}

// slots: [n_msgs][N/2] complex doubles on the device, or re: the real parts of the first `count` slots of one message;
// work: [n_msgs][N] words, may be `slots`; out: [n_msgs][n_limbs][N] NTT form, or with enc a workspace of that size
void launch_encode(const hemm_context *c, const double *slots, const double *re, size_t count, double scale, const LimbList &ll,
                   int n_limbs, int n_msgs, u64 *work, u64 *out, hipStream_t s, const EncryptTail *enc, u64 error_key) {
    if (c->N < 16) throw std::invalid_argument("encode needs N >= 16");
    const u32 n = (u32)c->N / 2;
    account(c, TR_POINTWISE, (size_t)n_msgs * 2 * c->N * 8, 2);
    if (ring_has_fused_forms(c)) {
        // the column pass goes through `out`, whose first words of each message the NTT writes only after the row pass
        double2 *z = (double2 *)out;
        Slots io{(double2 *)slots, (double *)re, (u32)count};
        cols_stages<false>(c, io, z, n_msgs, s);
        rows_stages<false>(c, z, (long long *)work, scale, nullptr, CentreArgs{}, n_msgs, s);
        const LiftSource ls{(const long long *)work, (size_t)c->N, error_key, enc != nullptr ? 1 : 0};
        (void)launch_ntt_lifted(c, ls, out, ll, n_limbs, n_msgs, (size_t)n_limbs * c->N, s, enc);
        return;
    }
    if (enc != nullptr || slots == nullptr) throw std::invalid_argument("this form of encode needs N >= 1024");
    double2 *z = (double2 *)work;
    if ((const double *)work != slots)
        HEMM_HIP(hipMemcpyAsync(work, slots, (size_t)n_msgs * c->N * 8, hipMemcpyDeviceToDevice, s));
    hipLaunchKernelGGL(emb_tile_kernel<false>, dim3(n_msgs), dim3(128), 0, s, z, n, tables_of(c).enc);
    hipLaunchKernelGGL(emb_lift_kernel, dim3((n + 255) / 256, n_msgs), dim3(256), 0, s, z, n, c->logN - 1, scale, c->d_modq, ll,
                       n_limbs, out);
    LimbList sl;
    for (int j = 0; j < HEMM_MAX_PRIMES; j++) sl.idx[j] = (uint8_t)j;
    launch_ntt_slots(c, out, ll, sl, n_limbs, n_msgs, (size_t)n_limbs * c->N, false, s);
}

// pt: [>= n_limbs][N] NTT form, limbs of chain primes 0 (and 1), or with a != nullptr the first polynomial of a ciphertext
// whose second is a (decrypted under sk); work: [n_limbs][N].  slots: [N/2] complex doubles; re != nullptr: slots is only a
// workspace and the real parts of the first `count` slots go to re
void launch_decode(const hemm_context *c, const u64 *pt, const u64 *a, const u64 *sk, int n_limbs, double scale, u64 *work,
                   double *slots, double *re, size_t count, hipStream_t s) {
    if (c->N < 16) throw std::invalid_argument("decode needs N >= 16");
    if (n_limbs < 1 || n_limbs > 2) throw std::invalid_argument("decode reads one or two limbs");
    const u32 n = (u32)c->N / 2;
    LimbList ll;
    for (int j = 0; j < HEMM_MAX_PRIMES; j++) ll.idx[j] = (uint8_t)j;
    const CentreArgs ca = centre_args(c, n_limbs, scale);
    double2 *z = (double2 *)slots;
    account(c, TR_POINTWISE, (size_t)(n_limbs + 1) * c->N * 8, 2);
    if (ring_has_fused_forms(c)) {
        if (a != nullptr)
            (void)launch_intt_decrypt(c, pt, a, sk, work, n_limbs, s);
        else
            (void)launch_intt_from(c, pt, (size_t)n_limbs * c->N, work, ll, ll, n_limbs, 1, (size_t)n_limbs * c->N, s);
        rows_stages<true>(c, z, nullptr, 0.0, work, ca, 1, s);
        cols_stages<true>(c, Slots{re == nullptr ? z : nullptr, re, (u32)count}, z, 1, s);
        return;
    }
    if (a != nullptr || re != nullptr) throw std::invalid_argument("this form of decode needs N >= 1024");
    HEMM_HIP(hipMemcpyAsync(work, pt, (size_t)n_limbs * c->N * 8, hipMemcpyDeviceToDevice, s));
    launch_ntt_slots(c, work, ll, ll, n_limbs, 1, (size_t)n_limbs * c->N, true, s);
    hipLaunchKernelGGL(emb_centre_kernel, dim3((n + 255) / 256), dim3(256), 0, s, work, n, c->logN - 1, ca, c->d_modq, z);
    hipLaunchKernelGGL(emb_tile_kernel<true>, dim3(1), dim3(128), 0, s, z, n, tables_of(c).dec);
}
