// Internal host-side declarations shared by the C-ABI translation units.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <stdexcept>
#include <string>
#include <vector>

#include "modarith.h"

#define HEMM_MAX_PRIMES 64

// Which prime each limb of an operand uses.  Limb j of an operand whose chain part has `nq`
// active limbs uses prime j when j < nq, and special prime nQ + (j - nq) otherwise; explicit
// lists cover everything else (digit subsets, benchmark batches).
struct __align__(4) LimbList {
    uint8_t idx[HEMM_MAX_PRIMES];
};
// Entry i, the same for the whole wavefront, of a byte table in the kernel arguments that starts at a multiple of four bytes.
// There are no scalar loads of a byte: read as one, the entry is a vector load, a trip to memory of its own at the start of every
// workgroup in front of the loads that need it; as a part of its word it comes through the scalar cache (rotation at N = 2^13 50.2 ->
// 48.9 us, ciphertext product at level 9 129.2 -> 126.8 us, 16 polynomials' ModDown 113 -> 111.5 us).
__device__ __forceinline__ u32 table_byte(const uint8_t *t, const u32 i) {
    u32 w;
    __builtin_memcpy(&w, __builtin_assume_aligned(t + (i & ~3u), 4), 4);
    return (u32)__builtin_amdgcn_readfirstlane((int)((w >> (8u * (i & 3u))) & 255u));   // i may come out of a division in vector registers
}

struct hemm_context {
    int device;
    int logN, N, nQ, nP, dnum, alpha;
    std::vector<u64> primes;        // nQ chain primes, then nP special primes
    std::vector<u64> psi;           // primitive 2N-th roots
    std::vector<ModQ> modq;         // host copy
    // device tables, all [prime][N] unless noted
    u64 *d_w, *d_iw;                // (psi^bitrev(i), Shoup quotient), forward and inverse transform; N >= 2^10: doubles of primes below
                                    // 2^44, of primes just below 2^60 (w, 2^32 w mod q), both cut at bit 29
    u64 *d_rw, *d_irw;              // N >= 2^10: the twiddles of the row passes' inner radix-16 blocks in the order their
                                    // threads read them, entry (r * 15 + 2^l - 1 + g) * 16 + c = entry
                                    // ((16 (N / 256 + r) + c) << l) + g of d_w / d_iw (nullptr for other ring sizes)
    u64 *d_ninv, *d_ninv_s;         // [prime]
    ModQ *d_modq;                   // [prime]
    double *d_fp;                   // [prime][4]: q, 1/q, 1/N mod q as doubles, 0; q = 0 marks a prime of
                                    // 44 bits or more, which only the integer code paths handle
    u64 *d_imag, *d_imag_s;         // [prime] psi^(N/2) and Shoup quotient
    // scratch owned by the context (single stream use)
    u64 *d_scratch;
    size_t scratch_bytes;
    // staging for the term lists of batched calls: one region per stream that has staged a list (a region has one
    // user at a time: the copy into it and the kernel that reads it are ordered on that stream)
    std::vector<std::pair<hipStream_t, void *>> d_desc;
    hipStream_t stream = nullptr;   // what a null stream argument of an entry point means for this context
    // a second stream (non-blocking, default priority) for the runs of a large transform batch: the odd runs go there,
    // forked from and joined back into the caller's stream with the two events inside the same call.  Made on first
    // use: a process has few hardware queues, and a stream that is never used would still share one with a busy stream
    hipStream_t aux = nullptr;
    hipEvent_t aux_fork = nullptr, aux_join = nullptr;
    // compact evaluation keys: offset of every prime's limb inside a (digit, polynomial) slice and, last entry, the
    // slice size, in units of 2N bytes (a prime below 2^44 takes 6 bytes per residue = 3 units, any other 4)
    std::vector<u32> key_off;
    u32 *d_key_off;
    // Algorithmic bytes of everything launched on this context since the last reset, by kind of work: for each
    // launch the operands it has to read once plus the results it has to write once (what a launch of that kind
    // cannot avoid moving), counted on the host when the launch is queued.  A 2^16-point transform counts one
    // read and one write of every limb although it runs as two launches.
    unsigned long long traffic[8], launches[8];
};
enum { TR_NTT = 0, TR_KEYPROD, TR_BCONV, TR_TENSOR, TR_MASKED, TR_POINTWISE, TR_KINDS };
inline void account(const hemm_context *c, int kind, size_t bytes, int n_launches = 1) {
    hemm_context *m = const_cast<hemm_context *>(c);
    m->traffic[kind] += bytes;
    m->launches[kind] += (unsigned long long)n_launches;
}

// Rings of 2^10 points and more run the register-blocked transforms, whose passes can begin in a basis conversion, end in
// a subtraction and a constant, and read through an automorphism (primes below 2^44 in double precision, twiddle tables
// laid out for it).
inline bool ring_has_fused_forms(const hemm_context *c) { return c->logN >= 10; }
// Whether a transform is one launch with a workgroup per limb: up to 2^12 points always.  A larger limb of 60 bits is slower in
// one workgroup than spread over several in two launches, until the limbs alone fill the CUs and the second trip through memory is
// what counts; one of 42 bits has fewer instructions to spread and gains earlier.  A launch may hold limbs of both, so the lines
// lie where 60-bit ones have crossed over.  Forward, us in one launch / in two:
//   2^13 points, limbs    1          8         48         64        128         768
//     60 bits     10.7/ 7.3  10.9/ 7.5  11.3/10.6  11.5/11.5  12.4/18.5   36.2/45.4
//     42 bits      8.0/ 6.6   8.2/ 6.7   8.5/ 9.5   8.8/10.3   9.4/16.6   27.2/38.0
//   2^14 points, limbs    8         48         64         80         96        128        768
//     60 bits     18.2/ 7.8  19.1/15.2  19.4/17.9  19.6/21.0  19.9/23.7  22.3/28.9  73.5/81.6
//     42 bits     12.4/ 7.0  13.2/13.3  13.6/15.7  13.8/18.5  14.0/20.9  15.1/25.7  55.0/68.6
// (inverse ones of 60 bits cross over a little later: 64 limbs of 2^13 points 12.5/12.0, 80 of 2^14 22.2/22.3; 768 of those 82.7/88.1.)
// plain: no conversion, tail or automorphism -- with them a workgroup of the 1024 threads a limb of 2^14 takes would spill.
inline bool one_launch(const hemm_context *c, size_t limbs, bool plain) {
    return c->logN >= 10 && (c->logN <= 12 || (c->logN == 13 && limbs >= 64) || (c->logN == 14 && plain && limbs >= 96));
}

// a constant and its Shoup quotient floor(w * 2^64 / q)
struct __align__(16) Cst {
    u64 w, ws;
};

// NTT-domain index of the automorphism X -> X^g: out[k] = in[galois_index(k)]
__device__ __forceinline__ u32 galois_index(u32 k, u32 g, int logN) {
    const u32 br = __brev(k) >> (32 - logN);
    const u32 e = ((2 * br + 1) * g) & ((2u << logN) - 1);
    return __brev(e >> 1) >> (32 - logN);
}

void hemm_set_error(const std::string &msg);

// Where a chain over several ciphertexts leaves its results when they do not lie back to back: polynomials 2 i and 2 i + 1 in
// at[i] (a chain's output stride apart).  Travels in the kernel arguments.
#define RESULT_PARTS 32
struct ResultList {
    u64 *at[RESULT_PARTS];
};

#define HEMM_HIP(call)                                                                       \
    do {                                                                                     \
        hipError_t e_ = (call);                                                              \
        if (e_ != hipSuccess)                                                                \
            throw std::runtime_error(std::string(#call) + ": " + hipGetErrorString(e_));     \
    } while (0)

// host modular helpers (context set-up only)
u64 h_mulmod(u64 a, u64 b, u64 q);
u64 h_powmod(u64 a, u64 e, u64 q);
u64 h_invmod(u64 a, u64 q);

LimbList limbs_default(const hemm_context *c, int nq, int with_p);

// kernel launchers (defined in the .hip files)
// final_scale (device, one (constant, Shoup quotient) pair per limb of the launch, or nullptr): an inverse transform
// of N >= 2^10 ends with that constant in place of 1/N
void launch_ntt_slots(const hemm_context *c, u64 *data, const LimbList &ll, const LimbList &sl, int n_limbs,
                      int n_polys, size_t poly_stride, bool inverse, hipStream_t s, const void *final_scale = nullptr);
bool launch_ntt_sub_scale(const hemm_context *c, u64 *data, int n_limbs, int n_polys, const u64 *minuend,
                          size_t minuend_stride, u64 *out, size_t out_stride, const void *cst_dev, hipStream_t s,
                          const ResultList *list = nullptr);
// A forward transform of N >= 2^10 whose input is a fast basis conversion: limb l of the launch is the conversion of
// the coefficient-form sources of digit digit_of[l] (already carrying their (S/q_i)^-1 factors) to prime ll[l],
// computed while the first pass loads its slab instead of being written by a conversion launch and read back.
#define CONV_MAX_DIGITS 4
#define CONV_MAX_SOURCES 8
struct ConvSources {
    struct Digit {
        const u64 *src;             // coefficient form, [n_polys][.][N]
        const Cst *hat;             // [n_src][hat_ld]  (S/q_i) mod prime and 2^30 times that, indexed by prime
        size_t src_poly_stride;
        int n_src;
        uint8_t src_slot[CONV_MAX_SOURCES];
    } d[CONV_MAX_DIGITS];
    int hat_ld;
    uint8_t digit_of[HEMM_MAX_PRIMES];
    // n_copy further limbs of the launch are plain copies (first pass only, no transform): slot copy_src_slot[i] of
    // copy_src (NTT form, polynomial stride copy_src_stride) to slot copy_dst_slot[i] of data
    const u64 *copy_src;
    size_t copy_src_stride;
    int n_copy;
    u32 copy_galois;            // != 0: the copies read their source through this automorphism
    uint8_t copy_src_slot[HEMM_MAX_PRIMES], copy_dst_slot[HEMM_MAX_PRIMES];
};
// data: [n_polys][.][N] (polynomial stride poly_stride), limb l written to slot sl[l].  With ep_* set the second pass
// ends with out = (minuend - transform) * cst[l] (slots of minuend / out = l) and data is only a workspace; ep_list: the
// polynomials of `out` lie where the list says.  cols_only: the first of two passes, left in data.
// false when the ring size or the source counts have no such form (nothing was launched).
bool launch_ntt_converted(const hemm_context *c, const ConvSources &cs, u64 *data, const LimbList &ll, const LimbList &sl,
                          int n_limbs, int n_polys, size_t poly_stride, hipStream_t s, const u64 *ep_minuend = nullptr,
                          size_t ep_minuend_stride = 0, u64 *ep_out = nullptr, size_t ep_out_stride = 0,
                          const void *ep_cst_dev = nullptr, const ResultList *ep_list = nullptr, bool cols_only = false);
// A forward transform of N >= 2^10 whose input is the rounded coefficients of an encoding (signed, [n_polys][stride >= N], the
// same for every limb; plus, with_error, the error of a stream), reduced while the first pass loads them.  enc: the second
// pass ends in an encryption instead of storing the transform (data is then only a workspace): a uniform from the streams
// sm64(sm64(a_base + prime)), b = transform - a s, b and a laid out like data, sk [prime][N].  false: no such form.
struct LiftSource {
    const long long *coef;
    size_t stride;
    u64 error_key;
    int with_error;
};
struct EncryptTail {
    u64 *b, *a;
    const u64 *sk;
    u64 a_base;
};
bool launch_ntt_lifted(const hemm_context *c, const LiftSource &ls, u64 *data, const LimbList &ll, int n_limbs, int n_polys,
                       size_t poly_stride, hipStream_t s, const EncryptTail *enc);
// data[j] = inverse transform of b[j] + a[j] s for the first n_limbs chain primes (all [n_limbs][N])
bool launch_intt_decrypt(const hemm_context *c, const u64 *b, const u64 *a, const u64 *sk, u64 *data, int n_limbs, hipStream_t s);
// slots: [n_msgs][N/2] complex doubles, or re: the real parts of the first `count` slots of one message, in device memory or
// in host memory the device reads; work: [n_msgs][N] words, may be `slots`; out: [n_msgs][n_limbs][N], with enc a
// workspace (which may be enc->b).  re and enc need N >= 2^10.
void launch_encode(const hemm_context *c, const double *slots, const double *re, size_t count, double scale, const LimbList &ll,
                   int n_limbs, int n_msgs, u64 *work, u64 *out, hipStream_t s, const EncryptTail *enc = nullptr,
                   u64 error_key = 0);
// pt: [>= n_limbs][N]; a != nullptr: pt is the first polynomial of a ciphertext, a its second.  slots: [N/2] complex doubles; re
// != nullptr: slots is a workspace and the real parts of the first `count` slots go to re.  a and re need N >= 2^10.
void launch_decode(const hemm_context *c, const u64 *pt, const u64 *a, const u64 *sk, int n_limbs, double scale, u64 *work,
                   double *slots, double *re, size_t count, hipStream_t s);
// out[p][j] = (y[p][j] - conversion of the n_src listed limbs of y[p] to chain prime j) * cst[j], j < nq_out, as inverse row
// pass (in place on the listed limbs; rows_done: it has run), one column-slab kernel (second inverse pass, conversion as lazy dot
// products, first forward pass into conv[n_polys][nq_out][N]) and forward row pass with the fused tail (not with cols_only).  final_scale
// / hat / cst: device tables in source order, [n_src][hat_ld] by prime (as in ConvSources), by target limb.  list: where the results
// lie, for one run of polynomials.  Primes below 2^60.  false when the shape has no such form (nothing was launched).
bool launch_moddown_slab(const hemm_context *c, u64 *y, size_t y_stride, const uint8_t *src_slot, const uint8_t *src_prime,
                         int n_src, const void *final_scale_dev, const void *hat_dev, int hat_ld, u64 *conv, int nq_out,
                         int n_polys, u64 *out, size_t out_stride, const void *cst_dev, hipStream_t s, const ResultList *list = nullptr,
                         bool rows_done = false, bool cols_only = false);
// whether that form is the faster one (N = 2^16, two to five sources); uncut: with rows_done and cols_only
bool takes_moddown_slab(const hemm_context *c, int n_src, int nq_out, int n_polys, bool uncut);
// inverse transform reading src (same slot numbering as data, polynomial stride src_poly_stride) and leaving the
// coefficients in data; false when this ring size has no out-of-place form (the caller copies, then transforms)
// galois != 0: src is read through that automorphism (the transform of the rotated polynomial, without a launch
// that rotates it first)
bool launch_intt_from(const hemm_context *c, const u64 *src, size_t src_poly_stride, u64 *data, const LimbList &ll,
                      const LimbList &sl, int n_limbs, int n_polys, size_t poly_stride, hipStream_t s,
                      const void *final_scale = nullptr, u32 galois = 0);
// the second pass of an inverse transform of two launches (N >= 2^13), in place
void launch_intt_cols(const hemm_context *c, u64 *data, const LimbList &ll, const LimbList &sl, int n_limbs, int n_polys,
                      size_t poly_stride, hipStream_t s, const void *final_scale);
void launch_ntt(const hemm_context *c, u64 *data, const LimbList &ll, int n_limbs, int n_polys,
                size_t poly_stride, bool inverse, hipStream_t s);
void launch_binary(const hemm_context *c, int op, const u64 *a, size_t a_stride, const u64 *b, size_t b_stride,
                   u64 *out, size_t out_stride, const LimbList &ll, int n_limbs, int n_polys, hipStream_t s);
void launch_mul_scalar(const hemm_context *c, const u64 *a, size_t a_stride, const u64 *scalars, u64 *out,
                       size_t out_stride, const LimbList &ll, int n_limbs, int n_polys, hipStream_t s);
void launch_add_scalar(const hemm_context *c, const u64 *a, const u64 *re, const u64 *im, u64 *out, const LimbList &ll,
                       int n_limbs, hipStream_t s);
void hemm_embedding_tables_free(const hemm_context *c);
void launch_zero(const hemm_context *c, u64 *out, size_t words, hipStream_t s);
void launch_mul_imag(const hemm_context *c, const u64 *a, size_t a_stride, u64 *out, size_t out_stride,
                     const LimbList &ll, int n_limbs, int n_polys, hipStream_t s);
void launch_tensor(const hemm_context *c, const u64 *c1, size_t s1, const u64 *c2, size_t s2, u64 *out,
                   size_t out_stride, int nq, bool accumulate, hipStream_t s);
void launch_galois(const hemm_context *c, const u64 *a, size_t a_stride, u64 *out, size_t out_stride, u64 g,
                   int n_limbs, int n_polys, hipStream_t s);
void launch_sample_uniform(const hemm_context *c, const u64 *stream_keys, const LimbList &ll, int n_limbs, u64 *out,
                           hipStream_t s);
void launch_sample_error(const hemm_context *c, u64 stream_key, const LimbList &ll, int n_limbs, u64 *out, hipStream_t s);
size_t hemm_scratch_words(const hemm_context *c);
u64 *hemm_scratch(hemm_context *c);
void launch_modup(hemm_context *c, const u64 *in, int nq, u64 *ext, u64 *coef, bool fill_own, hipStream_t s);
void launch_inner_product(hemm_context *c, const u64 *in, const u64 *ext, const u64 *evk, int nq, u64 *acc,
                          hipStream_t s);
void launch_moddown(hemm_context *c, u64 *acc, int nq, int n_polys, u64 *out, size_t out_stride, const u64 *add,
                    size_t add_stride, int add_polys, u64 *conv, hipStream_t s);
// galois != 0 (N >= 2^10): the key switch of the automorphism of `in`, which is read through it where the ModUp reads
// it; b_rotates: add_b is read through the same automorphism where the key product adds it; add_a (N >= 512, with
// add_b): out[1] = ks_a + add_a as well, both addends entering the sum in the extended basis
void launch_keyswitch(hemm_context *c, const u64 *in, const u64 *evk, int nq, u64 *out, size_t out_stride,
                      const u64 *add_b, hipStream_t s, u32 galois = 0, bool b_rotates = false,
                      const u64 *add_a = nullptr);
void launch_rescale(hemm_context *c, const u64 *in, size_t in_stride, u64 *out, size_t out_stride, int nq,
                    int n_polys, hipStream_t s, const ResultList *list = nullptr);
void launch_modup_batch(hemm_context *c, const u64 *in, size_t in_stride, int nq, int n_in, u64 *ext, u64 *coef,
                        hipStream_t s, u32 galois = 0);
// whether launch_modup_batch at this level takes a non-zero `galois` (its input read through that automorphism)
bool modup_through_automorphism_ok(const hemm_context *c, int nq);
// A list of rotation terms (merged; RotTermDev) and the offsets of its groups: in host memory, and in device memory as well where it
// is too long for the kernel arguments (terms_dev, then the only copy the kernels read).  All keys in one layout.
struct HoistedList {
    const void *terms;
    const u32 *offsets;
    const void *terms_dev;
    const u32 *offsets_dev;
    int n_terms;
    // a single key switch whose ModUp is not finished: the first term's ext holds the column passes' results only, and the digits' own
    // limbs are those of this polynomial [nq][N] (nullptr: none of that), of its automorphism switched_galois (1: none)
    const u64 *switched;
    u32 switched_galois;
};
int hoisted_arg_capacity();
void launch_hoisted_terms(hemm_context *c, const HoistedList &l, int n_out, int nq, u64 *y, bool b_premultiplied, hipStream_t s);
// outs: the two polynomials of result o at outs[o], out_stride apart (nullptr: back to back at out)
void launch_hoisted_moddown(hemm_context *c, const HoistedList &l, int n_out, int nq, u64 *y, bool b_premultiplied, int drop_last, u64 *out,
                            size_t out_stride, u64 *const *outs, u64 *conv, hipStream_t s);
void launch_moddown_batch(hemm_context *c, u64 *y, int nq, int n_polys, int drop_last, u64 *out, size_t out_stride,
                          u64 *conv, hipStream_t s, bool slab = false, const ResultList *list = nullptr, bool rows_done = false,
                          bool cols_only = false);
void launch_masked_sum(hemm_context *c, const void *terms_dev, const u32 *group_off_dev, int n_out, int nq, int n_polys,
                       u64 *out, hipStream_t s, const void *terms_host, int n_terms);
// y[o][p][j] = sum_{q < parts} part[o * parts + q][p][j] over the extended basis, y / part: [.][2][nq+K][N]
void launch_sum_parts(hemm_context *c, const u64 *part, int parts, int n_out, int nq, u64 *y, hipStream_t s);
size_t key_compact_words(const hemm_context *c);
void launch_key_compact(const hemm_context *c, const u64 *evk, u64 *out, hipStream_t s);
void launch_key_expand(const hemm_context *c, const u64 *compact, u64 *evk, hipStream_t s);
int masked_arg_capacity();
// table[j][r] = mask[j][r << shift]; true when every aligned run of 2^shift residues of the mask is constant
bool launch_compact_mask(hemm_context *c, const u64 *mask, int n_limbs, int shift, u64 *table, hipStream_t s);
// Products with a plaintext matrix over its diagonals (diagonals.hip): k x k tiles, rows of w slots, g baby steps, 2k / g giant ones.
bool diagonals_ok(const hemm_context *c, u32 k, u32 w, u32 g, int nq);
size_t diagonal_table_words(const hemm_context *c, u32 k, u32 w, u32 g, int nq);
// block: the first k rows of the matrix's slots, [k][w] complex doubles
void launch_diagonal_tables(hemm_context *c, const double *block, u32 k, u32 w, u32 g, double scale, int nq, u64 *tables, hipStream_t s);
// l: the g - 1 rotations, one term each; a: the ciphertext itself (chain limbs, polynomials a_stride apart); y: [2k/g][2][nq+K][N]
void launch_diagonal_sums(hemm_context *c, const HoistedList &l, const u64 *a, size_t a_stride, u32 k, u32 w, u32 g, int nq, bool b_premultiplied,
                          const u64 *tables, u64 *y, hipStream_t s);
const void *encode_roots(const hemm_context *c);     // complex roots of an encoding's butterflies (encode.hip)
const Cst *pmod_table(const hemm_context *c);        // P mod q_j for the chain primes, on the device
void launch_masked_sum_args(hemm_context *c, const void *terms_host, int n_terms, const u32 *group_off_host, int n_out,
                            int nq, int n_polys, u64 *out, hipStream_t s);
// several tensor sums in one launch: acc[i] (+)= sum over n_pairs[i] pairs of t1[i], t2[i] (distinct accumulators)
#define TENSOR_MAX_GROUPS 8
struct TensorGroupHost {
    const u64 *t1, *t2;
    u64 *acc;
    int n_pairs;
    bool accumulate;
};
int tensor_max_groups();
void launch_tensor_groups(hemm_context *c, const TensorGroupHost *g, int n_groups, int nq, size_t acc_stride,
                          hipStream_t s);
void launch_tensor_batch(hemm_context *c, const u64 *t1, const u64 *t2, int G, int nq, u64 *acc3, size_t acc_stride,
                         bool accumulate, hipStream_t s);
