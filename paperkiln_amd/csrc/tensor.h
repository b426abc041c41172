// Internal side of the device tensors: the kernel launchers used by the
// host-side tape. The types themselves (Tensor, Buffer, the allocator, the
// tape context) are public and live in include/paperkiln_amd.hpp.
#pragma once
#include <memory>
#include <vector>
#include <hip/hip_runtime.h>

#include "paperkiln_amd.hpp"

namespace pk {

void hip_check(hipError_t e, const char* what);  // throws Error(PK_ERR_HIP), as cuda_check throws (cuda_ops.cu:34-38)

// ---- kernel launchers (elementwise.hip) -----------------------------------
// All take row-major contiguous tensors; T = fp32 or bf16 storage, fp32 math.
void k_fill(const Tensor& y, float v);
void k_cast(const Tensor& src, const Tensor& dst);                      // dtype conversion / copy
void k_cast_cols(const Tensor& src, const Tensor& dst, int64_t col_off);
// many such casts (fp32 -> a column block of a bf16 or fp32 matrix) as one launch; false = not applicable, nothing done
struct CastJob {
    Tensor src, dst;
    int64_t col_off;
};
bool k_cast_many(const std::vector<CastJob>& list);  // dst[:, off:off+src.cols] = src
void k_add(const Tensor& a, const Tensor& b, const Tensor& y);          // y = a + b      (ops.cpp:60-65)
void k_mul(const Tensor& a, const Tensor& b, const Tensor& y);          // y = a .* b     (ops.cpp:76-83)
void k_scale(const Tensor& a, float s, const Tensor& y);                // y = a * s
void k_axpy(const Tensor& y, float a, const Tensor& x);                 // y += a * x     (autograd.cpp:16-24)
void k_silu_fwd(const Tensor& x, const Tensor& y);                      // ops.cpp:404-411
void k_silu_bwd(const Tensor& x, const Tensor& dy, const Tensor& dx);   // ops.cpp:412-423
void k_silu_mul_fwd(const Tensor& gate, const Tensor& up, const Tensor& y);  // silu(gate) .* up, llama.cpp:55-58
void k_silu_mul_bwd(const Tensor& gate, const Tensor& up, const Tensor& dy, const Tensor& dgate, const Tensor& dup);
// the same on the two halves of one [rows, 2*cols] matrix [gate | up]
void k_silu_mul_cat_fwd(const Tensor& gu, const Tensor& y);
void k_silu_mul_cat_bwd(const Tensor& gu, const Tensor& dy, const Tensor& dgu);
void k_rmsnorm_fwd(const Tensor& x, const Tensor& w, float eps, const Tensor& y, float* rinv);  // ops.cpp:437-445
// ops.cpp:447-478; with an addend (dx's shape and type) dx = addend + the gradient through the norm
// With `held`, dw's sum over the workgroups' shares may be left to do (held->part is set then) for k_add_held, which takes many.
struct HeldSum {
    std::shared_ptr<Buffer> part;  // [nparts][cols]
    int nparts = 0, cols = 0;
    float* dw = nullptr;           // dw[c] += sum over the parts
};
void k_rmsnorm_bwd(const Tensor& dy, const Tensor& x, const float* rinv, const Tensor& w, const Tensor* dw_f32,
                   const Tensor* dx, const Tensor* addend = nullptr, HeldSum* held = nullptr);
void k_add_held(const HeldSum* held, int count);  // no two with the same dw
// apply_rope on a fused [N, 3d] matrix (ops.cpp:481-537): rotates adjacent pairs of the
// first `rot_heads` heads of the q third and of the k third; inverse = backward.
void k_rope(const Tensor& x, const int* pos, float theta, int d, int head_dim, int rot_heads, bool inverse,
            const Tensor& y);
void k_rope_inplace(const Tensor& x, const int* pos, float theta, int d, int head_dim, int rot_heads, bool inverse);
// table[p][i] = cosine and sine of position p's angle for pair i of a head, the ones that k_rope forms
void k_rope_table(float theta, int head_dim, int64_t positions, float* table);
// How a product that is a fused [rows, 3 d] projection turns its q and k thirds on the way out; row r has position r % seq_len.
struct Turn {
    const float* table;  // [seq_len or more][head_dim / 2] pairs of k_rope_table
    int seq_len, d, head_dim;
    int cols;  // the first so many columns of the q and of the k third turn
};
void k_embedding_fwd(const Tensor& table_f32, const int* ids, const Tensor& y);       // ops.cpp:329-337
// scatter-add, ops.cpp:338-347; held sums (no two with the same dw) may ride along: true if they did
bool k_embedding_bwd(const Tensor& dy, const int* ids, const Tensor& dtable_f32, const HeldSum* held = nullptr, int count = 0);
// Whether n rows of d columns go without the sort, by workgroups that look through all ids. For tests.
extern "C" int pk_embedding_scans(int64_t n, int64_t d);
// Row-wise softmax cross-entropy on a block of logits (ops.cpp:350-376): writes
// dlogits = (P - onehot) * gscale in place and the per-row nll (fp32) with the
// reference's max(p, 1e-12) clamp.
void k_ce_rows(const Tensor& logits, const int* targets, float gscale, float* nll_rows);
// The same on fp32 logits that are read once and left untouched: dl == nullptr computes only the nll, otherwise
// dlogits go to *dl (fp32 or bf16). Returns false when the shape does not fit (the caller then uses k_ce_rows).
bool k_ce_rows_once(const Tensor& logits, const int* targets, float gscale, float* nll_rows, const Tensor* dl,
                    int64_t dl_ld = 0);  // dl_ld: row pitch of dl in its own elements (0 = cols)
double k_sum_f32_to_host(const float* x, int64_t n);                   // double accumulation, ops.cpp:360-367
// the same sum / n into a [1,1] float, no host round trip; if given, a 1 into another and the mean to pinned host memory
void k_mean_f32(const float* x, int64_t n, const Tensor& out, const Tensor* one = nullptr, float* pinned = nullptr);
double k_sumsq_to_host(const Tensor& g);                               // clip_grad_norm's sum, ops.cpp:1046-1052
// The same in two halves, so that many gradients cost one host round trip: per-block partial sums (at most
// SUMSQ_MAX_PARTS doubles) into device memory, then one copy and a host sum over all of them.
constexpr int SUMSQ_MAX_PARTS = 1024;
int k_sumsq_parts(const Tensor& g, double* part_dev);
double k_sum_f64_to_host(const double* part_dev, int64_t n);
// What ops::clip_grad_norm multiplies the gradients by (1 where the norm is within max_norm), from those partial sums,
// left on the device for k_adamw; the norm itself goes to pinned host memory, to be read after a wait for the stream.
void k_clip_factor(const double* part_dev, int n, float max_norm, float* factor_dev, float* norm_pinned);
// the same asked for with the optimiser step; factor: room for it
struct Clip {
    const double* part_dev = nullptr;  // null: no clip
    int n = 0;
    float max_norm = 0.0f;
    float* factor = nullptr;
    float* norm_pinned = nullptr;
};
// clear = 0 (fp32), to[i] = pinned[i]; for a batch of few tokens with y = table[pinned[0 .. y.rows - 1]] in the same launch: true if so
bool k_begin_pass(const Tensor& clear, const int* pinned, int* to, int64_t n, const Tensor& table, const Tensor& y);
void k_word_to_pinned(const void* src, void* pinned);  // one float for the host, cheaper than a copy
// clip_dev (may be null): g is scaled in place by *clip_dev first, in the same pass
void k_adamw(const Tensor& p, const Tensor& g, const Tensor& m, const Tensor& v, float lr, float b1, float b2,
             float eps, float wd, float c1, float c2, const float* clip_dev = nullptr);         // nn.cpp:301-321
// The same over parts of the slabs, each of which may have a copy that is written with it: element e of the part to column
// col_off + e % cols of row e / cols. False, with nothing done, for parts that are not whole groups of four.
struct AdamWPart {
    int64_t at, count, cols;
    Tensor copy;
    int64_t col_off;
};
bool k_adamw_parts(const Tensor& p, const Tensor& g, const Tensor& m, const Tensor& v, const std::vector<AdamWPart>& parts, float lr,
                   float b1, float b2, float eps, float wd, float c1, float c2, const Clip& clip);

// How a product of x's normalised rows forms them itself (k_rmsnorm_fwd): x comes as it is, w [K] goes into it, 1 / rms of a row into the
// sums. The normalised rows (x's type) go to y and 1 / rms to rinv, where a backward pass will ask for them; both may be null.
struct Norm {
    const float* w;
    float eps;
    void* y;
    float* rinv;
};

// C[M,N] (+)= op(A) . op(B), row-major, bf16 or fp32 operands, fp32 accumulate
// (device::gemm, src/device.cpp:91-125). C may be a column slice of a wider
// matrix (ldc). beta is 0 or 1.
void gemm(const Tensor& A, bool tA, const Tensor& B, bool tB, void* C, int c_dtype, int64_t M, int64_t N, int64_t ldc,
          float beta, int64_t lda = 0);
// gemm_mfma.hip: the hand-written bf16 matrix-core GEMM. Returns false (nothing done) for operands it does not take.
// With an addend (C's type and row pitch; beta must be 1) C = addend + op(A) op(B), the sum rounded once.
bool gemm_mfma_bf16(const void* a, bool tA, int64_t lda, const void* b, bool tB, int64_t ldb, void* c, int c_dtype,
                    int64_t M, int64_t N, int64_t K, int64_t ldc, float beta, hipStream_t st, const void* addend = nullptr);
// The same product left as fp32 partial products part[s][M][N], s < nparts (the contraction cut into slices where the
// output alone would leave the chip idle), for a caller that adds them on the way to where the result goes.
bool gemm_mfma_bf16_parts(const void* a, bool tA, int64_t lda, const void* b, bool tB, int64_t ldb, int64_t M, int64_t N,
                          int64_t K, hipStream_t st, std::unique_ptr<Buffer>& part, int& nparts);
// The tied head's cross-entropy inside its logits product A B^T (bf16 [M, K] and [N, K]): the logits are formed tile
// by tile, twice, and never stored. gemm_head_rows: per row the maximum, 1 / sum exp(z - maximum) and the loss
// (stats: scratch of gemm_head_spans(M, N) * M float pairs, zt: of M floats); gemm_head_dlogits: bf16 dlogits, of which the
// columns from `vocab` on are 0 (N is the vocabulary padded to a multiple of 8, in the rows of b as well).
// Both return false, having done nothing, for operands the kernel does not take.
// Several weight-gradient products C_p += A_p^T B_p (A_p [K, M_p], B_p [K, N_p] bf16; C_p [M_p, N_p] fp32) that share
// the contraction length, as one launch of the hand-written kernel. False, with nothing done, where that does not
// apply (operands it does not take, too few tiles): the caller multiplies them one by one.
struct GroupedProduct {
    const void* a;
    int64_t lda;
    const void* b;
    int64_t ldb;
    float* c;
    int64_t ldc;
    int64_t M, N;
};
bool gemm_mfma_grouped_tn(const GroupedProduct* ps, int count, int64_t K, hipStream_t st);
// gemm_small.hip: C_p = op(A_p) op(B_p) + (addend_p, or C_p if beta is 1), bf16 operands, C of c_dtype, for up to eight
// products of one orientation in one launch; for sizes where tiles of 128 x 128 are few. False, with nothing done, for
// operands it does not take (odd pitches or sizes, both transposed, a contraction below 32, a gigabyte or more).
struct SmallProduct {
    const void* a;
    int64_t lda;
    const void* b;
    int64_t ldb;
    void* c;
    int64_t ldc;
    const void* addend;  // C's type and row pitch; may be null
    int64_t M, N, K;
};
bool gemm_small(const SmallProduct* ps, int count, bool tA, bool tB, int c_dtype, float beta, hipStream_t st);
bool gemm_small_is_ahead(bool tA, bool tB, int64_t M, int64_t N, int64_t K);  // of gemm_mfma.hip's tiles, for one product
double gemm_small_us(bool tA, bool tB, int64_t tiles, int64_t K);               // tiles of 32 x 32, of all products together
// gemm_f32.hip: C_p = op(A_p) op(B_p) + (addend_p, or C_p if beta is 1) for up to eight products of one orientation in one
// launch, fp32 throughout on the matrix cores; any sizes and row pitches. False, with nothing done, if A and B are both
// transposed or an operand has 2 GiB or more.
struct F32Product {
    const float* a;
    int64_t lda;
    const float* b;
    int64_t ldb;
    float* c;
    int64_t ldc;
    const float* addend;  // row pitch ldc; may be null
    int64_t M, N, K;
};
bool gemm_f32(const F32Product* ps, int count, bool tA, bool tB, float beta, hipStream_t st);
bool gemm_f32_is_ahead(bool tA, int64_t M, int64_t N, int64_t K);  // of the library, for one product of this size
bool gemm_f32_held_is_ahead(int64_t M, int64_t N, int64_t K);      // the same for a weight gradient among several
// SwiGLU inside the products beside it, row-major without gaps. *_gated: h [M, N] = silu(x gate) .* (x up) for x [M, K] and
// w = [gate | up] [K, 2 N], and [x gate | x up] to gu unless that is null. *_gated_grad: d = dy w^T (dy [M, K], w [N, K]) is
// the gradient of silu(gate) .* up; that of gu = [gate | up] goes to dgu. False, with nothing done, for what they do not take.
bool gemm_f32_gated(const float* x, const float* w, float* gu, float* h, int64_t M, int64_t N, int64_t K, hipStream_t st, const Norm* norm = nullptr);
bool gemm_f32_gated_grad(const float* dy, const float* w, const float* gu, float* dgu, int64_t M, int64_t N, int64_t K, hipStream_t st);
bool gemm_small_gated(const void* x, const void* w, void* gu, void* h, int64_t M, int64_t N, int64_t K, hipStream_t st, const Norm* norm = nullptr);
bool gemm_small_gated_grad(const void* dy, const void* w, const void* gu, void* dgu, int64_t M, int64_t N, int64_t K, hipStream_t st);
bool gemm_mfma_gated(const void* x, const void* w, void* gu, void* h, int64_t M, int64_t N, int64_t K, hipStream_t st, const Norm* norm = nullptr);
bool gemm_mfma_gated_grad(const void* dy, const void* w, const void* gu, void* dgu, int64_t M, int64_t N, int64_t K, hipStream_t st);
// y [M, 3 d] = x w (x [M, K], w [K, 3 d], row-major without gaps) with q and k turned, y of the operands' type. False, with nothing
// done, for what they do not take.
bool gemm_f32_turned(const float* x, const float* w, float* y, int64_t M, int64_t K, const Turn& turn, hipStream_t st, const Norm* norm = nullptr);
bool gemm_small_turned(const void* x, const void* w, void* y, int64_t M, int64_t K, const Turn& turn, hipStream_t st, const Norm* norm = nullptr);
bool gemm_mfma_turned(const void* x, const void* w, void* y, int64_t M, int64_t K, const Turn& turn, hipStream_t st, const Norm* norm = nullptr);
int64_t gemm_head_spans(int64_t M, int64_t N);
bool gemm_head_takes(const void* a, int64_t lda, const void* b, int64_t ldb, int64_t M, int64_t N, int64_t K);
bool gemm_head_rows(const void* a, int64_t lda, const void* b, int64_t ldb, int64_t M, int64_t N, int64_t K, const int* target,
                    void* stats, float* zt, float* row_max, float* row_inv, float* nll, hipStream_t st);
bool gemm_head_dlogits(const void* a, int64_t lda, const void* b, int64_t ldb, int64_t M, int64_t N, int64_t K,
                       int64_t vocab, const int* target, const float* row_max, const float* row_inv, float gscale, void* dl,
                       int64_t ldc, hipStream_t st);
// Which GEMM serves bf16 operands: 1 (default) and 2 = the hand-written kernel for everything it takes (1 also
// groups a backward pass's weight-gradient products into shared launches), 0 = the library only. Set from the environment
// (PK_GEMM=library) or by a caller that wants to compare them.
void set_gemm_backend(int hand_written);
void gemm_mfma_force_tiles(int which);  // -1: by shape (default); 0, 1, 5 .. 11: one kernel form always (measurement)
int gemm_backend();
// How the chunked tied head forms its cross-entropy from bf16 operands: 1 (default) = inside the logits product
// (gemm_head_rows / gemm_head_dlogits: no logits in memory), 0 = a logits product into fp32 and a row kernel over it.
void set_head_kernel(int in_product);
int head_kernel();
// dst[k] ([A.cols, B.cols/nsplit] fp32, contiguous) = beta * dst[k] + A^T B[:, k-th column block], k < nsplit <= 4
void gemm_tn_split(const Tensor& A, const Tensor& B, float* const* dst, int nsplit, float beta);

}  // namespace pk
