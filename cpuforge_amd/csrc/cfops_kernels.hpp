// Internal launch interface of the layer-op kernels (layer_ops.hip) used by
// the C ABI in cfops_capi.cpp.  All pointers are device memory, f32 unless
// stated, row-major and contiguous.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace cfattn {

// RMSNorm (crates/core/src/ops/rmsnorm.rs:4-67).  Forward overwrites y and
// rstd.  Backward adds to (acc) or overwrites dx and, when non-null, dw; it
// needs `partial` scratch of rmsnorm_bwd_partial_floats(rows, dim) floats.
hipError_t launch_rmsnorm_fwd(const float* x, const float* w, float* y, float* rstd, size_t rows, size_t dim, float eps,
                              hipStream_t st);
size_t rmsnorm_bwd_partial_floats(size_t rows, size_t dim);
hipError_t launch_rmsnorm_bwd(const float* dy, const float* x, const float* w, const float* rstd, float* dx, float* dw,
                              float* partial, size_t rows, size_t dim, int acc, hipStream_t st);

// SwiGLU gate (crates/core/src/ops/swiglu.rs:10-30): forward overwrites h,
// backward adds to (acc) or overwrites dg and du.
hipError_t launch_silu_mul_fwd(const float* g, const float* u, float* h, size_t n, hipStream_t st);
hipError_t launch_silu_mul_bwd(const float* dh, const float* g, const float* u, float* dg, float* du, size_t n, int acc,
                               hipStream_t st);

// Cross-entropy with its gradient (crates/core/src/ops/loss.rs:9-55), in three
// launches over a `misc` block of kCeMiscBytes (valid-row count, first bad
// row, loss) and `row_loss` scratch of `rows` floats:
//   ce_begin:  count the rows to score, reset the bad-row marker;
//   ce_rows:   rows [row0, row0 + nrows): `logits` and `dlogits` point at
//              row row0 (dlogits may alias logits: each row is read before it
//              is written), targets and row_loss are indexed from row 0; a
//              target outside [0, vocab) marks its row as bad;
//   ce_finish: the mean loss, summed in f64 in row order.
constexpr size_t kCeMiscBytes = 256;
struct CeMisc {
    int n_valid;
    int bad_row;  // first row with a target out of range, or INT_MAX
    float loss;
};
hipError_t launch_ce_begin(const int64_t* targets, size_t rows, void* misc, hipStream_t st);
hipError_t launch_ce_rows(const float* logits, const int64_t* targets, float* dlogits, float* row_loss, size_t row0,
                          size_t nrows, size_t vocab, void* misc, hipStream_t st);
hipError_t launch_ce_finish(const int64_t* targets, const float* row_loss, size_t rows, void* misc, hipStream_t st);

// One AdamW update (crates/train/src/optim.rs:9-30) of `count` tensors, none
// empty; bc1, bc2 are the bias corrections 1 - beta^t, computed by the caller.
constexpr int kAdamwBatch = 64;
struct AdamwTensor {
    float* p;
    const float* g;
    float *m, *v;
    long n;
    float weight_decay;
    int vec;      // set by launch_adamw, as block0
    long block0;
};
struct AdamwArgs {
    AdamwTensor t[kAdamwBatch];
    int count;
    float lr, beta1, beta2, eps, bc1, bc2;
};
hipError_t launch_adamw(AdamwArgs a, hipStream_t st);

// f32 GEMMs over a common row count m (gemm_f32.hip).  Problem i is
//   C_i[m, n_i] (+)= sum over its segments s of A_s B_s,
// the segments being runs of one long contraction (a base product and an
// adapter's, or the products of several linears into one gradient).  A
// element (row, k) is at a[row * lda + k], or a[k * lda + row] with
// a_strided; B element (k, col) at b[col * ldb + k], or b[k * ldb + col] with
// b_strided.  No operand needs more than its natural alignment.
constexpr int kGemmSegs = 8, kGemmProblems = 4;
struct GemmSeg {
    const float *a, *b;
    long lda, ldb;
    int k;
};
struct GemmProblem {
    GemmSeg seg[kGemmSegs];
    int nseg = 0;
    float* c = nullptr;
    int n = 0;
    float scale = 1.0f;  // of the sum (launch_gemm_rows only)
};
struct GemmF32 {
    GemmProblem pr[kGemmProblems];
    int npr = 0, m = 0;
    int acc = 0;  // 1: add to C, 0: overwrite it
    bool a_strided = false, b_strided = false;
};
// `ws` is scratch for the partial sums of a split contraction.
hipError_t launch_gemm_f32(const GemmF32& g, float* ws, size_t ws_floats, hipStream_t st);
// The same products on the f32 MFMA, a workgroup to 16 rows and 16 columns, for
// a_strided = false: an adapter's products with its rank as n, and those of few
// rows, which launch_gemm_f32 passes on.
hipError_t launch_gemm_rows(const GemmF32& g, hipStream_t st);

// The gradients of LoRA adapters in Linear::backward (linear.rs:75-90), for up
// to kGemmProblems linears over the same t tokens in one launch (lora.hip):
//   out (+)= big^T small, [ncol x r] (gb from dy and xs), or its transpose
//   [r x ncol] (ga from x and dxa).
struct LoraGradJob {
    const float *big, *small;
    float* out;
    int ncol, r, transposed;
    long off;  // of its partial sums (set by lora_grad_plan)
};
struct LoraGrad {
    LoraGradJob job[2 * kGemmProblems];
    int njobs = 0, t = 0, acc = 1;
    int chunks, tokens;     // set by lora_grad_plan
    float* part = nullptr;  // scratch of as many floats as lora_grad_plan returns
};
size_t lora_grad_plan(LoraGrad& g);
hipError_t launch_lora_grad(const LoraGrad& g, hipStream_t st);

}  // namespace cfattn
