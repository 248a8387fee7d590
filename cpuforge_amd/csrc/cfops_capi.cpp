// C ABI of the layer ops (declared in include/cfops.h).
//
// Host-side plumbing only: argument checks, scratch from the context's pool
// and dispatch to the gfx950 kernels of gemm_f32.hip, lora.hip and
// layer_ops.hip.  There is no CPU compute path.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstddef>
#include <cstdint>
#include <cstring>

#include "cfattn_ctx.hpp"
#include "cfops.h"
#include "cfops_kernels.hpp"

namespace {

using namespace cfcapi;

hipStream_t to_stream(void* st) { return static_cast<hipStream_t>(st); }

// Scratch of a GEMM that splits its contraction (partial products).
constexpr size_t kGemmWorkspace = (size_t)32 << 20;

bool fits_int(size_t x) { return x <= (size_t)INT_MAX; }

int launch_gemm(cfattn_ctx* c, const cfattn::GemmF32& g, hipStream_t st) {
    int rc = CFATTN_OK;
    float* ws = static_cast<float*>(slot(c, cfattn_ctx::OPS_WS, kGemmWorkspace, &rc));
    if (!ws) return rc;
    CF_HIP(c, cfattn::launch_gemm_f32(g, ws, kGemmWorkspace / sizeof(float), st), "GEMM launch");
    return CFATTN_OK;
}

// An overwritten gradient of a call without rows: the empty sum.
int zero_grad(cfattn_ctx* c, float* g, size_t n, hipStream_t st) {
    if (g && n) CF_HIP(c, cfattn::launch_fill_zero(g, n, st), "zero-fill launch");
    return CFATTN_OK;
}

// Row-major C[m,n] = op(A) op(B) (+ C when acc), as matmul.rs's
// matmul_nn / matmul_nt / matmul_tn (core/src/matmul.rs:127-147).
int gemm(cfattn_ctx* c, int kind, const float* a, const float* b, float* out, size_t m, size_t k, size_t n, bool acc,
         hipStream_t st) {
    if (m == 0 || n == 0) return CFATTN_OK;
    if (!fits_int(m) || !fits_int(n) || !fits_int(k))
        return fail(c, CFATTN_ERR_UNSUPPORTED, "GEMM dimension above 2^31 (m=%zu, k=%zu, n=%zu)", m, k, n);
    if (k == 0) {  // matmul.rs:58-67: zero C unless accumulating
        if (!acc) CF_HIP(c, cfattn::launch_fill_zero(out, m * n, st), "zero-fill launch");
        return CFATTN_OK;
    }
    if (kind != CFOPS_NN && kind != CFOPS_NT && kind != CFOPS_TN)
        return fail(c, CFATTN_ERR_ARG, "unknown matmul kind %d", kind);
    cfattn::GemmF32 g;
    g.npr = 1, g.m = (int)m, g.acc = acc;
    g.a_strided = kind == CFOPS_TN, g.b_strided = kind != CFOPS_NT;
    g.pr[0].nseg = 1, g.pr[0].c = out, g.pr[0].n = (int)n;
    g.pr[0].seg[0] = {a, b, (long)(kind == CFOPS_TN ? m : k), (long)(kind == CFOPS_NT ? k : n), (int)k};
    return launch_gemm(c, g, st);
}

// Whether a buffer that one tensor's update writes shares memory with any of
// another's (a parameter under two names, or beside a view of itself).
bool adamw_overlaps(const cfattn::AdamwArgs& a) {
    struct Range {
        uintptr_t lo, hi;
        bool written;
    } r[4 * cfattn::kAdamwBatch];
    int n = 0;
    for (int i = 0; i < a.count; i++) {
        const cfattn::AdamwTensor& t = a.t[i];
        const float* const ptr[4] = {t.p, t.m, t.v, t.g};
        for (int j = 0; j < 4; j++) {
            const uintptr_t lo = reinterpret_cast<uintptr_t>(ptr[j]);
            r[n++] = {lo, lo + (size_t)t.n * sizeof(float), j < 3};
        }
    }
    std::sort(r, r + n, [](const Range& x, const Range& y) { return x.lo < y.lo; });
    uintptr_t end = 0, end_written = 0;
    for (int i = 0; i < n; i++) {
        if (r[i].lo < (r[i].written ? end : end_written)) return true;
        end = std::max(end, r[i].hi);
        if (r[i].written) end_written = std::max(end_written, r[i].hi);
    }
    return false;
}

int check_linears(cfattn_ctx* c, size_t t, size_t in, const cfops_linear* lin, size_t n) {
    if (!fits_int(t) || !fits_int(in)) return fail(c, CFATTN_ERR_UNSUPPORTED, "t=%zu, in=%zu above 2^31", t, in);
    for (size_t i = 0; i < n; i++)
        if (!fits_int(lin[i].out) || (lin[i].lora_a && !fits_int(lin[i].rank)))
            return fail(c, CFATTN_ERR_UNSUPPORTED, "out=%zu, rank=%zu above 2^31", lin[i].out, lin[i].rank);
    return CFATTN_OK;
}

// Linear::forward (linear.rs:58-69) of up to kGemmProblems linears of one
// input: xs_i = scale_i x A_i^T in one launch, then y_i = [x xs_i] [W_i B_i]^T in one.
int linears_forward(cfattn_ctx* c, const float* x, size_t t, size_t in, const cfops_linear* lin, size_t n,
                    hipStream_t st) {
    cfattn::GemmF32 g, down;
    down.m = g.m = (int)t;
    for (size_t i = 0; i < n; i++) {
        const cfops_linear& l = lin[i];
        if (l.lora_a) {
            cfattn::GemmProblem& p = down.pr[down.npr++];
            p.seg[p.nseg++] = {x, l.lora_a, (long)in, (long)in, (int)in};
            p.c = l.xs, p.n = (int)l.rank, p.scale = l.lora_scale;
        }
        if (l.out == 0) continue;
        cfattn::GemmProblem& p = g.pr[g.npr++];
        p.c = l.y, p.n = (int)l.out;
        p.seg[p.nseg++] = {x, l.w, (long)in, (long)in, (int)in};
        if (l.lora_a) p.seg[p.nseg++] = {l.xs, l.lora_b, (long)l.rank, (long)l.rank, (int)l.rank};
    }
    CF_HIP(c, cfattn::launch_gemm_rows(down, st), "GEMM launch");
    return g.npr ? launch_gemm(c, g, st) : CFATTN_OK;
}

// Linear::backward (linear.rs:75-90) of up to kGemmProblems linears of one
// input: dxa_i = scale_i dy_i B_i in one launch; dx (+)= [dy_1 dxa_1 dy_2 ..]
// [W_1; A_1; W_2; ..] in one; the adapters' gradients in two.
int linears_backward(cfattn_ctx* c, const float* x, size_t t, size_t in, float* dx, const cfops_linear* lin, size_t n,
                     bool acc_dx, bool acc, hipStream_t st) {
    cfattn::GemmF32 g, down;
    cfattn::LoraGrad lg;
    int rc = CFATTN_OK;
    size_t dxa_floats = 0;
    for (size_t i = 0; i < n; i++) dxa_floats += lin[i].lora_a ? t * lin[i].rank : 0;
    float* dxa = nullptr;
    if (dxa_floats) {
        dxa = static_cast<float*>(slot(c, cfattn_ctx::OPS_DXA, dxa_floats * sizeof(float), &rc));
        if (!dxa) return rc;
    }
    down.m = g.m = lg.t = (int)t;
    down.b_strided = g.b_strided = true, g.acc = acc_dx, lg.acc = acc;
    g.npr = 1, g.pr[0].c = dx, g.pr[0].n = (int)in;
    for (size_t i = 0; i < n; i++) {
        const cfops_linear& l = lin[i];
        cfattn::GemmSeg* seg = g.pr[0].seg;
        seg[g.pr[0].nseg++] = {l.dy, l.w, (long)l.out, (long)in, (int)l.out};
        if (!l.lora_a) continue;
        if (dx || l.ga) {
            cfattn::GemmProblem& p = down.pr[down.npr++];
            p.seg[p.nseg++] = {l.dy, l.lora_b, (long)l.out, (long)l.rank, (int)l.out};
            p.c = dxa, p.n = (int)l.rank, p.scale = l.lora_scale;
            seg[g.pr[0].nseg++] = {dxa, l.lora_a, (long)l.rank, (long)in, (int)l.rank};
        }
        if (l.gb && l.out) lg.job[lg.njobs++] = {l.dy, l.xs, l.gb, (int)l.out, (int)l.rank, 0, 0};
        if (l.ga && in) lg.job[lg.njobs++] = {x, dxa, l.ga, (int)in, (int)l.rank, 1, 0};
        dxa += t * l.rank;
    }
    CF_HIP(c, cfattn::launch_gemm_rows(down, st), "GEMM launch");
    if (dx && in) CF_TRY(launch_gemm(c, g, st));
    for (size_t i = 0; i < n; i++)
        if (lin[i].gw) CF_TRY(gemm(c, CFOPS_TN, lin[i].dy, x, lin[i].gw, lin[i].out, t, in, acc, st));
    if (lg.njobs == 0) return CFATTN_OK;
    lg.part = static_cast<float*>(
        slot(c, cfattn_ctx::OPS_LORA, cfattn::lora_grad_plan(lg) * sizeof(float), &rc));
    if (!lg.part) return rc;
    CF_HIP(c, cfattn::launch_lora_grad(lg, st), "lora launch");
    return CFATTN_OK;
}

// Rust's f32::powi at run time (compiler-rt __powisf2): square-and-multiply
// from the low bit of the exponent, reciprocal for a negative one.
float powi_f32(float a, int b) {
    const bool recip = b < 0;
    unsigned int e = recip ? (unsigned int)(-(long)b) : (unsigned int)b;
    float r = 1.0f;
    for (;;) {
        if (e & 1u) r *= a;
        e >>= 1;
        if (e == 0) break;
        a *= a;
    }
    return recip ? 1.0f / r : r;
}

// Reads the loss block after the stream has drained; reports a target out
// of range as the reference's panic message.
int ce_result(cfattn_ctx* c, const void* misc, const int64_t* targets, size_t vocab, float* loss, hipStream_t st) {
    cfattn::CeMisc m{};
    CF_HIP(c, hipMemcpyAsync(&m, misc, sizeof m, hipMemcpyDeviceToHost, st), "hipMemcpyAsync D2H loss");
    CF_HIP(c, hipStreamSynchronize(st), "cross-entropy");
    if (m.bad_row != INT_MAX) {
        int64_t t = 0;
        CF_HIP(c, hipMemcpy(&t, targets + m.bad_row, sizeof t, hipMemcpyDeviceToHost), "hipMemcpy D2H target");
        return fail(c, CFATTN_ERR_ARG, "target %lld out of range for vocab %zu", (long long)t, vocab);
    }
    *loss = m.loss;
    return CFATTN_OK;
}

#define CF_LOCK(c, stream)                                                                  \
    if (!(c)) return CFATTN_ERR_ARG;                                                      \
    std::lock_guard<std::mutex> lk((c)->mu);                                              \
    (c)->err.clear();                                                                     \
    DeviceGuard dev_guard_((c)->device);                                                  \
    if (!dev_guard_.ok) return fail((c), CFATTN_ERR_HIP, "hipSetDevice(%d) failed", (c)->device); \
    note_capture((c), to_stream(stream))

}  // namespace

extern "C" {

int cfops_matmul(cfattn_ctx* c, int kind, const float* a, const float* b, float* out, size_t m, size_t k, size_t n,
                 int acc, void* stream) {
    CF_LOCK(c, stream);
    if ((m && n && !out) || (m && n && k && (!a || !b))) return fail(c, CFATTN_ERR_ARG, "null buffer");
    return gemm(c, kind, a, b, out, m, k, n, acc != 0, to_stream(stream));
}

int cfops_rmsnorm_forward(cfattn_ctx* c, const float* x, const float* w, float* y, float* rstd, size_t rows,
                          size_t dim, float eps, void* stream) {
    CF_LOCK(c, stream);
    if (rows == 0 || dim == 0) return CFATTN_OK;
    if (!x || !w || !y || !rstd) return fail(c, CFATTN_ERR_ARG, "null buffer");
    if (!fits_int(dim)) return fail(c, CFATTN_ERR_UNSUPPORTED, "dim=%zu above 2^31", dim);
    CF_HIP(c, cfattn::launch_rmsnorm_fwd(x, w, y, rstd, rows, dim, eps, to_stream(stream)), "rmsnorm forward launch");
    return CFATTN_OK;
}

int cfops_rmsnorm_backward(cfattn_ctx* c, const float* dy, const float* x, const float* w, const float* rstd,
                           float* dx, float* dw, size_t rows, size_t dim, void* stream) {
    return cfops_rmsnorm_grad(c, dy, x, w, rstd, dx, dw, rows, dim, 1, stream);
}

int cfops_rmsnorm_grad(cfattn_ctx* c, const float* dy, const float* x, const float* w, const float* rstd, float* dx,
                       float* dw, size_t rows, size_t dim, int acc, void* stream) {
    CF_LOCK(c, stream);
    if (rows == 0 && !acc) return zero_grad(c, dw, dim, to_stream(stream));
    if (rows == 0 || dim == 0) return CFATTN_OK;
    if (!dy || !x || !w || !rstd || !dx) return fail(c, CFATTN_ERR_ARG, "null buffer");
    if (!fits_int(dim)) return fail(c, CFATTN_ERR_UNSUPPORTED, "dim=%zu above 2^31", dim);
    float* partial = nullptr;
    if (dw) {
        int rc = CFATTN_OK;
        partial = static_cast<float*>(
            slot(c, cfattn_ctx::OPS_PARTIAL, cfattn::rmsnorm_bwd_partial_floats(rows, dim) * sizeof(float), &rc));
        if (!partial) return rc;
    }
    CF_HIP(c, cfattn::launch_rmsnorm_bwd(dy, x, w, rstd, dx, dw, partial, rows, dim, acc != 0, to_stream(stream)),
           "rmsnorm backward launch");
    return CFATTN_OK;
}

int cfops_silu_mul_forward(cfattn_ctx* c, const float* g, const float* u, float* h, size_t n, void* stream) {
    CF_LOCK(c, stream);
    if (n == 0) return CFATTN_OK;
    if (!g || !u || !h) return fail(c, CFATTN_ERR_ARG, "null buffer");
    CF_HIP(c, cfattn::launch_silu_mul_fwd(g, u, h, n, to_stream(stream)), "silu_mul forward launch");
    return CFATTN_OK;
}

int cfops_silu_mul_backward(cfattn_ctx* c, const float* dh, const float* g, const float* u, float* dg, float* du,
                            size_t n, void* stream) {
    return cfops_silu_mul_grad(c, dh, g, u, dg, du, n, 1, stream);
}

int cfops_silu_mul_grad(cfattn_ctx* c, const float* dh, const float* g, const float* u, float* dg, float* du, size_t n,
                        int acc, void* stream) {
    CF_LOCK(c, stream);
    if (n == 0) return CFATTN_OK;
    if (!dh || !g || !u || !dg || !du) return fail(c, CFATTN_ERR_ARG, "null buffer");
    CF_HIP(c, cfattn::launch_silu_mul_bwd(dh, g, u, dg, du, n, acc != 0, to_stream(stream)), "silu_mul backward launch");
    return CFATTN_OK;
}

int cfops_cross_entropy_fwd_bwd(cfattn_ctx* c, const float* logits, const int64_t* targets, float* dlogits,
                                size_t rows, size_t vocab, float* loss, void* stream) {
    CF_LOCK(c, stream);
    if (!loss) return fail(c, CFATTN_ERR_ARG, "null loss");
    *loss = 0.0f;
    if (rows == 0) return CFATTN_OK;
    if (!logits || !targets || !dlogits) return fail(c, CFATTN_ERR_ARG, "null buffer");
    if (rows > (size_t)INT_MAX) return fail(c, CFATTN_ERR_UNSUPPORTED, "rows=%zu above 2^31", rows);
    const hipStream_t st = to_stream(stream);
    int rc = CFATTN_OK;
    void* misc = slot(c, cfattn_ctx::OPS_MISC, cfattn::kCeMiscBytes, &rc);
    if (!misc) return rc;
    float* row_loss = static_cast<float*>(slot(c, cfattn_ctx::OPS_ROWLOSS, rows * sizeof(float), &rc));
    if (!row_loss) return rc;
    CF_HIP(c, cfattn::launch_ce_begin(targets, rows, misc, st), "cross-entropy launch");
    CF_HIP(c, cfattn::launch_ce_rows(logits, targets, dlogits, row_loss, 0, rows, vocab, misc, st),
           "cross-entropy launch");
    CF_HIP(c, cfattn::launch_ce_finish(targets, row_loss, rows, misc, st), "cross-entropy launch");
    return ce_result(c, misc, targets, vocab, loss, st);
}

int cfops_set_head_chunk_limit(cfattn_ctx* c, size_t bytes) {
    if (!c) return CFATTN_ERR_ARG;
    std::lock_guard<std::mutex> lk(c->mu);
    c->head_chunk_bytes = bytes;
    return CFATTN_OK;
}

// The LM head and loss queued on `st` with the loss block at `misc` (device
// memory: n_valid, bad_row, loss); the caller holds the context lock and
// has checked the arguments.
static int lm_head_ce_queue(cfattn_ctx* c, const float* hn, const float* head, const int64_t* targets, size_t t, size_t d,
                     size_t vocab, float* dhn, float* dhead, void* misc, hipStream_t st) {
    size_t chunk = c->head_chunk_bytes / (vocab * sizeof(float));
    if (chunk < 1) chunk = 1;
    if (chunk > t) chunk = t;
    int rc = CFATTN_OK;
    float* row_loss = static_cast<float*>(slot(c, cfattn_ctx::OPS_ROWLOSS, t * sizeof(float), &rc));
    if (!row_loss) return rc;
    float* logits = static_cast<float*>(slot(c, cfattn_ctx::OPS_LOGITS, chunk * vocab * sizeof(float), &rc));
    if (!logits) return rc;
    CF_HIP(c, cfattn::launch_ce_begin(targets, t, misc, st), "cross-entropy launch");
    for (size_t r0 = 0; r0 < t; r0 += chunk) {
        const size_t nr = t - r0 < chunk ? t - r0 : chunk;
        // logits = hn . head^T (model.rs:438), then dlogits in place.
        CF_TRY(gemm(c, CFOPS_NT, hn + r0 * d, head, logits, nr, d, vocab, false, st));
        CF_HIP(c, cfattn::launch_ce_rows(logits, targets, logits, row_loss, r0, nr, vocab, misc, st),
               "cross-entropy launch");
        // dhn = dlogits . head (model.rs:454, overwritten); dhead += dlogits^T . hn (:457).
        CF_TRY(gemm(c, CFOPS_NN, logits, head, dhn + r0 * d, nr, vocab, d, false, st));
        if (dhead) CF_TRY(gemm(c, CFOPS_TN, logits, hn + r0 * d, dhead, vocab, nr, d, true, st));
    }
    CF_HIP(c, cfattn::launch_ce_finish(targets, row_loss, t, misc, st), "cross-entropy launch");
    return CFATTN_OK;
}

int cfops_lm_head_ce(cfattn_ctx* c, const float* hn, const float* head, const int64_t* targets, size_t t, size_t d,
                     size_t vocab, float* dhn, float* dhead, float* loss, void* stream) {
    CF_LOCK(c, stream);
    if (!loss) return fail(c, CFATTN_ERR_ARG, "null loss");
    *loss = 0.0f;
    if (t == 0) return CFATTN_OK;
    if (!hn || !head || !targets || !dhn) return fail(c, CFATTN_ERR_ARG, "null buffer");
    if (vocab == 0) return fail(c, CFATTN_ERR_ARG, "vocab must be positive");
    if (t > (size_t)INT_MAX) return fail(c, CFATTN_ERR_UNSUPPORTED, "t=%zu above 2^31", t);
    const hipStream_t st = to_stream(stream);
    int rc = CFATTN_OK;
    void* misc = slot(c, cfattn_ctx::OPS_MISC, cfattn::kCeMiscBytes, &rc);
    if (!misc) return rc;
    CF_TRY(lm_head_ce_queue(c, hn, head, targets, t, d, vocab, dhn, dhead, misc, st));
    return ce_result(c, misc, targets, vocab, loss, st);
}

static_assert(sizeof(cfops_ce_result) == sizeof(cfattn::CeMisc) &&
                  offsetof(cfops_ce_result, bad_row) == offsetof(cfattn::CeMisc, bad_row) &&
                  offsetof(cfops_ce_result, loss) == offsetof(cfattn::CeMisc, loss),
              "cfops_ce_result is the kernels' loss block");

int cfops_lm_head_ce_dev(cfattn_ctx* c, const float* hn, const float* head, const int64_t* targets, size_t t,
                         size_t d, size_t vocab, float* dhn, float* dhead, cfops_ce_result* result, void* stream) {
    CF_LOCK(c, stream);
    if (!result) return fail(c, CFATTN_ERR_ARG, "null result");
    if (t == 0) return fail(c, CFATTN_ERR_ARG, "t must be positive");
    if (!hn || !head || !targets || !dhn) return fail(c, CFATTN_ERR_ARG, "null buffer");
    if (vocab == 0) return fail(c, CFATTN_ERR_ARG, "vocab must be positive");
    if (t > (size_t)INT_MAX) return fail(c, CFATTN_ERR_UNSUPPORTED, "t=%zu above 2^31", t);
    return lm_head_ce_queue(c, hn, head, targets, t, d, vocab, dhn, dhead, result, to_stream(stream));
}

int cfops_linear_forward(cfattn_ctx* c, const float* x, const float* w, const float* lora_a, const float* lora_b,
                         float lora_scale, size_t t, size_t in, size_t out, size_t rank, float* y, float* xs,
                         void* stream) {
    CF_LOCK(c, stream);
    if (t == 0 || out == 0) return CFATTN_OK;
    if (!x || !w || !y) return fail(c, CFATTN_ERR_ARG, "null buffer");
    if (lora_a && (!lora_b || !xs || rank == 0)) return fail(c, CFATTN_ERR_ARG, "adapter needs A, B, xs and rank > 0");
    cfops_linear l{};
    l.w = w, l.lora_a = lora_a, l.lora_b = lora_b, l.lora_scale = lora_scale, l.out = out, l.rank = rank;
    l.y = y, l.xs = xs;
    CF_TRY(check_linears(c, t, in, &l, 1));
    return linears_forward(c, x, t, in, &l, 1, to_stream(stream));
}

int cfops_linear_backward(cfattn_ctx* c, const float* x, const float* xs, const float* dy, const float* w,
                          const float* lora_a, const float* lora_b, float lora_scale, size_t t, size_t in, size_t out,
                          size_t rank, float* dx, float* gw, float* ga, float* gb, void* stream) {
    CF_LOCK(c, stream);
    if (t == 0) return CFATTN_OK;
    if (!x || !dy || !w || !dx) return fail(c, CFATTN_ERR_ARG, "null buffer");
    if (lora_a && (!lora_b || !xs || rank == 0)) return fail(c, CFATTN_ERR_ARG, "adapter needs A, B, xs and rank > 0");
    cfops_linear l{};
    l.w = w, l.lora_a = lora_a, l.lora_b = lora_b, l.lora_scale = lora_scale, l.out = out, l.rank = rank;
    l.xs = const_cast<float*>(xs), l.dy = dy, l.gw = gw, l.ga = lora_a ? ga : nullptr, l.gb = lora_a ? gb : nullptr;
    CF_TRY(check_linears(c, t, in, &l, 1));
    return linears_backward(c, x, t, in, dx, &l, 1, true, true, to_stream(stream));
}

int cfops_linears_forward(cfattn_ctx* c, const float* x, size_t t, size_t in, const cfops_linear* lin, size_t n,
                          void* stream) {
    CF_LOCK(c, stream);
    if (t == 0 || n == 0) return CFATTN_OK;
    if (!x || !lin) return fail(c, CFATTN_ERR_ARG, "null buffer");
    for (size_t i = 0; i < n; i++) {
        const cfops_linear& l = lin[i];
        if (l.out && (!l.w || !l.y)) return fail(c, CFATTN_ERR_ARG, "null buffer");
        if (l.lora_a && (!l.lora_b || !l.xs || l.rank == 0))
            return fail(c, CFATTN_ERR_ARG, "adapter needs A, B, xs and rank > 0");
    }
    CF_TRY(check_linears(c, t, in, lin, n));
    for (size_t i = 0; i < n; i += cfattn::kGemmProblems) {
        const size_t m = n - i < (size_t)cfattn::kGemmProblems ? n - i : (size_t)cfattn::kGemmProblems;
        CF_TRY(linears_forward(c, x, t, in, lin + i, m, to_stream(stream)));
    }
    return CFATTN_OK;
}

int cfops_linears_backward(cfattn_ctx* c, const float* x, size_t t, size_t in, float* dx, const cfops_linear* lin,
                           size_t n, int acc, void* stream) {
    CF_LOCK(c, stream);
    if (t == 0 && !acc)
        for (size_t i = 0; lin && i < n; i++) {
            const cfops_linear& l = lin[i];
            CF_TRY(zero_grad(c, l.gw, l.out * in, to_stream(stream)));
            CF_TRY(zero_grad(c, l.ga, l.rank * in, to_stream(stream)));
            CF_TRY(zero_grad(c, l.gb, l.out * l.rank, to_stream(stream)));
        }
    if (n == 0 && !acc) return zero_grad(c, dx, t * in, to_stream(stream));
    if (t == 0 || n == 0) return CFATTN_OK;
    if (!x || !lin) return fail(c, CFATTN_ERR_ARG, "null buffer");
    for (size_t i = 0; i < n; i++) {
        const cfops_linear& l = lin[i];
        if (!l.dy || !l.w) return fail(c, CFATTN_ERR_ARG, "null buffer");
        if (l.lora_a && (!l.lora_b || !l.xs || l.rank == 0))
            return fail(c, CFATTN_ERR_ARG, "adapter needs A, B, xs and rank > 0");
    }
    CF_TRY(check_linears(c, t, in, lin, n));
    for (size_t i = 0; i < n; i += cfattn::kGemmProblems) {
        const size_t m = n - i < (size_t)cfattn::kGemmProblems ? n - i : (size_t)cfattn::kGemmProblems;
        CF_TRY(linears_backward(c, x, t, in, dx, lin + i, m, acc || i > 0, acc != 0, to_stream(stream)));
    }
    return CFATTN_OK;
}

int cfops_adamw_update(cfattn_ctx* c, float* p, const float* g, float* m, float* v, size_t n, uint64_t t, float lr,
                       float beta1, float beta2, float eps, float weight_decay, void* stream) {
    return cfops_adamw_update_multi(c, 1, &p, &g, &m, &v, &n, &weight_decay, t, lr, beta1, beta2, eps, stream);
}

int cfops_adamw_update_multi(cfattn_ctx* c, size_t count, float* const* p, const float* const* g, float* const* m,
                             float* const* v, const size_t* n, const float* weight_decay, uint64_t t, float lr,
                             float beta1, float beta2, float eps, void* stream) {
    CF_LOCK(c, stream);
    if (count && (!p || !g || !m || !v || !n || !weight_decay)) return fail(c, CFATTN_ERR_ARG, "null array");
    for (size_t i = 0; i < count; i++)
        if (n[i] && (!p[i] || !g[i] || !m[i] || !v[i])) return fail(c, CFATTN_ERR_ARG, "null buffer");
    cfattn::AdamwArgs a;
    a.count = 0, a.lr = lr, a.beta1 = beta1, a.beta2 = beta2, a.eps = eps;
    // optim.rs:21-22: the bias corrections, `t as i32` as in the reference.
    a.bc1 = 1.0f - powi_f32(beta1, (int)(int32_t)t);
    a.bc2 = 1.0f - powi_f32(beta2, (int)(int32_t)t);
    for (size_t i = 0; i < count; i++) {
        if (n[i]) a.t[a.count++] = {p[i], g[i], m[i], v[i], (long)n[i], weight_decay[i], 0, 0};
        if (a.count == cfattn::kAdamwBatch || (i + 1 == count && a.count)) {
            // Tensors of one launch are updated side by side.
            const int step = adamw_overlaps(a) ? 1 : a.count;
            for (int k = 0; k < a.count; k += step) {
                cfattn::AdamwArgs b = a;
                std::copy(a.t + k, a.t + k + step, b.t);
                b.count = step;
                CF_HIP(c, cfattn::launch_adamw(b, to_stream(stream)), "adamw launch");
            }
            a.count = 0;
        }
    }
    return CFATTN_OK;
}

}  // extern "C"
