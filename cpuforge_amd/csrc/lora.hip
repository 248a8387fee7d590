// The gradients of LoRA adapters in Linear::backward (crates/model/src/
// linear.rs:75-90), gb += dy^T xs and ga += dxa^T x, as streaming passes over
// their long operand on the f32 MFMA: per-chunk partial sums over the tokens,
// then the chunks added in order.  Several linears go in one launch.  Every sum
// has a fixed order (no atomics): results are reproducible bit for bit.  Any
// rank, in blocks of 16; no alignment beyond a float's.  (The adapters' other
// products are gemm_f32.hip's: xs = scale x A^T and dxa = scale dy B on its rows
// kernel, xs B^T and dxa A as segments of the base products.)
//
// Bound: latency of one pass over the long operand (9.4 MB for 4096 x 576,
// resident in the memory-side cache).  The operands come straight from
// memory in MFMA layout, 16 bytes a lane: no LDS but for the waves' sums.
// 4096 tokens, rank 16, SmolLM's gate and up projections: 15 + 4.8 us.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "cfops_kernels.hpp"

namespace cfattn {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

// Lane l of v_mfma_f32_16x16x4_f32 holds A[l % 16][l / 16], B[l / 16][l % 16]
// and C[4 * (l / 16) + i][l % 16], i = 0..3.
__device__ __forceinline__ f32x4 mfma16(float a, float b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// p[0..3], elements at or past n zero (and not read).
__device__ __forceinline__ f32x4 load4(const float* __restrict__ p, int n) {
    if (n >= 4) return *reinterpret_cast<const f32x4u*>(p);
    f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int i = 0; i < n; i++) v[i] = p[i];
    return v;
}

constexpr int kBatch = 4;  // runs of a wave whose loads are in flight together

// part[chunk][n][j] = sum over the chunk's tokens i of big[i][n] * small[i][j].
// A workgroup takes 64 columns n and 16 j of one chunk; lane l loads columns
// 4 * (l % 16) .. + 3 of token l / 16 of four, one MFMA per column of the four.
// Its waves take every fourth run of four tokens; their sums are added in wave order.
__global__ __launch_bounds__(256) void lora_grad_kernel(const LoraGrad g) {
    __shared__ float red[4][64][17];
    int b = blockIdx.x, ji = 0;
    for (;; ji++) {
        const int n = (g.job[ji].ncol + 63) / 64 * ((g.job[ji].r + 15) / 16);
        if (b < n) break;
        b -= n;
    }
    const LoraGradJob& p = g.job[ji];
    const int nrb = (p.r + 15) / 16;
    const int n0 = b / nrb * 64, j0 = b % nrb * 16;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int l16 = lane & 15, tq = lane >> 4;
    // (Unsigned: past the last token by up to a batch without overflow.)
    const unsigned i0 = blockIdx.y * g.tokens, i1 = min((unsigned)g.t, i0 + g.tokens);
    const int left = max(0, min(4, p.ncol - n0 - 4 * l16));
    const long col = (long)n0 + 4 * l16;
    const int j = min(j0 + l16, p.r - 1);
    f32x4 acc[4] = {};
    auto add = [&](unsigned i, bool in) {
        f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
        float s = 0.0f;
        if (in) {
            v = load4(p.big + (long)i * p.ncol + col, left);
            s = p.small[(long)i * p.r + j];
        }
#pragma unroll
        for (int q = 0; q < 4; q++) acc[q] = mfma16(v[q], s, acc[q]);
    };
    unsigned i = i0 + 4 * wave;
    if (p.ncol - n0 >= 64)
        for (; i + 16 * (kBatch - 1) + 4 <= i1; i += 16 * kBatch) {
            f32x4 v[kBatch];
            float s[kBatch];
#pragma unroll
            for (int u = 0; u < kBatch; u++) {
                const long r = i + 16 * u + tq;
                v[u] = load4(p.big + r * p.ncol + col, 4);
                s[u] = p.small[r * p.r + j];
            }
#pragma unroll
            for (int u = 0; u < kBatch; u++)
#pragma unroll
                for (int q = 0; q < 4; q++) acc[q] = mfma16(v[u][q], s[u], acc[q]);
        }
    for (; i + 4 <= i1; i += 16) add(i + tq, true);
    if (i < i1) add(i + tq, i + tq < i1);
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
        for (int e = 0; e < 4; e++) red[wave][4 * (4 * tq + e) + q][l16] = acc[q][e];
    __syncthreads();
    float* out = g.part + p.off + (long)blockIdx.y * p.ncol * p.r;
    for (int e = tid; e < 1024; e += 256) {
        const int n = e >> 4, jj = e & 15;
        if (n >= p.ncol - n0 || jj >= p.r - j0) continue;
        out[((long)n0 + n) * p.r + j0 + jj] = red[0][n][jj] + red[1][n][jj] + red[2][n][jj] + red[3][n][jj];
    }
}

// The chunks' sums, in chunk order, into a gradient [ncol][r] (gb) or
// [r][ncol] (ga, TRANSPOSED).
__global__ __launch_bounds__(256) void lora_grad_reduce_kernel(const LoraGrad g) {
    int b = blockIdx.x, ji = 0;
    for (;; ji++) {
        const int n = (int)(((long)g.job[ji].ncol * g.job[ji].r + 255) / 256);
        if (b < n) break;
        b -= n;
    }
    const LoraGradJob& p = g.job[ji];
    const long e = (long)b * 256 + threadIdx.x, n = (long)p.ncol * p.r;
    if (e >= n) return;
    const float* q = g.part + p.off + e;
    float s = 0.0f;
#pragma unroll 8
    for (int c = 0; c < g.chunks; c++) s += q[c * n];
    float* o = p.transposed ? p.out + (e % p.r) * p.ncol + e / p.r : p.out + e;
    *o = g.acc ? *o + s : s;
}

int cdiv(long a, long b) { return (int)((a + b - 1) / b); }

}  // namespace

size_t lora_grad_plan(LoraGrad& g) {
    // Chunks of whole 64-token batches, as many as make about 768 workgroups
    // (three to a CU).
    long blocks = 0;
    for (int i = 0; i < g.njobs; i++) blocks += (long)cdiv(g.job[i].ncol, 64) * cdiv(g.job[i].r, 16);
    const int most = cdiv(g.t, 64);
    int chunks = blocks ? cdiv(768, blocks) : 1;
    if (chunks > most) chunks = most;
    g.tokens = std::min((long)cdiv(cdiv(g.t, chunks), 64) * 64, (long)INT32_MAX);
    g.chunks = cdiv(g.t, g.tokens);
    long off = 0;
    for (int i = 0; i < g.njobs; i++) {
        g.job[i].off = off;
        off += (long)g.chunks * g.job[i].ncol * g.job[i].r;
    }
    return (size_t)off;
}

hipError_t launch_lora_grad(const LoraGrad& g, hipStream_t st) {
    long blocks = 0, rblocks = 0;
    for (int i = 0; i < g.njobs; i++) {
        blocks += (long)cdiv(g.job[i].ncol, 64) * cdiv(g.job[i].r, 16);
        rblocks += cdiv((long)g.job[i].ncol * g.job[i].r, 256);
    }
    if (blocks == 0) return hipSuccess;
    if (blocks > INT32_MAX || rblocks > INT32_MAX || g.chunks > 65535) return hipErrorInvalidConfiguration;
    lora_grad_kernel<<<dim3((unsigned)blocks, g.chunks), 256, 0, st>>>(g);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    lora_grad_reduce_kernel<<<(unsigned)rblocks, 256, 0, st>>>(g);
    return hipGetLastError();
}

}  // namespace cfattn
