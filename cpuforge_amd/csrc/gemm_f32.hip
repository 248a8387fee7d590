// f32 GEMMs of the layer ops (matmul_nn / matmul_nt / matmul_tn,
// crates/core/src/matmul.rs:127-147, and Linear's products,
// crates/model/src/linear.rs:56-91) on the bf16 matrix cores, each f32
// operand split into three bf16 pieces (split3.hpp).
//
// What bounds it: on a full chip the board's power.  2000 x 2048 x 8192 (m, k,
// n) ran at 1.85 of 2.4 GHz with the matrix cores busy in 62% of the cycles:
// 160-200 TFLOP/s of f32 work, 960-1200 of bf16, against 133-144 for the f32 MFMA
// library GEMM it replaced (the bf16 MFMA alone reaches 1704 on random
// operands).  On the small grids of a layer (160 tiles of 128 x 128 for 4096
// x 576) it is a workgroup's own chain: two waves to a SIMD, 49% matrix-core
// busy between the splitting, the LDS reads and one barrier a step.  Before
// and after, in us: 4096 x 1536 x 576 70 and 65 (A B^T), 71 and 70 (A B); 4096 x 576 x
// 1536 65 and 53, 62 and 54; 2000 x 2048 x 8192 465 and 345; the LM head's 2730 x 576 x
// 49152 1160 and 926, its gradients 2730 x 49152 x 576 2610 and 983 and 49152 x 2730 x
// 576 1150 and 965.  (Of these 2-7% is the scaling of the values, split3.hpp: 885,
// 933 and 917 for the last three without.)  From 128 to 512 rows by a layer's
// widths it is slower than the library was: 128 x 1536 x 576 7.5 and 12.4, 256 x 576 x 1536
// 8.1 and 14.6, 512 x 576 x 1536 10.8 and 15.0, 576 x 512 x 1536 (A^T B) 11.7 and 17.2; with
// fewer rows the kernel for few rows (below) runs.  (There, two or three groups of
// waves to a tile, each over its part of k: 12.6 where this takes 15.0, 16.0 for 18.0.)
//
// A workgroup splits its tiles as it stores them to LDS (three planes), so
// memory is read in f32, once per tile.  Two LDS buffers and two register
// sets: the loads of a step are two steps old when they are split.  (One more
// buffer, so that no wave waits at a step's first LDS read, and one wave to a SIMD:
// slower, 73 us where this takes 60.  Unpacking with v_dot2_f32_bf16, one
// instruction for two: slower, it needs wait states.)
//
// Relative error against 64 bits, normal values, before and after: k = 576
// 4.3e-7 and 1.4e-7, k = 4096 1.1e-6 and 2.2e-7.  The leading product has its
// own sums: in one sum with the other five the MFMA cuts off their low bits as it
// aligns them to the larger values (towards minus infinity, so every sum came
// out 4e-8 to 1.5e-7 of its size too small, and a training step's gradients four times
// further off than before).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "cfops_kernels.hpp"
#include "split3.hpp"

namespace cfattn {
namespace {

constexpr int kOct = 4;       // octets (runs of eight k) of a step
constexpr int kBK = 8 * kOct;  // k values of a step

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

struct GemmArgs {
    GemmProblem pr[kGemmProblems];
    int npr, m, acc;
    int mt, nt;          // tiles over m, and over all problems' n
    int per;             // k steps per split
    int n_inner;
    float* part;         // partial products of the splits, or null
    int y0;              // rows kernel: first column block of the launch
};

template <bool STRIDED>
__device__ __forceinline__ float elem(const float* __restrict__ p, long ld, long row, long k) {
    return STRIDED ? p[k * ld + row] : p[row * ld + k];
}

// k steps of a problem: a step is kOct octets.  First the whole steps of each
// segment in turn, then the segments' remaining octets, kOct to a step.
__host__ __device__ __forceinline__ int whole_steps(const GemmProblem& p) {
    int n = 0;
    for (int s = 0; s < p.nseg; s++) n += p.seg[s].k / kBK;
    return n;
}
__host__ __device__ __forceinline__ int all_steps(const GemmProblem& p) {
    int n = 0;
    for (int s = 0; s < p.nseg; s++) n += (p.seg[s].k % kBK + 7) / 8;
    return whole_steps(p) + (n + kOct - 1) / kOct;
}
// The octet `o` of the rest: its segment, first k and length (0 past the last).
struct Octet {
    int seg, k, len;
};
__device__ __forceinline__ Octet rest_octet(const GemmProblem& p, int o) {
    Octet r{0, 0, 0};
    for (int s = 0; s < p.nseg; s++) {
        const int k = p.seg[s].k, n = (k % kBK + 7) / 8;
        if (o >= 0 && o < n) {
            const int k0 = k / kBK * kBK + 8 * o;
            r = Octet{s, k0, min(8, k - k0)};
        }
        o -= n;
    }
    return r;
}

// This thread's share of an operand tile of ROWS rows and kOct octets, NT
// threads: U units of one row and eight consecutive k.
//   k along memory: kOct lanes cover the 32 * kOct bytes of a row;
//   STRIDED: a wave covers 64 consecutive rows at each of its eight k.
// Off: type of a byte offset within a tile.
template <bool STRIDED, int ROWS, int NT, typename Off>
struct TileLoad {
    static constexpr int U = ROWS * kOct / NT;
    // 16-byte LDS chunks from octet to octet: eight lanes of a write (two rows,
    // kOct octets) land on eight different 16-byte bank groups.
    static constexpr int PITCH = ROWS + 2;
    static_assert(U * NT == ROWS * kOct, "a tile must be whole units per thread");
    float v[U][8];
    __device__ __forceinline__ static int row(int tid, int u) {
        return STRIDED ? (tid & 63) + 64 * (tid / (64 * kOct)) + (NT / kOct) * u : tid / kOct + (NT / kOct) * u;
    }
    __device__ __forceinline__ static int oct(int tid) {
        return (STRIDED ? wave_uniform(tid >> 6) : tid) % kOct;
    }
    // Byte offset of unit u in a tile that starts at its first row and k.
    // Rows past the last one repeat it (their results are not stored).
    __device__ __forceinline__ static Off offset(int tid, int u, int last, Off ld) {
        const Off r = min(row(tid, u), last);
        return STRIDED ? 4 * r : 4 * (r * ld + oct(tid) * 8);
    }
    __device__ __forceinline__ void load(const float* __restrict__ base, long ld, const Off (&off)[U], int tid) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            if constexpr (STRIDED) {
                const float* q = base + oct(tid) * 8 * ld;
#pragma unroll
                for (int j = 0; j < 8; j++)
                    v[u][j] = *reinterpret_cast<const float*>(reinterpret_cast<const char*>(q + j * ld) + off[u]);
            } else {
                const char* q = reinterpret_cast<const char*>(base) + off[u];
                const f32x4u a = *reinterpret_cast<const f32x4u*>(q), b = *reinterpret_cast<const f32x4u*>(q + 16);
#pragma unroll
                for (int j = 0; j < 4; j++) v[u][j] = a[j], v[u][j + 4] = b[j];
            }
        }
    }
    // One octet of a segment, zero past its length.
    __device__ __forceinline__ void load_octet(const float* __restrict__ p, long ld, int row0, int last, int k, int len,
                                               int tid) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int r = row0 + min(row(tid, u), last);
#pragma unroll
            for (int j = 0; j < 8; j++) v[u][j] = j < len ? elem<STRIDED>(p, ld, r, k + j) : 0.0f;
        }
    }
    // Split and stored as three planes of [kOct][PITCH] chunks.
    __device__ __forceinline__ void store(uint4* s, int tid) const {
        constexpr int P = kOct * PITCH;
#pragma unroll
        for (int u = 0; u < U; u++) {
            const Split8 sp = split8_scaled(v[u]);
            uint4* d = s + oct(tid) * PITCH + row(tid, u);
            d[0] = sp.p[0];
            d[P] = sp.p[1];
            d[2 * P] = sp.p[2];
        }
    }
};

// The LDS writes of this step are done in every wave; loads to registers stay
// in flight (__syncthreads would wait for them).
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// C tile of BM x BN, NT / 64 waves in WR = NT / 128 rows of two.
template <bool AS, bool BS, int BM, int BN, int NT, typename Off = uint32_t>
__global__ __launch_bounds__(NT, 2) void gemm_f32_kernel(const GemmArgs g) {
    constexpr int WR = NT / 128;
    constexpr int MB = BM / WR / 32, NB = BN / 64;  // 32 x 32 blocks of a wave
    using LoadA = TileLoad<AS, BM, NT, Off>;
    using LoadB = TileLoad<BS, BN, NT, Off>;
    constexpr int PA = kOct * LoadA::PITCH, PB = kOct * LoadB::PITCH;
    __shared__ uint4 sA[2][3 * PA];
    __shared__ uint4 sB[2][3 * PB];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = wave_uniform(tid >> 6);
    const int l32 = lane & 31, hh = lane >> 5;
    int id = xcd_remap(blockIdx.x, gridDim.x, 1);
    const int tiles = g.mt * g.nt;
    const int split = id / tiles;
    id %= tiles;
    const int tm = g.n_inner ? id / g.nt : id % g.mt;
    int tn = g.n_inner ? id % g.nt : id / g.mt;
    int pi = 0;
    long part_off = 0;  // columns of the problems before this one
    for (; pi + 1 < g.npr && tn > (g.pr[pi].n - 1) / BN; pi++) {
        tn -= (g.pr[pi].n - 1) / BN + 1;
        part_off += g.pr[pi].n;
    }
    const GemmProblem& p = g.pr[pi];
    const int m0 = tm * BM, n0 = tn * BN;
    const int lastA = g.m - 1 - m0, lastB = p.n - 1 - n0;
    const int n_whole = whole_steps(p);
    const int st0 = split * g.per, st1 = min(all_steps(p), st0 + g.per);

    f32x16 acc[MB][NB], low[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
        for (int j = 0; j < NB; j++) acc[i][j] = low[i][j] = zero16();

    const int ar = (wave >> 1) * (BM / WR) + l32, br = (wave & 1) * (BN / 2) + l32;
    auto products = [&](int cur) {
#pragma unroll
        for (int s = 0; s < kOct / 2; s++) {
            bf16x8 a[3][MB], b[3][NB];
#pragma unroll
            for (int q = 0; q < 3; q++) {
#pragma unroll
                for (int i = 0; i < MB; i++)
                    a[q][i] = __builtin_bit_cast(bf16x8, sA[cur][q * PA + (2 * s + hh) * LoadA::PITCH + ar + 32 * i]);
#pragma unroll
                for (int j = 0; j < NB; j++)
                    b[q][j] = __builtin_bit_cast(bf16x8, sB[cur][q * PB + (2 * s + hh) * LoadB::PITCH + br + 32 * j]);
            }
            // The five products below the first go to sums of their own, smallest first.
            constexpr int pa[5] = {2, 0, 1, 1, 0}, pb[5] = {0, 2, 1, 0, 1};
#pragma unroll
            for (int q = 0; q < 5; q++)
#pragma unroll
                for (int i = 0; i < MB; i++)
#pragma unroll
                    for (int j = 0; j < NB; j++) low[i][j] = mfma32(a[pa[q]][i], b[pb[q]][j], low[i][j]);
#pragma unroll
            for (int i = 0; i < MB; i++)
#pragma unroll
                for (int j = 0; j < NB; j++) acc[i][j] = mfma32(a[0][i], b[0][j], acc[i][j]);
        }
    };

    // Whole k steps.  A step: the products of one LDS buffer; beside them the
    // next step's tile (in registers since two steps ago) is split into the
    // other buffer, and then the loads of the step three ahead go out into
    // the same registers.  Past the end the last step's loads are repeated: a
    // load that may or may not be in flight would make every wait one for
    // all of them.
    const int end = min(st1, n_whole);
    if (st0 < end) {
        struct Regs {
            LoadA a;
            LoadB b;
        } r0, r1;
        // Where the next load is: segment, its pointers and whole steps left.
        int sg = 0, left = st0, todo = end - st0;
        while (left >= p.seg[sg].k / kBK) left -= p.seg[sg++].k / kBK;
        const float *pa, *pb;
        long lda, ldb;
        Off offa[LoadA::U], offb[LoadB::U];
        auto enter = [&](int skip) {
            const GemmSeg& s = p.seg[sg];
            lda = s.lda, ldb = s.ldb;
            left = s.k / kBK - skip;
            pa = AS ? s.a + m0 + (long)skip * kBK * lda : s.a + m0 * lda + (long)skip * kBK;
            pb = BS ? s.b + n0 + (long)skip * kBK * ldb : s.b + n0 * ldb + (long)skip * kBK;
#pragma unroll
            for (int u = 0; u < LoadA::U; u++) offa[u] = LoadA::offset(tid, u, lastA, (Off)lda);
#pragma unroll
            for (int u = 0; u < LoadB::U; u++) offb[u] = LoadB::offset(tid, u, lastB, (Off)ldb);
        };
        enter(left);
        auto load = [&](Regs& r) {
            r.a.load(pa, lda, offa, tid);
            r.b.load(pb, ldb, offb, tid);
            if (--todo > 0) {
                if (--left > 0) {
                    pa += AS ? kBK * lda : kBK;
                    pb += BS ? kBK * ldb : kBK;
                } else {
                    do sg++;
                    while (p.seg[sg].k < kBK);
                    enter(0);
                }
            }
        };
        load(r0);
        load(r1);
        r0.a.store(sA[0], tid);
        r0.b.store(sB[0], tid);
        load(r0);
        int st = st0;
        auto step = [&](int cur, Regs& r) {
            products(cur);
            r.a.store(sA[cur ^ 1], tid);
            r.b.store(sB[cur ^ 1], tid);
            load(r);
            lds_barrier();
        };
        lds_barrier();
        for (; st + 1 < end; st += 2) {
            step(0, r1);
            step(1, r0);
        }
        if (st < end) step(0, r1);
    }
    for (int st = max(st0, n_whole); st < st1; st++) {
        LoadA a;
        LoadB b;
        const Octet oa = rest_octet(p, kOct * (st - n_whole) + LoadA::oct(tid));
        const Octet ob = rest_octet(p, kOct * (st - n_whole) + LoadB::oct(tid));
        a.load_octet(p.seg[oa.seg].a, p.seg[oa.seg].lda, m0, lastA, oa.k, oa.len, tid);
        b.load_octet(p.seg[ob.seg].b, p.seg[ob.seg].ldb, n0, lastB, ob.k, ob.len, tid);
        a.store(sA[0], tid);
        b.store(sB[0], tid);
        lds_barrier();
        products(0);
        lds_barrier();
    }

    // A sum that is not finite may only be so in the pieces: such a wave forms
    // its tile again with f32 MFMAs.  Its operands come straight from memory,
    // four k a lane (lanes 0-31 the first four of eight, 32-63 the others).  The
    // LM head with its gradients, 512 x 576 x 8192: 0.39 ms finite, 0.56 with NaN
    // in one row, 0.73 in all (with a scalar loop over k per output 6.0 and 8.5);
    // 4096 x 576 x 49152: 5.6, 8.9 and 21.
    bool odd = false;
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
        for (int j = 0; j < NB; j++) {
            acc[i][j] += low[i][j];
#pragma unroll
            for (int r = 0; r < 16; r++) odd |= !(fabsf(acc[i][j][r]) < INFINITY);
            acc[i][j] *= kSplitUnscale * kSplitUnscale;
        }
    if (__any(odd)) {
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
            for (int j = 0; j < NB; j++) acc[i][j] = zero16();
        auto run = [&](const GemmSeg& s, int k0, int k1) {
            // Two groups of eight k: the loads of both are in flight together.
            const unsigned n = max(k1 - k0, 0);
            for (unsigned d = 0; d < n; d += 16) {
                float a[2][MB][4], b[2][NB][4];
#pragma unroll
                for (int h = 0; h < 2; h++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const unsigned de = d + 8 * h + 4 * hh + e;
                        const long k = k0 + (long)de;
#pragma unroll
                        for (int i = 0; i < MB; i++)
                            a[h][i][e] = de < n ? elem<AS>(s.a, s.lda, m0 + min(ar + 32 * i, lastA), k) : 0.0f;
#pragma unroll
                        for (int j = 0; j < NB; j++)
                            b[h][j][e] = de < n ? elem<BS>(s.b, s.ldb, n0 + min(br + 32 * j, lastB), k) : 0.0f;
                    }
#pragma unroll
                for (int h = 0; h < 2; h++)
#pragma unroll
                    for (int e = 0; e < 4; e++)
#pragma unroll
                        for (int i = 0; i < MB; i++)
#pragma unroll
                            for (int j = 0; j < NB; j++)
                                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[h][i][e], b[h][j][e], acc[i][j], 0,
                                                                                 0, 0);
            }
        };
        int first = 0;  // whole steps of the segments before
        for (int s = 0; s < p.nseg; s++) {
            const int n = p.seg[s].k / kBK;
            run(p.seg[s], (max(st0, first) - first) * kBK, (min(st1, first + n) - first) * kBK);
            first += n;
        }
        for (int o = kOct * (max(st0, n_whole) - n_whole); o < kOct * (st1 - n_whole); o++) {
            const Octet oc = rest_octet(p, o);
            run(p.seg[oc.seg], oc.k, oc.k + oc.len);
        }
    }
    // (Unsigned: a tile's last rows and columns may lie past 2^31.)
    const unsigned mw = (unsigned)m0 + (wave >> 1) * (BM / WR) + 4 * hh, nw = (unsigned)n0 + br;

    // Partial products: [split][m][all problems' columns, problem by problem].
    float* out = p.c;
    if (g.part) {
        long cols = 0;
        for (int i = 0; i < g.npr; i++) cols += g.pr[i].n;
        out = g.part + (split * cols + part_off) * g.m;
    }
    const bool add = g.acc && !g.part;
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
        for (int j = 0; j < NB; j++) {
            const unsigned col = nw + 32 * j;
            if (col >= (unsigned)p.n) continue;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const unsigned row = mw + 32 * i + 8 * (r >> 2) + (r & 3);
                if (row >= (unsigned)g.m) continue;
                float* o = out + (long)row * p.n + col;
                *o = add ? *o + acc[i][j][r] : acc[i][j][r];
            }
        }
}

// C (+)= the splits' partial products, added in split order.
__global__ __launch_bounds__(256) void gemm_f32_reduce_kernel(const GemmArgs g, int splits, long cols) {
    const GemmProblem& p = g.pr[blockIdx.y];
    long off = 0;
    for (int i = 0; i < (int)blockIdx.y; i++) off += g.pr[i].n;
    const long mn = (long)g.m * p.n, stride = cols * g.m;
    const float* part = g.part + off * g.m;
    for (long e = (long)blockIdx.x * 256 + threadIdx.x; e < mn; e += (long)gridDim.x * 256) {
        float s = part[e];
        for (int i = 1; i < splits; i++) s += part[i * stride + e];
        p.c[e] = g.acc ? p.c[e] + s : s;
    }
}

// ------------------------------------------------------------------- rows
typedef float f32x4 __attribute__((ext_vector_type(4)));

// p[0..3], elements at or past n zero (and not read).
__device__ __forceinline__ f32x4 load4(const float* __restrict__ p, int n) {
    if (n >= 4) return *reinterpret_cast<const f32x4u*>(p);
    f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int i = 0; i < n; i++) v[i] = p[i];
    return v;
}

constexpr int kRowWaves = 8;
constexpr int kRowBatch = 4;  // runs of a wave whose loads are in flight together

// The product on the f32 MFMA for few rows or few columns, where a tile of the
// kernel above is mostly padding and its chain of steps (and the pass that adds
// a split's sums) all there is: a workgroup takes 16 rows and 16 columns, its
// waves every kRowWaves-th run of 16 k, straight from memory in MFMA layout (lane
// l: row and column l % 16, four consecutive k, one per MFMA), and their sums
// are added in wave order.  Bound: the latency of a wave's loads, four runs in
// flight (1.7 us a batch), on each CU one workgroup after the other.
// In us for m x k x n, a library's f32 kernels, the kernel above and this: 1 x 576 x
// 1536 4.8, 8.5, 3.8; 16 x 576 x 1536 4.8, 8.8, 4.5; 16 x 1536 x 576 6.1, 10.2, 7.6; 64 x
// 576 x 1536 6.6, 9.8, 6.3; 1 x 576 x 49152 20.3, 29.6, 19.7; 16 x 2048 x 8192 13.8, 22.8,
// 17.5.  An adapter's products at 4096 tokens, rank 16: 7.7 (xs) and 9.4 (dxa) for
// the gate and up projections.  (32 x 32 tiles, and eight runs in flight: slower.)
// Relative error against 64 bits, the same three: k = 576 2.2e-7, 0.8e-7, 1.0e-7; k
// = 2048 4.1e-7, 1.3e-7, 1.6e-7.
// Off: type of a byte offset within 16 rows of B.
template <bool BS, typename Off = uint32_t>
__global__ __launch_bounds__(64 * kRowWaves) void gemm_rows_kernel(const GemmArgs g) {
    __shared__ float red[kRowWaves][16][17];
    int y = blockIdx.y + g.y0, pi = 0;
    while (y > (g.pr[pi].n - 1) / 16) y -= (g.pr[pi++].n - 1) / 16 + 1;
    const GemmProblem& p = g.pr[pi];
    const int tid = threadIdx.x, wave = wave_uniform(tid >> 6), lane = tid & 63;
    const int l16 = lane & 15, kq = (lane >> 4) * 4;
    const int row0 = blockIdx.x * 16, j0 = y * 16;
    const int row = row0 + min(l16, g.m - 1 - row0), j = j0 + min(l16, p.n - 1 - j0);
    // Lane l of v_mfma_f32_16x16x4_f32 holds A[l % 16][l / 16], B[l / 16][l % 16]
    // and C[4 * (l / 16) + i][l % 16], i = 0..3.
    // Four chains of sums (and the waves' in pairs): a quarter of the roundings
    // at the full sum's size.
    f32x4 acc[4] = {};
    auto add = [&](const f32x4& a, const f32x4& b) {
#pragma unroll
        for (int i = 0; i < 4; i++) acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], acc[i], 0, 0, 0);
    };
    for (int s = 0; s < p.nseg; s++) {
        const GemmSeg& sg = p.seg[s];
        const float* a = sg.a + (long)row * sg.lda + kq;
        const float* b = BS ? sg.b : sg.b + (long)j * sg.ldb + kq;
        const Off at = BS ? 4 * ((Off)kq * (Off)sg.ldb + (Off)j) : 0;
        // Run c's k, of which this lane has n (at most four).
        auto operand = [&](int c, int n) {
            if constexpr (!BS) return load4(b + c * 16, n);
            const float* q = b + (long)c * 16 * sg.ldb;
            f32x4 v;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const char* e = reinterpret_cast<const char*>(q + i * sg.ldb) + at;
                v[i] = i < n ? *reinterpret_cast<const float*>(e) : 0.0f;
            }
            return v;
        };
        const int whole = sg.k / 16;
        int c = wave;
        for (; c + (kRowBatch - 1) * kRowWaves < whole; c += kRowBatch * kRowWaves) {
            f32x4 av[kRowBatch], bv[kRowBatch];
#pragma unroll
            for (int u = 0; u < kRowBatch; u++) {
                av[u] = load4(a + (c + u * kRowWaves) * 16, 4);
                bv[u] = operand(c + u * kRowWaves, 4);
            }
#pragma unroll
            for (int u = 0; u < kRowBatch; u++) add(av[u], bv[u]);
        }
#pragma unroll 1
        for (; c < whole; c += kRowWaves) add(load4(a + c * 16, 4), operand(c, 4));
        if (c == whole && sg.k % 16) {
            const int n = max(0, min(4, sg.k - c * 16 - kq));
            add(load4(a + c * 16, n), operand(c, n));
        }
    }
#pragma unroll
    for (int i = 0; i < 4; i++) red[wave][kq + i][l16] = (acc[0][i] + acc[1][i]) + (acc[2][i] + acc[3][i]);
    __syncthreads();
    if (tid >= 256) return;
    const int r = tid >> 4, jj = tid & 15;
    if (r > g.m - 1 - row0 || jj > p.n - 1 - j0) return;
    float w[kRowWaves];
#pragma unroll
    for (int i = 0; i < kRowWaves; i++) w[i] = red[i][r][jj];
    static_assert(kRowWaves == 8, "the sum below");
    const float sum = p.scale * (((w[0] + w[1]) + (w[2] + w[3])) + ((w[4] + w[5]) + (w[6] + w[7])));
    float* o = p.c + ((long)row0 + r) * p.n + j0 + jj;
    *o = g.acc ? *o + sum : sum;
}

int cdiv(int a, int b) { return (a - 1) / b + 1; }  // a > 0

// The tiles.  A step (32 k) of each, measured with one workgroup to a CU and
// with the chip full (power then holds the clock near 1.8 of 2.4 GHz):
//   256 x 128, 8 waves of 64 x 64, 1 workgroup to a CU:  1.7-1.8 / 2.3 us
//   128 x 128, 8 waves of 32 x 64, 1 to a CU:            0.93 / 1.15 us
//   64 x 64, 4 waves of 32 x 32, 3 to a CU:              0.45 / 1.2 us for three
// The larger the tile, the fewer times an operand is split and the fewer LDS
// bytes a product takes; the smaller, the better a small grid fills the CUs.
// (128 x 64 with two workgroups to a CU, 128 x 128 in steps of 16 k with two
// or three, and 256 x 256 were never the best.)
enum Tile { kTile256, kTile128, kTile64, kNumTiles };
constexpr int kTileM[kNumTiles] = {256, 128, 64}, kTileN[kNumTiles] = {128, 128, 64};
constexpr int kTileLogThreads[kNumTiles] = {9, 9, 8};
constexpr int kCus = 256;

// Modelled time of one launch, in us: rounds over the CUs of a workgroup's steps
// plus its first loads and stores.
double tile_time(Tile tile, long wgs, int steps) {
    const double rounds = (double)((wgs + kCus - 1) / kCus);
    if (tile == kTile256) return rounds * (steps * (wgs > kCus / 2 ? 2.1 : 1.8) + 5.0);
    if (tile == kTile128) return rounds * (steps * (wgs > kCus / 2 ? 1.1 : 0.95) + 4.0);
    return rounds < 2 ? steps * 0.45 + 3.0 : rounds * steps * 0.41 + 3.0;
}

template <bool AS, bool BS>
void launch_tile(const GemmArgs& g, Tile tile, bool far, int grid, hipStream_t st) {
    if (far)
        gemm_f32_kernel<AS, BS, 64, 64, 256, uint64_t><<<grid, 256, 0, st>>>(g);
    else if (tile == kTile256)
        gemm_f32_kernel<AS, BS, 256, 128, 512><<<grid, 512, 0, st>>>(g);
    else if (tile == kTile128)
        gemm_f32_kernel<AS, BS, 128, 128, 512><<<grid, 512, 0, st>>>(g);
    else
        gemm_f32_kernel<AS, BS, 64, 64, 256><<<grid, 256, 0, st>>>(g);
}

// Modelled time of the rows kernel: rounds over the CUs of a workgroup's batches.
double rows_time(const GemmF32& g) {
    long wgs = 0, longest = 0;
    for (int i = 0; i < g.npr; i++) {
        long k = 0;
        for (int s = 0; s < g.pr[i].nseg; s++) k += g.pr[i].seg[s].k;
        longest = std::max(longest, k);
        wgs += cdiv(g.pr[i].n, 16);
    }
    wgs *= cdiv(g.m, 16);
    return 2.5 + (double)((wgs + kCus - 1) / kCus) * 1.65 * (double)longest / (16 * kRowWaves * kRowBatch);
}

template <bool BS, typename Off = uint32_t>
hipError_t launch_rows(const GemmF32& in, hipStream_t st) {
    GemmArgs g{};
    int blocks = 0;
    for (int i = 0; i < in.npr; i++) {
        g.pr[i] = in.pr[i];
        blocks += cdiv(in.pr[i].n, 16);
    }
    // A launch has fewer than 2^32 threads along x and 2^16 blocks along y.
    constexpr int kRows = (1 << 27) - 16, kBlocksY = 65535;
    g.npr = in.npr, g.acc = in.acc;
    for (g.y0 = 0; g.y0 < blocks; g.y0 += kBlocksY)
        for (int m0 = 0; m0 < in.m; m0 += g.m) {
            g.m = std::min(kRows, in.m - m0);
            for (int i = 0; i < in.npr; i++) {
                for (int s = 0; s < in.pr[i].nseg; s++)
                    g.pr[i].seg[s].a = in.pr[i].seg[s].a + m0 * in.pr[i].seg[s].lda;
                g.pr[i].c = in.pr[i].c + (long)m0 * in.pr[i].n;
            }
            const dim3 grid(cdiv(g.m, 16), std::min(blocks - g.y0, kBlocksY));
            gemm_rows_kernel<BS, Off><<<grid, 64 * kRowWaves, 0, st>>>(g);
            const hipError_t e = hipGetLastError();
            if (e != hipSuccess) return e;
        }
    return hipSuccess;
}

}  // namespace

hipError_t launch_gemm_rows(const GemmF32& g, hipStream_t st) {
    if (g.npr == 0 || g.m == 0) return hipSuccess;
    if (!g.b_strided) return launch_rows<false>(g, st);
    long ldb = 0;
    for (int i = 0; i < g.npr; i++)
        for (int s = 0; s < g.pr[i].nseg; s++) ldb = std::max(ldb, g.pr[i].seg[s].ldb);
    return ldb < 1L << 26 ? launch_rows<true>(g, st) : launch_rows<true, uint64_t>(g, st);
}

hipError_t launch_gemm_f32(const GemmF32& in, float* ws, size_t ws_floats, hipStream_t st) {
    GemmArgs g{};
    int steps = 1;
    long cols = 0;
    bool far = false;  // offsets within a tile past 32 bits
    for (int i = 0; i < in.npr; i++) {
        const GemmProblem& p = g.pr[i] = in.pr[i];
        const int n = all_steps(p);
        if (n > steps) steps = n;
        cols += p.n;
        for (int s = 0; s < p.nseg; s++) {
            const long lda = in.a_strided ? 0 : p.seg[s].lda, ldb = in.b_strided ? 0 : p.seg[s].ldb;
            far |= (lda > ldb ? lda : ldb) >= 1L << 22;  // 256 rows of 4 bytes below 2^32
        }
    }
    g.npr = in.npr, g.m = in.m, g.acc = in.acc;
    // The tile and split of the least modelled time.  A split's partial sums
    // cost their pass through memory (4 bytes written and read, at 4 TB/s)
    // and a launch; a split is at least four steps.
    Tile tile = kTile64;
    int splits = 1;
    double best = -1.0;
    for (int ti = far ? kTile64 : kTile256; ti < kNumTiles; ti++) {
        int nt = 0;
        for (int i = 0; i < g.npr; i++) nt += cdiv(g.pr[i].n, kTileN[ti]);
        const long tiles = (long)cdiv(g.m, kTileM[ti]) * nt;
        for (int sp = 1; sp <= 32 && sp * 4 <= steps + 3; sp++) {
            const int per = cdiv(steps, sp);
            if (cdiv(steps, per) != sp) continue;
            if (sp > 1 && (size_t)(sp * cols) * g.m > ws_floats) break;
            if ((tiles * sp) << kTileLogThreads[ti] > UINT32_MAX) break;  // threads of a launch
            double t = tile_time((Tile)ti, tiles * sp, per);
            if (sp > 1) t += 4.0 + (2.0 * sp + 1.0) * cols * g.m * 4.0 / 4e6;
            if (best < 0 || t < best) best = t, tile = (Tile)ti, splits = sp;
        }
    }
    if (!in.a_strided && (best < 0 || rows_time(in) < best)) return launch_gemm_rows(in, st);
    if (best < 0) return hipErrorInvalidConfiguration;
    g.per = cdiv(steps, splits);
    splits = cdiv(steps, g.per);
    g.mt = cdiv(g.m, kTileM[tile]);
    for (int i = 0; i < g.npr; i++) g.nt += cdiv(g.pr[i].n, kTileN[tile]);
    g.part = splits > 1 ? ws : nullptr;
    // Neighbouring workgroups share an XCD's L2: run over n first where B is
    // the smaller operand (each XCD then reads all of it), else over m.
    g.n_inner = cols < g.m;
    const long grid = (long)g.mt * g.nt * splits;
    if (in.a_strided)
        launch_tile<true, true>(g, tile, far, (int)grid, st);
    else if (in.b_strided)
        launch_tile<false, true>(g, tile, far, (int)grid, st);
    else
        launch_tile<false, false>(g, tile, far, (int)grid, st);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || splits == 1) return e;
    int widest = 0;
    for (int i = 0; i < g.npr; i++) widest = g.pr[i].n > widest ? g.pr[i].n : widest;
    const long blocks = ((long)g.m * widest + 255) / 256;
    gemm_f32_reduce_kernel<<<dim3((unsigned)(blocks < 2048 ? blocks : 2048), g.npr), 256, 0, st>>>(g, splits, cols);
    return hipGetLastError();
}

}  // namespace cfattn
