// The fp32 attention forward's work unit on the bf16 matrix cores, every f32
// operand split into three bf16 pieces (split3.hpp), for head_dim 64 and 128.
// Included by attn_f32.hip, whose f32-MFMA unit of the same shape runs where a
// unit's result is not finite (the pieces of an infinite input, or of one that
// rounds to infinity, give NaN where f32 gives an infinity or a finite value).
//
// A tile of 32 keys is loaded in f32 to registers, one step ahead, split once
// by the workgroup and stored to LDS in the forms its products read, each
// operand a ds_read_b128 without bank conflicts:
//   rows (K): octet o of head dims of tile row r, for S^T = K Q^T;
//   cols (V): head dim d of an octet of tile rows, for O^T += V^T P^T: octet
//         2s + h holds the rows acc_row(8s + j, h), j = 0..7, which are the
//         accumulator registers 8s + j of lane half h, so P goes from the
//         accumulators of one product to an operand of the next.
// Each product keeps two sums, the leading pieces' and the other five's
// (split3.hpp: in one sum the small products lose low bits in one direction).
//
// Bound: the two waves of a SIMD issue 48 MFMAs (1536 cycles) and about 300
// VALU instructions (softmax, the pieces of P and of the tiles) a step; with f32
// MFMAs it was 64 of 64 cycles each.  B8 S2048 9/3 heads D64 0.362 -> 0.242 ms
// (0.235 without the split's power of two), B4 S1024 16/8 D128 0.180 -> 0.155.  (dK/dV the same way: its K and V pieces,
// four pairs of sums and scores take 460 registers, one wave to a SIMD, which
// hides nothing: 850 us where two waves of the f32 kernel take 720.)
#pragma once
#include "attn_params.hpp"
#include "cfattn_common.hpp"
#include "split3.hpp"

namespace cfattn {
namespace {

struct Op3 {
    bf16x8 p[3];
};
__device__ __forceinline__ Op3 op3(const Split8& s) {
    Op3 o;
#pragma unroll
    for (int i = 0; i < 3; i++) o.p[i] = __builtin_bit_cast(bf16x8, s.p[i]);
    return o;
}
// main += a0 b0, low += the other products.
__device__ __forceinline__ void mul3(const Op3& a, const Op3& b, f32x16& main, f32x16& low) {
    low = mfma32(a.p[2], b.p[0], low);
    low = mfma32(a.p[0], b.p[2], low);
    low = mfma32(a.p[1], b.p[1], low);
    low = mfma32(a.p[1], b.p[0], low);
    low = mfma32(a.p[0], b.p[1], low);
    main = mfma32(a.p[0], b.p[0], main);
}

// The rows form of a tile of 32 rows, 256 threads.
template <int DP>
struct RowsX3 {
    static constexpr int OCT = DP / 8, U = DP / 64, STEP = 256 / OCT;
    static constexpr int PITCH = 33;                 // eight lanes of a write: eight octets of one row
    static constexpr int PLANE = OCT * PITCH, SIZE = 3 * PLANE;  // 16-byte chunks
    float v[U][8];
    __device__ __forceinline__ void load(const float* __restrict__ g, long rs, int row0, int last, int tid) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int r = min(row0 + tid / OCT + STEP * u, last);
            const float* q = g + r * rs + tid % OCT * 8;
            const float4 a = *reinterpret_cast<const float4*>(q), b = *reinterpret_cast<const float4*>(q + 4);
            v[u][0] = a.x, v[u][1] = a.y, v[u][2] = a.z, v[u][3] = a.w;
            v[u][4] = b.x, v[u][5] = b.y, v[u][6] = b.z, v[u][7] = b.w;
        }
    }
    __device__ __forceinline__ void store(uint4* s, int tid) const {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const Split8 sp = split8_scaled(v[u]);
            uint4* d = s + tid % OCT * PITCH + tid / OCT + STEP * u;
#pragma unroll
            for (int i = 0; i < 3; i++) d[i * PLANE] = sp.p[i];
        }
    }
    // Head dims 16c + 8hh .. + 7 of tile row l32.
    __device__ __forceinline__ static Op3 read(const uint4* s, int c, int l32, int hh) {
        Op3 o;
#pragma unroll
        for (int i = 0; i < 3; i++)
            o.p[i] = __builtin_bit_cast(bf16x8, s[i * PLANE + (2 * c + hh) * PITCH + l32]);
        return o;
    }
};

// The cols form.
template <int DP>
struct ColsX3 {
    static constexpr int U = DP / 64, PITCH = DP + 1;
    static constexpr int PLANE = 4 * PITCH, SIZE = 3 * PLANE;
    float v[U][8];
    __device__ __forceinline__ void load(const float* __restrict__ g, long rs, int row0, int last, int tid) {
        const int o = wave_uniform(tid >> 6);
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int r = min(row0 + 16 * (o >> 1) + 8 * (j >> 2) + 4 * (o & 1) + (j & 3), last);
            const float* q = g + r * rs;
#pragma unroll
            for (int u = 0; u < U; u++) v[u][j] = q[(tid & 63) + 64 * u];
        }
    }
    __device__ __forceinline__ void store(uint4* s, int tid) const {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const Split8 sp = split8_scaled(v[u]);
            uint4* d = s + (tid >> 6) * PITCH + (tid & 63) + 64 * u;
#pragma unroll
            for (int i = 0; i < 3; i++) d[i * PLANE] = sp.p[i];
        }
    }
    // Tile rows acc_row(8s + j, hh), j = 0..7, of head dim db * 32 + l32.
    __device__ __forceinline__ static Op3 read(const uint4* s, int st, int db, int l32, int hh) {
        Op3 o;
#pragma unroll
        for (int i = 0; i < 3; i++)
            o.p[i] = __builtin_bit_cast(bf16x8, s[i * PLANE + (2 * st + hh) * PITCH + db * 32 + l32]);
        return o;
    }
};

// Head dims 16c + 8hh .. + 7 of a row in memory, c = 0 .. DP/16 - 1.
template <int DP>
__device__ __forceinline__ void row_ops(const float* __restrict__ row, int hh, Op3 (&o)[DP / 16]) {
#pragma unroll
    for (int c = 0; c < DP / 16; c++) {
        float v[8];
        const float4 a = *reinterpret_cast<const float4*>(row + 16 * c + 8 * hh);
        const float4 b = *reinterpret_cast<const float4*>(row + 16 * c + 8 * hh + 4);
        v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
        o[c] = op3(split8_scaled(v));
    }
}

// (m + log2(l)) ln 2, the larger sum rounded once.
__device__ __forceinline__ float lse_of(float m, float l) { return __builtin_fmaf(m, kLn2, __log2f(l) * kLn2); }

// LDS of a step is written and read; loads to registers stay in flight.
__device__ __forceinline__ void x3_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ bool any_odd(const f32x16& v) {
    bool odd = false;
#pragma unroll
    for (int r = 0; r < 16; r++) odd |= !(fabsf(v[r]) < INFINITY);
    return odd;
}

template <int DP>
struct FwdX3 {
    static constexpr int STAGE = RowsX3<DP>::SIZE + ColsX3<DP>::SIZE;
    static constexpr int LDS = 2 * STAGE;  // 16-byte chunks
};

// The forward's unit (fwd_f32_unit).  False, and nothing written, where some
// result of the workgroup is not finite.
template <int DP>
__device__ __forceinline__ bool fwd_x3_unit(const FwdParams& p, const F32Unit un, int rest, uint4* sm) {
    constexpr int BN = 32, NDB = DP / 32, NC = DP / 16, STAGE = FwdX3<DP>::STAGE;
    constexpr float kLazy = 8.0f;
    // K, Q and V are split scaled, P is not: a P below 2^-110 keeps an absolute
    // error of 2^-134, beside a sum of 2^-8 and more.
    const float sl2 = p.sl2 * (kSplitUnscale * kSplitUnscale);
    using Rows = RowsX3<DP>;
    using Cols = ColsX3<DP>;

    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63;
    const int l32 = lane & 31, hh = lane >> 5;

    const int TT = 32 * p.tpw;
    const int tile = un.tile;
    const int sub = rest % p.n_sub;
    rest /= p.n_sub;
    const int g = rest % p.nkv;
    const int b = rest / p.nkv;
    const int head = g * p.group + sub * p.hpw + wave % p.hpw;
    const int t_wave = tile * TT + (wave / p.hpw) * 32;
    const int tq = t_wave + l32;
    const int wg_end = min(p.seq, tile * TT + TT);
    const int kt_all = (wg_end + BN - 1) / BN;
    const int kt0 = un.ns > 1 ? un.split * p.ksplit : 0;
    const int n_kt = un.ns > 1 ? min(kt_all, kt0 + p.ksplit) : kt_all;
    const bool wave_active = t_wave < p.seq;
    const int wave_last = min(t_wave + 31, p.seq - 1);

    const long qrs = (long)p.nh * DP, kvrs = (long)p.nkv * DP;
    const float* kg = static_cast<const float*>(p.k) + (long)b * p.kv_bs + (long)g * DP;
    const float* vg = static_cast<const float*>(p.v) + (long)b * p.kv_bs + (long)g * DP;

    Rows rk;
    Cols rv;
    auto load = [&](int kt) {
        rk.load(kg, kvrs, kt * BN, p.seq - 1, tid);
        rv.load(vg, kvrs, kt * BN, p.seq - 1, tid);
    };
    auto store = [&](uint4* s) {
        rk.store(s, tid);
        rv.store(s + Rows::SIZE, tid);
    };
    load(kt0);
    Op3 qf[NC];
    row_ops<DP>(static_cast<const float*>(p.q) + (long)b * p.q_bs + (long)min(tq, p.seq - 1) * qrs + (long)head * DP,
                hh, qf);
    store(sm);
    load(kt0 + 1);
    x3_barrier();

    f32x16 oacc[NDB], olow[NDB];
#pragma unroll
    for (int i = 0; i < NDB; i++) oacc[i] = olow[i] = zero16();
    float m2 = -INFINITY, lsum = 0.0f;

    for (int kt = kt0; kt < n_kt; kt++) {
        const uint4* Ks = sm + ((kt - kt0) & 1) * STAGE;
        const uint4* Vs = Ks + Rows::SIZE;
        uint4* nxt = sm + ((kt - kt0 + 1) & 1) * STAGE;
        const int k0 = kt * BN;
        if (wave_active && k0 <= wave_last) {
            f32x16 sc = zero16(), sl = zero16();
#pragma unroll
            for (int c = 0; c < NC; c++) mul3(Rows::read(Ks, c, l32, hh), qf[c], sc, sl);
            store(nxt);
            load(kt + 2);
            sc += sl;
            float mx = -INFINITY;
            const bool masked = k0 + 31 > t_wave;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                if (masked && k0 + acc_row(r, hh) > tq) sc[r] = -INFINITY;
                mx = fmaxf(mx, sc[r]);
            }
            mx = max_halves(mx) * sl2;
            const float mnew = mx > m2 + kLazy ? mx : m2;
            if (__any(mnew != m2)) {
                const float alpha = __builtin_amdgcn_exp2f(m2 - mnew);
                lsum *= alpha;
#pragma unroll
                for (int i = 0; i < NDB; i++) oacc[i] *= alpha, olow[i] *= alpha;
                m2 = mnew;
            }
            float pr[16];
#pragma unroll
            for (int r = 0; r < 16; r++) {
                pr[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[r], sl2, -m2));
                lsum += pr[r];
            }
#pragma unroll
            for (int s = 0; s < 2; s++) {
                const Op3 pf = op3(split8(pr + 8 * s));
#pragma unroll
                for (int db = 0; db < NDB; db++) mul3(Cols::read(Vs, s, db, l32, hh), pf, oacc[db], olow[db]);
            }
        } else {
            store(nxt);
            load(kt + 2);
        }
        x3_barrier();
    }

    const float ltot = sum_halves(lsum);
    bool odd = false;
    if (wave_active && (un.ns == 1 || t_wave >= kt0 * BN)) {
        odd = !(ltot < INFINITY);
#pragma unroll
        for (int i = 0; i < NDB; i++) {
            oacc[i] += olow[i];
            odd |= any_odd(oacc[i]);
            oacc[i] *= kSplitUnscale;
        }
    }
    if (__syncthreads_or(odd)) return false;
    if (!wave_active || tq >= p.seq) return true;
    if (un.ns > 1) {
        if (t_wave < kt0 * BN) return true;
        const long row = (long)un.split * p.part_rows + ((long)b * p.nh + head) * p.seq + tq;
        float* prow = p.part + row * DP;
#pragma unroll
        for (int db = 0; db < NDB; db++)
#pragma unroll
            for (int rq = 0; rq < 4; rq++)
                *reinterpret_cast<float4*>(prow + db * 32 + rq * 8 + hh * 4) =
                    make_float4(oacc[db][rq * 4], oacc[db][rq * 4 + 1], oacc[db][rq * 4 + 2], oacc[db][rq * 4 + 3]);
        if (hh == 0) p.part_ml[row] = make_float2(m2, ltot);
        return true;
    }
    const float inv = 1.0f / ltot;
    float* orow = p.o + (long)b * p.q_bs + (long)tq * qrs + (long)head * DP;
#pragma unroll
    for (int db = 0; db < NDB; db++)
#pragma unroll
        for (int rq = 0; rq < 4; rq++)
            *reinterpret_cast<float4*>(orow + db * 32 + rq * 8 + hh * 4) =
                make_float4(oacc[db][rq * 4] * inv, oacc[db][rq * 4 + 1] * inv, oacc[db][rq * 4 + 2] * inv,
                            oacc[db][rq * 4 + 3] * inv);
    if (hh == 0) p.lse[((long)b * p.nh + head) * p.seq + tq] = lse_of(m2, ltot);
    return true;
}

}  // namespace
}  // namespace cfattn
