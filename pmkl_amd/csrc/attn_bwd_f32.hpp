// fp32 backward of the attention output (gfx950, fp32 MFMA): the reference's
// algorithm (fused_self_attention.cpp:66-135) in the same two passes and with
// the same workspace as the 16-bit kernels (attn_bwd_kernels.hpp).
//
//   attn_bwd_f32_dq_kernel    a workgroup owns 32 query rows; its four waves
//                             take the key tiles (of 32) w, w + 4, ... .  Per
//                             tile dP^T = V dout^T and S^T = K Q^T, then P and
//                             dS in the accumulator registers, which are the B
//                             operand of dQ^T += K^T dS^T as they stand.
//                             Writes lse2_i and D_i to the workspace.
//   attn_bwd_f32_dkdv_kernel  a workgroup owns 32 key rows, its waves split
//                             the query tiles: dP = dout V^T, S = Q K^T,
//                             dK^T += Q^T dS, dV^T += dout^T P.
//
// Bound: v_mfma_f32_32x32x2f32 (attn_f32.hpp).  Each wave stages its own
// tiles, V then K (dout, Q, dout) through one LDS tile and one set of staging
// registers, the next one in flight under the products of the one before: the
// waves of a SIMD (4 / 3 / 1 at head_dim 32 / 64 / 128; at 64 the dK/dV pass
// spills 2-3 registers for its third) drift apart and one's
// exponentials and LDS writes pass under the other's MFMAs.  32 owned rows and
// a four-way split give many short, equal workgroups: the chains of dependent
// tiles are a quarter as long as with one wave per row block, which bounds the
// small shapes, and the long causal rows start first.
// Hidden keys and queries must add nothing, whatever they hold.  In the products
// over a whole tile their weight is 0, and 0 times an infinity or a NaN is a
// NaN: a row whose sum is not finite is computed again, over its visible keys or
// queries alone (attn_bwd_f32_rows.hpp).  The check of the sums costs 1-2% where
// a workgroup has one round of tiles (1,024 heads of S128 D64 causal, whole
// call, 171.8 / 176.2 us) and nothing from S1024 on; masking P, dS and the tiles
// themselves cost 10-18% at every causal size.
// Measured against one wave per owned row on the vector ALUs (dq / dkdv, us):
// B4 H16 S1024 D64 causal 3,141 / 3,303 -> 132 / 180 (96 and 128 fp32 MFMAs per
// tile: 84 and 112 us at the MFMA's 154 TFLOP/s), B2 H16 S128 D128 90 / 123 ->
// 14 / 16 (one tile per wave: latency).
#pragma once

#include "attn_bwd_f32_rows.hpp"
#include "attn_f32.hpp"

namespace pmkl_amd {

template <int D, bool CAUSAL>
__global__ __launch_bounds__(kF32Threads, D >= 128 ? 1 : D >= 64 ? 3 : 4) void attn_bwd_f32_dq_kernel(BwdParams p) {
    using TL = F32Tile<D>;
    constexpr int NW = kF32Waves, BN = kF32Rows, NDB = D / 32;
    __shared__ __attribute__((aligned(16))) float smem[NW][TL::FLOATS];   // each wave's V or K tile
    __shared__ __attribute__((aligned(16))) float dtile[TL::FLOATS];      // dout of the owned rows
    __shared__ float dvec[NW][BN];   // D_i, or each wave's part of it

    const int lane = threadIdx.x & 63;
    const int hi = lane >> 5, col = lane & 31;
    const int bh = blockIdx.x % p.BH;
    const int qt = CAUSAL ? p.n_qtiles - 1 - (int)blockIdx.x / p.BH : (int)blockIdx.x / p.BH;   // longest first
    const int wave = f32_wave(bh, qt);
    const int S = p.S;
    const float *kg = bwd_head<const float>(p, p.k, BK, bh);
    const float *vg = bwd_head<const float>(p, p.v, BV, bh);
    const int kss = p.ss[BK], vss = p.ss[BV];
    const int q0 = qt * BN;
    const int qi = q0 + col;                  // this lane's query row
    const int qrow = min(qi, S - 1);
    const int lim = CAUSAL ? qrow : S - 1;    // its last visible key
    const int nt = (CAUSAL ? min(q0 + BN - 1, S - 1) : S - 1) / BN + 1;

    float *tile = smem[wave];
    F32Stage<D, 64> st;
    auto load_v = [&](int kt) __attribute__((always_inline)) { st.load(vg, kt * BN, kt < nt ? S : 0, vss, lane); };

    // The owned rows, loaded once by the whole workgroup and handed to the
    // waves through LDS; D_i = <dout_i, o_i> from the same
    // loads where the caller passes O.
    F32Stage<D, kF32Threads> qst, dst, ost;
    qst.load(bwd_head<const float>(p, p.q, BQ, bh), q0, S, p.ss[BQ], threadIdx.x);
    dst.load(bwd_head<const float>(p, p.dout, BDOUT, bh), q0, S, p.ss[BDOUT], threadIdx.x);
    if (p.o != nullptr) ost.load(bwd_head<const float>(p, p.o, BO, bh), q0, S, p.ss[BO], threadIdx.x);
    const float m_i = bwd_load_ml<float>(p.m, (int64_t)bh * S + qrow, true);
    const float l_i = bwd_load_ml<float>(p.l, (int64_t)bh * S + qrow, true);
    load_v(wave);
    const float lse2 = m_i * 1.4426950408889634f + __log2f(l_i);
    const float c = p.scale_log2;
    qst.store(smem[0], threadIdx.x);
    dst.store(dtile, threadIdx.x);
    if (p.o != nullptr) {
#pragma unroll
        for (int j = 0; j < decltype(ost)::LOADS; ++j) {
            float part = 0.f;
#pragma unroll
            for (int e = 0; e < 4; ++e) part = __builtin_fmaf(ost.reg[j][e], dst.reg[j][e], part);
#pragma unroll
            for (int o = TL::CPR / 2; o >= 1; o >>= 1) part += __shfl_xor(part, o, 64);   // the row's chunks
            if (threadIdx.x % TL::CPR == 0) dvec[0][threadIdx.x / TL::CPR + j * decltype(ost)::STEP] = part;
        }
    }
    __syncthreads();
    f32x4_t qf[D / 8];
    f32_rows<D>(qf, smem[0], col, hi);
    float drow = p.o != nullptr ? dvec[0][col] : 0.f;
    __syncthreads();

    // This wave's tiles; work(P, dP) gets the probabilities and dP of a tile.
    // The wave's own LDS: its reads of the previous tile are issued before
    // the writes of the next, and one wave's LDS operations run in order, so
    // neither side needs a barrier.  On return the first tile is in flight
    // again where another loop follows.
    auto tiles = [&](auto last_c, auto &&work) __attribute__((always_inline)) {
        for (int kt = wave; kt < nt; kt += NW) {
            asm volatile("" ::: "memory");
            st.store(tile, lane);
            asm volatile("" ::: "memory");
            st.load(kg, kt * BN, S, kss, lane);
            f32x16_t s{}, dp{};
            f32_scores<D>(tile, dtile, dp, col, hi);
            asm volatile("" ::: "memory");
            st.store(tile, lane);
            asm volatile("" ::: "memory");
            load_v(decltype(last_c)::value || kt + NW < nt ? kt + NW : wave);
            f32_scores<D>(tile, qf, s, col, hi);
            const int d = lim - kt * BN - 4 * hi;   // f32_acc_row up to d is visible
            if (kt * BN + BN - 1 > (CAUSAL ? q0 : S - 1)) {
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    s[r] = f32_acc_row(r) <= d ? fast_exp2(__builtin_fmaf(s[r], c, -lse2)) : 0.f;
            } else {
#pragma unroll
                for (int r = 0; r < 16; ++r) s[r] = fast_exp2(__builtin_fmaf(s[r], c, -lse2));
            }
            work(s, dp);
        }
    };

    if (p.o == nullptr) {   // D_i = sum_j P_ij dP_ij over the keys
        float part = 0.f;
        tiles(std::false_type{}, [&](const f32x16_t &pr, const f32x16_t &dp) __attribute__((always_inline)) {
#pragma unroll
            for (int r = 0; r < 16; ++r) part = __builtin_fmaf(pr[r], dp[r], part);
        });
        part = half_sum(part);
        if (hi == 0) dvec[wave][col] = part;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < NW; ++w) drow += dvec[w][col];   // waves without tiles wrote 0
    }
    if (wave == 0 && hi == 0 && qi < S) {
        p.lse2[(int64_t)bh * S + qi] = lse2;
        p.drow[(int64_t)bh * S + qi] = drow;
    }

    f32x16_t acc[NDB];   // dQ^T (head_dim x owned rows), this wave's tiles
#pragma unroll
    for (int db = 0; db < NDB; ++db) acc[db] = f32x16_t{};
    tiles(std::true_type{}, [&](f32x16_t &pr, const f32x16_t &dp) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 16; ++r) pr[r] *= dp[r] - drow;   // dS
        f32_accumulate<D>(tile, pr, acc, col, hi);
    });

    asm volatile("" ::: "memory");
    if (wave < nt) f32_put<D>(tile, acc, col, hi);
    __syncthreads();
    f32_combine<D>(smem[0], TL::FLOATS, min(NW, nt), p.scale, bwd_head<float>(p, p.dq, BDQ, bh), q0, S, p.ss[BDQ],
                   [&](int row) { f32_dq_row<D, CAUSAL, true>(p, bh, row); });
}

template <int D, bool CAUSAL>
__global__ __launch_bounds__(kF32Threads, D >= 128 ? 1 : D >= 64 ? 3 : 4) void attn_bwd_f32_dkdv_kernel(BwdParams p) {
    using TL = F32Tile<D>;
    constexpr int NW = kF32Waves, BN = kF32Rows, NDB = D / 32;
    __shared__ __attribute__((aligned(16))) float smem[NW][TL::FLOATS];   // each wave's dout or Q tile
    __shared__ __attribute__((aligned(16))) float own[2][TL::FLOATS];     // the owned K and V rows
    __shared__ __attribute__((aligned(16))) float svec[NW][2][BN];        // lse2, D_i of its rows

    const int lane = threadIdx.x & 63;
    const int hi = lane >> 5, col = lane & 31;
    const int bh = blockIdx.x % p.BH;
    const int kt = (int)blockIdx.x / p.BH;   // the first keys have the most queries (causal)
    const int wave = f32_wave(bh, kt);
    const int S = p.S;
    const float *qg = bwd_head<const float>(p, p.q, BQ, bh);
    const float *dog = bwd_head<const float>(p, p.dout, BDOUT, bh);
    const int qss = p.ss[BQ], doss = p.ss[BDOUT];
    const int k0 = kt * BN;
    const int kj = k0 + col;                 // this lane's key row
    const int t0 = CAUSAL ? kt : 0;          // first query tile with a visible query
    const int nq = (S - 1) / BN + 1;

    float *tile = smem[wave], *vec = svec[wave][0];
    F32Stage<D, 64> st;
    float vreg;   // lanes 0-31: lse2, 32-63: D_i of the tile's rows
    const float *vecg = (hi ? p.drow : p.lse2) + (int64_t)bh * S;
    auto load_do = [&](int t) __attribute__((always_inline)) { st.load(dog, t * BN, t < nq ? S : 0, doss, lane); };
    auto load_vec = [&](int t) __attribute__((always_inline)) {
        // rows past S: lse2 = +inf and zero Q, dout rows give P = 0, dS = 0
        vreg = t * BN + col < S ? vecg[t * BN + col] : (hi ? 0.f : INFINITY);
    };

    {
        F32Stage<D, kF32Threads> kst, vst;
        kst.load(bwd_head<const float>(p, p.k, BK, bh), k0, S, p.ss[BK], threadIdx.x);
        vst.load(bwd_head<const float>(p, p.v, BV, bh), k0, S, p.ss[BV], threadIdx.x);
        load_do(t0 + wave);
        load_vec(t0 + wave);
        kst.store(own[0], threadIdx.x);
        vst.store(own[1], threadIdx.x);
        __syncthreads();
    }
    const float c = p.scale_log2;

    f32x16_t dk_acc[NDB], dv_acc[NDB];   // dK^T, dV^T (head_dim x owned keys), this wave's tiles
#pragma unroll
    for (int db = 0; db < NDB; ++db) dk_acc[db] = dv_acc[db] = f32x16_t{};
    for (int t = t0 + wave; t < nq; t += NW) {
        asm volatile("" ::: "memory");
        st.store(tile, lane);
        vec[lane] = vreg;
        asm volatile("" ::: "memory");
        st.load(qg, t * BN, S, qss, lane);
        load_vec(t + NW);
        f32x16_t s{}, dp{};
        f32_scores<D>(tile, own[1], dp, col, hi);
        asm volatile("" ::: "memory");
        st.store(tile, lane);
        asm volatile("" ::: "memory");
        load_do(t);
        f32_scores<D>(tile, own[0], s, col, hi);
        const int d = kj - t * BN - 4 * hi;   // causal: f32_acc_row from d on sees the key
        const bool mask = CAUSAL && t == t0;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const f32x4_t l4 = *(const f32x4_t *)(vec + 8 * g + 4 * hi), d4 = *(const f32x4_t *)(vec + BN + 8 * g + 4 * hi);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int r = 4 * g + e;
                const float pv = fast_exp2(__builtin_fmaf(s[r], c, -l4[e]));
                s[r] = !mask || f32_acc_row(r) >= d ? pv : 0.f;
                dp[r] = s[r] * (dp[r] - d4[e]);
            }
        }
        f32_accumulate<D>(tile, dp, dk_acc, col, hi);
        asm volatile("" ::: "memory");
        st.store(tile, lane);
        asm volatile("" ::: "memory");
        load_do(t + NW);
        f32_accumulate<D>(tile, s, dv_acc, col, hi);
    }

    // dK, then dV, through the waves' tiles
    const int n = min(NW, nq - t0);
    asm volatile("" ::: "memory");
    if (t0 + wave < nq) f32_put<D>(tile, dk_acc, col, hi);
    __syncthreads();
    auto redo = [&](int row) { f32_dkdv_row<D, CAUSAL, true>(p, bh, row); };
    f32_combine<D>(smem[0], TL::FLOATS, n, p.scale, bwd_head<float>(p, p.dk, BDK, bh), k0, S, p.ss[BDK], redo);
    __syncthreads();
    if (t0 + wave < nq) f32_put<D>(tile, dv_acc, col, hi);
    __syncthreads();
    f32_combine<D>(smem[0], TL::FLOATS, n, 1.f, bwd_head<float>(p, p.dv, BDV, bh), k0, S, p.ss[BDV], redo);
}

}  // namespace pmkl_amd
