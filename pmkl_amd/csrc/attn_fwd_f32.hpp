// fp32 forward with split keys (gfx950): one workgroup per (head, 32-row query
// block); its four waves take the block's key tiles w, w + 4, ..., each staging
// its own tiles in LDS (no workgroup barrier in the loop), then the partial
// (O, m, l) of the waves are combined by the log-sum-exp rule.  Per tile the
// arithmetic of attn_fwd_f32_kernel: v_mfma_f32_32x32x2f32, exact rescale.
// K and V take turns in one LDS tile and one set of staging registers, V in
// flight under the scores, the next K under the P V product: half the LDS and
// registers, so 4 / 3 / 2 waves per SIMD at head_dim 32 / 64 / 128 (with a tile
// each, 3 / 2 / 1: B1 H32 S4096 D128 causal 1,406 us against 1,109, B1 H16 S4096
// D64 307 against 286; 124 and 120 of the 154 TFLOP/s that the fp32 MFMA
// sustains).  A 32-row workgroup per block instead of 128 rows on shared tiles:
// B4 H16 S1024 D64 126 -> 96 us.
#pragma once

#include "attn_f32.hpp"

namespace pmkl_amd {

template <int D, bool CAUSAL>
__global__ __launch_bounds__(kF32Threads, D >= 128 ? 2 : D >= 64 ? 3 : 4) void attn_fwd_f32_split_kernel(AttnParams p) {
    using TL = F32Tile<D>;
    constexpr int NW = kF32Waves, BN = kF32Rows, NDB = D / 32;
    __shared__ __attribute__((aligned(16))) float smem[NW][TL::FLOATS];   // each wave's K or V tile
    __shared__ float mlvec[NW][2][BN];                                    // its m and l

    const int lane = threadIdx.x & 63;
    const int hi = lane >> 5, col = lane & 31;
    const int bh = blockIdx.x % p.BH;
    const int qt = CAUSAL ? p.n_qtiles - 1 - (int)blockIdx.x / p.BH : (int)blockIdx.x / p.BH;   // longest first
    const int wave = f32_wave(bh, qt);
    const int b = bh / p.H, h = bh - b * p.H;
    const int S = p.S;
    const float *kg = (const float *)p.k + b * p.k_sb + h * p.k_sh;
    const float *vg = (const float *)p.v + b * p.v_sb + h * p.v_sh;
    const int kss = (int)p.k_ss, vss = (int)p.v_ss;   // a 64-row tile spans < 2 GiB (checked)
    const int q0 = qt * BN;
    const int qi = q0 + col;                            // this lane's query row
    const int lim = CAUSAL ? min(qi, S - 1) : S - 1;    // its last visible key
    const int nt = (CAUSAL ? min(q0 + BN - 1, S - 1) : S - 1) / BN + 1;
    const float c = p.scale_log2;

    float *tile = smem[wave];
    F32Stage<D, 64> st;
    // the owned rows, loaded once by the workgroup, through the first wave's tile
    f32x4_t qf[D / 8];
    {
        F32Stage<D, kF32Threads> qst;
        qst.load((const float *)p.q + b * p.q_sb + h * p.q_sh, q0, S, (int)p.q_ss, threadIdx.x);
        st.load(kg, wave * BN, wave < nt ? S : 0, kss, lane);
        qst.store(smem[0], threadIdx.x);
        __syncthreads();
        f32_rows<D>(qf, smem[0], col, hi);
        __syncthreads();
    }

    f32x16_t acc[NDB];   // O^T (head_dim x owned rows) of this wave's tiles, relative to m_run
#pragma unroll
    for (int db = 0; db < NDB; ++db) acc[db] = f32x16_t{};
    float m_run = -INFINITY, l_run = 0.f;   // raw dot-product units; l_run of this lane half's keys
    for (int kt = wave; kt < nt; kt += NW) {
        // The wave's own LDS: its reads of the tile before are issued before
        // these writes, and one wave's LDS operations run in order, so neither
        // side needs a barrier.
        asm volatile("" ::: "memory");
        st.store(tile, lane);
        asm volatile("" ::: "memory");
        st.load(vg, kt * BN, S, vss, lane);
        f32x16_t s{};
        f32_scores<D>(tile, qf, s, col, hi);
        const int d = lim - kt * BN - 4 * hi;   // f32_acc_row up to d is visible
        if (kt * BN + BN - 1 > (CAUSAL ? q0 : S - 1)) {
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (f32_acc_row(r) > d) s[r] = -INFINITY;
        }
        float mx = s[0];
#pragma unroll
        for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
        mx = half_max(mx);
        if (__builtin_amdgcn_ballot_w64(mx > m_run)) {   // else alpha is 1 for every row
            const float m_new = fmaxf(m_run, mx);
            // 0 on the wave's first tile, also for a row of -inf scores
            const float alpha = fast_exp2((m_run - (m_new == -INFINITY ? 0.f : m_new)) * c);
            m_run = m_new;
            l_run *= alpha;
#pragma unroll
            for (int db = 0; db < NDB; ++db) acc[db] *= alpha;
        }
        const float moff = m_run == -INFINITY ? 0.f : -m_run * c;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            s[r] = fast_exp2(__builtin_fmaf(s[r], c, moff));
            l_run += s[r];
        }
        asm volatile("" ::: "memory");
        st.store(tile, lane);
        asm volatile("" ::: "memory");
        st.load(kg, (kt + NW) * BN, kt + NW < nt ? S : 0, kss, lane);
        f32_accumulate<D>(tile, s, acc, col, hi);
    }

    // O = sum_w 2^((m_w - M) c) O_w / l over the waves, M = max_w m_w and l the
    // sum of theirs likewise: each wave scales its own O, the scaled ones are
    // added.  A wave without tiles holds m = -inf and weighs 0; a row of -inf
    // scores alone has M = -inf, and l and O NaN as in the reference.
    const float l_w = half_sum(l_run);
    if (hi == 0) {
        mlvec[wave][0][col] = m_run;
        mlvec[wave][1][col] = l_w;
    }
    __syncthreads();
    float M = -INFINITY, l_tot = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) M = fmaxf(M, mlvec[w][0][col]);
#pragma unroll
    for (int w = 0; w < NW; ++w) l_tot += fast_exp2((mlvec[w][0][col] - M) * c) * mlvec[w][1][col];
    const float f = fast_exp2((m_run - M) * c) * (1.0f / l_tot);
    if (wave < nt) {
#pragma unroll
        for (int db = 0; db < NDB; ++db) acc[db] *= f;
        f32_put<D>(tile, acc, col, hi);
    }
    if (wave == 0 && hi == 0 && qi < S) {
        ((float *)p.m)[(int64_t)bh * S + qi] = M * p.scale;
        ((float *)p.l)[(int64_t)bh * S + qi] = l_tot;
    }
    __syncthreads();
    f32_combine<D>(smem[0], TL::FLOATS, min(NW, nt), 1.f, (float *)p.o + b * p.o_sb + h * p.o_sh, q0, S,
                   (int)p.o_ss);
}

}  // namespace pmkl_amd
