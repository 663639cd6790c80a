// Building blocks of the fp32 kernels (gfx950): 32-row tiles in LDS and the
// products over them on v_mfma_f32_32x32x2f32.
//
// The fp32 MFMA takes 64 clocks for one float per lane of each operand, so the
// kernels are bound by the matrix cores and move few LDS bytes per clock: a
// workgroup owns 32 rows, its four waves split the streamed 32-row tiles and
// each stages its own in LDS, with no workgroup barrier in the loop; the
// waves' partial sums are added through LDS at the end.
#pragma once

#include "attn_fwd_kernels.hpp"

namespace pmkl_amd {

constexpr int kF32Rows = 32;    // owned rows per workgroup = streamed rows per tile
constexpr int kF32Waves = 4;    // each takes a share of the streamed tiles
constexpr int kF32Threads = 64 * kF32Waves;

// This wave's place in the split, 0 .. 3 (wave w takes the tiles w, w + 4, ...).
// Rotated by block, or the SIMD that runs every workgroup's first wave would get
// every workgroup's odd tile.
__device__ __forceinline__ int f32_wave(int bh, int row_block) {
    return ((__builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) + row_block + (bh >> 3)) & (kF32Waves - 1));
}

// A 32-row tile of a [S, D] float matrix in LDS: rows padded by 16 bytes, so
// that 16 lanes reading the same 16-byte chunk of 16 rows hit 64 banks.
template <int D>
struct F32Tile {
    static constexpr int LD = D + 4;
    static constexpr int FLOATS = kF32Rows * LD;
    static constexpr int CPR = D / 4;   // 16-byte chunks per row
};

// A tile on its way from memory to LDS, carried by THREADS threads: one wave
// (the streamed tiles) or the whole workgroup (the owned rows).  Thread t
// holds chunk t % CPR of rows t / CPR + j THREADS / CPR: whole rows per load
// instruction.  (Each lane loading its own row instead touches 32 lines with
// every instruction: the forward of B2 H16 S128 D128 17 us instead of 11.)
template <int D, int THREADS>
struct F32Stage {
    using TL = F32Tile<D>;
    static constexpr int LOADS = kF32Rows * TL::CPR / THREADS;
    static constexpr int STEP = THREADS / TL::CPR;   // rows per load
    f32x4_t reg[LOADS];

    // Rows r0 .. r0 + 31 of base (row stride ss elements); rows past S read as
    // zero, without touching memory where r0 >= S.  Called unconditionally (a
    // load under a branch costs a second register set).
    __device__ __forceinline__ void load(const float *base, int r0, int S, int ss, int t) {
        const int rows = min(kF32Rows, S - r0);
        const auto r = __builtin_amdgcn_make_buffer_rsrc((void *)(base + (int64_t)r0 * ss), (short)0,
                                                         rows > 0 ? ((rows - 1) * ss + D) * 4 : 0, 0x00020000);
        // one running lane offset, opaque to the compiler, which else keeps an
        // offset per load (across the loop, too) and spills
        int off = ((t / TL::CPR) * ss + 4 * (t % TL::CPR)) * 4;
#pragma unroll
        for (int j = 0; j < LOADS; ++j) {
            asm volatile("" : "+v"(off));
            reg[j] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
            off += STEP * ss * 4;
        }
    }
    __device__ __forceinline__ void store(float *lds, int t) const {
        float *p = lds + (t / TL::CPR) * TL::LD + 4 * (t % TL::CPR);
#pragma unroll
        for (int j = 0; j < LOADS; ++j) *(f32x4_t *)(p + j * STEP * TL::LD) = reg[j];
    }
};

// Fragments of the products over head_dim: lane (row col, half hi) holds
// elements 8x + 4 hi .. + 3 of its row in f[x]; MFMA e of chunk x contracts
// elements 8x + e (half 0) and 8x + 4 + e (half 1).
template <int D>
__device__ __forceinline__ void f32_rows(f32x4_t (&f)[D / 8], const float *tile, int col, int hi) {
#pragma unroll
    for (int x = 0; x < D / 8; ++x) f[x] = *(const f32x4_t *)(tile + col * F32Tile<D>::LD + 8 * x + 4 * hi);
}

// s += A f^T for the 32-row tile A in LDS, fragments read one chunk (4 MFMAs)
// ahead; left to itself the compiler reads each right before its MFMA.
template <int D>
__device__ __forceinline__ void f32_scores(const float *A, const f32x4_t (&f)[D / 8], f32x16_t &s, int col, int hi) {
    const float *ar = A + col * F32Tile<D>::LD + 4 * hi;
    f32x4_t a = *(const f32x4_t *)ar;
#pragma unroll
    for (int x = 0; x < D / 8; ++x) {
        f32x4_t an = a;
        if (x + 1 < D / 8) an = *(const f32x4_t *)(ar + 8 * (x + 1));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], f[x][e], s, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        a = an;
    }
}

// The same with the owned rows F in LDS too.
template <int D>
__device__ __forceinline__ void f32_scores(const float *A, const float *F, f32x16_t &s, int col, int hi) {
    const float *ar = A + col * F32Tile<D>::LD + 4 * hi, *fr = F + col * F32Tile<D>::LD + 4 * hi;
    f32x4_t a = *(const f32x4_t *)ar, f = *(const f32x4_t *)fr;
#pragma unroll
    for (int x = 0; x < D / 8; ++x) {
        f32x4_t an = a, fn = f;
        if (x + 1 < D / 8) {
            an = *(const f32x4_t *)(ar + 8 * (x + 1));
            fn = *(const f32x4_t *)(fr + 8 * (x + 1));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], f[e], s, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        a = an;
        f = fn;
    }
}

// Register r of lane half hi holds streamed row f32_acc_row(r) + 4 hi (of 32)
// in the 32x32 accumulator layout; the same row is contracted by MFMA r of the
// products over the streamed rows.
__device__ __forceinline__ constexpr int f32_acc_row(int r) { return 8 * (r >> 2) + (r & 3); }

// acc^T (head_dim x owned rows) += tile^T w, w in accumulator layout; the
// fragments of the next G streamed rows (at least four MFMAs' worth) are read
// while those before are multiplied.
template <int D>
__device__ __forceinline__ void f32_accumulate(const float *tile, const f32x16_t &w, f32x16_t (&acc)[D / 32], int col,
                                               int hi) {
    constexpr int NDB = D / 32, G = NDB == 1 ? 4 : 2;
    int off = 4 * hi * F32Tile<D>::LD + col;
    asm volatile("" : "+v"(off));   // else the pairwise reads' base addresses (up to 32) are kept across the loop
    const float *base = tile + off;
    float a[2][G][NDB];
    auto read = [&](int g) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < G; ++e)
#pragma unroll
            for (int db = 0; db < NDB; ++db)
                a[g & 1][e][db] = base[f32_acc_row(G * g + e) * F32Tile<D>::LD + 32 * db];
    };
    read(0);
#pragma unroll
    for (int g = 0; g < 16 / G; ++g) {
        if (g + 1 < 16 / G) read(g + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < G; ++e)
#pragma unroll
            for (int db = 0; db < NDB; ++db)
                acc[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[g & 1][e][db], w[G * g + e], acc[db], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// One wave's partial of the owned rows to LDS, [row][head_dim] with the tile's row length.
template <int D>
__device__ __forceinline__ void f32_put(float *part, const f32x16_t (&acc)[D / 32], int col, int hi) {
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const f32x4_t w = {acc[db][4 * g], acc[db][4 * g + 1], acc[db][4 * g + 2], acc[db][4 * g + 3]};
            *(f32x4_t *)(part + col * F32Tile<D>::LD + 32 * db + 8 * g + 4 * hi) = w;
        }
}

// Adds the partials of the first n waves (wave_floats apart) and stores
// scale times the sum to rows r0 .. of out, whole rows at a time.  Then
// redo(row) for each row whose sum is not finite, by the one wave that stored
// it (nothing is checked with the default).
struct F32Keep {};
template <int D, typename Redo = F32Keep>
__device__ __forceinline__ void f32_combine(const float *part, int wave_floats, int n, float scale, float *out,
                                                int r0, int S, int ss, Redo redo = {}) {
    using TL = F32Tile<D>;
    constexpr int THREADS = kF32Threads, SLOTS = kF32Rows * TL::CPR / THREADS;
    const int ch = threadIdx.x % TL::CPR;
    auto row_of = [](int i) __attribute__((always_inline)) { return (i * THREADS + (int)threadIdx.x) / TL::CPR; };
    auto sum_of = [&](int i) __attribute__((always_inline)) {
        f32x4_t sum = *(const f32x4_t *)(part + row_of(i) * TL::LD + 4 * ch);
        for (int w = 1; w < n; ++w) sum += *(const f32x4_t *)(part + w * wave_floats + row_of(i) * TL::LD + 4 * ch);
        return sum * scale;
    };
    auto add_zeros = [](float z, const f32x4_t &x) __attribute__((always_inline)) {   // NaN if x is not finite
#pragma unroll
        for (int e = 0; e < 4; ++e) z = __builtin_fmaf(x[e], 0.f, z);
        return z;
    };
    float z = 0.f;
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) {
        const f32x4_t sum = sum_of(i);
        if constexpr (!std::is_same_v<Redo, F32Keep>) z = add_zeros(z, sum);
        if (r0 + row_of(i) < S) *(f32x4_t *)(out + (int64_t)(r0 + row_of(i)) * ss + 4 * ch) = sum;
    }
    if constexpr (!std::is_same_v<Redo, F32Keep>) {
        if (__builtin_amdgcn_ballot_w64(z != z) == 0) return;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");   // other lanes of the wave store the rows again
        constexpr uint64_t lanes = (1ull << TL::CPR) - 1;    // a row's, from its first
#pragma unroll 1
        for (int i = 0; i < SLOTS; ++i) {
            const float zi = add_zeros(0.f, sum_of(i));
            const uint64_t bad = __builtin_amdgcn_ballot_w64(zi != zi && r0 + row_of(i) < S);
            const int first = __builtin_amdgcn_readfirstlane(row_of(i));
#pragma unroll 1
            for (int w = 0; w < 64 / TL::CPR; ++w)
                if (bad >> (w * TL::CPR) & lanes) redo(r0 + first + w);
        }
    }
}

}  // namespace pmkl_amd
