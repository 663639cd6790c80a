// gfx950 row softmax / log-softmax over rows of up to 1024 elements.
//
// Replaces the kernel body of pmkl::norm::warp_softmax_forward,
// warp_softmax_forward_impl (pmkl/norm/warp_softmax.h:74-157).  Per row r
// (elements x_i = src[r*stride + i], i < n), in fp32:
//   m = max_i x_i                                   (:108-118)
//   s = sum_i exp(x_i - m)                          (:120-133)
//   softmax:     y_i = exp(x_i - m) / s, NaN if s == 0   (:147-150)
//   log-softmax: y_i = (x_i - m) - log(s)                 (:140, :146)
//
// Work layout.  A row is owned by a group of G = 2^g lanes of one wave64
// (G = 1 .. 64, so one wave holds 64/G rows; the reference fixes a 32-lane
// warp and two rows per warp for rows of <= 128 elements).  Lane j of a group
// holds C chunks of W consecutive elements, chunk c starting at element
// (c*G + j)*W: one load instruction of the wave reads G*W consecutive
// elements of each of its rows.  W is 16 bytes of the input type (4 fp32 or 8
// fp16/bf16 elements): aligned vectors when the row length, the stride and both
// base pointers allow them, else (RAGGED) vectors at element alignment; 1 for
// rows shorter than a vector.  The whole row sits in registers between the
// load and the store, so src is read once and dst written once (2 passes of
// HBM traffic in total: the aligned form is HBM-bound, 131,072 x 1,024 fp32
// 166 us and bf16 80 us, 6.5 and 6.7 TB/s).  The max and the sum are reduced
// over the G lanes of the group without the LDS (softmax_reduce).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace pmkl_amd {

struct SoftmaxParams {
    void *dst;
    const void *src;
    int64_t stride;  // elements between row starts, src and dst alike
    int64_t batch;   // rows
    int32_t n;       // elements per row, 1 .. 1024
    int32_t log2g;   // lanes per row = 1 << log2g, 0 .. 6
};

constexpr int kSoftmaxThreads = 256;  // 4 waves per workgroup

template <typename T, int W>
struct SoftmaxVec {
    T v[W];
};

// Streaming accesses: every element is read once and written once, so loads
// and stores carry the nontemporal hint (the "nt" bit), which keeps the
// stream from displacing other data in the caches; measured ~10% faster than
// plain accesses on 131,072 x 1,024 fp32.  A vector moves as words of up to
// 16 bytes.
// A is the alignment in bytes that is known of the address: below the word's
// size the word is loaded and stored unaligned, which the global memory
// instructions take at any element alignment.
template <int BYTES, int A> struct SoftmaxWord;
#define PMKL_SOFTMAX_WORD(BYTES, A, T, ...) \
    template <> struct SoftmaxWord<BYTES, A> { typedef T type __attribute__((__VA_ARGS__ aligned(A))); };
PMKL_SOFTMAX_WORD(16, 16, unsigned, ext_vector_type(4),)
PMKL_SOFTMAX_WORD(16, 4, unsigned, ext_vector_type(4),)
PMKL_SOFTMAX_WORD(16, 2, unsigned, ext_vector_type(4),)
PMKL_SOFTMAX_WORD(8, 8, unsigned, ext_vector_type(2),)
PMKL_SOFTMAX_WORD(8, 2, unsigned, ext_vector_type(2),)
PMKL_SOFTMAX_WORD(4, 4, unsigned,)
PMKL_SOFTMAX_WORD(2, 2, unsigned short,)
#undef PMKL_SOFTMAX_WORD

template <int A, typename V>
__device__ __forceinline__ V softmax_nt_load(const void *p) {
    constexpr int WB = sizeof(V) >= 16 ? 16 : (int)sizeof(V);
    typedef typename SoftmaxWord<WB, (A < WB ? A : WB)>::type U;
    struct Words { U w[sizeof(V) / WB]; } r;
#pragma unroll
    for (int i = 0; i < (int)(sizeof(V) / WB); ++i) r.w[i] = __builtin_nontemporal_load(static_cast<const U *>(p) + i);
    return __builtin_bit_cast(V, r);
}
template <int A, typename V>
__device__ __forceinline__ void softmax_nt_store(void *p, const V &v) {
    constexpr int WB = sizeof(V) >= 16 ? 16 : (int)sizeof(V);
    typedef typename SoftmaxWord<WB, (A < WB ? A : WB)>::type U;
    struct Words { U w[sizeof(V) / WB]; };
    const Words r = __builtin_bit_cast(Words, v);
#pragma unroll
    for (int i = 0; i < (int)(sizeof(V) / WB); ++i) __builtin_nontemporal_store(r.w[i], static_cast<U *>(p) + i);
}

// exp(d) for d = x - max <= 0 on v_exp_f32 (2^t).  t = d*log2(e) is rounded
// to fp32, so 2^t alone would carry a relative error up to |t| * 2^-24; what it
// misses, exp(d - t ln 2), is put back as 1 + (d - t ln 2), the difference taken
// exactly with fmas against a two-part ln 2 (head = fp32(ln 2), tail = the
// remainder).  Error: that of v_exp_f32 plus about one rounding.  d below -120
// (exp < 1e-52, zero in fp32; this includes the -inf of padding and of masked
// inputs) is clamped to -120 so the fmas stay finite; a NaN d stays NaN (IEEE
// maximum, one v_maximum3_f32).
__device__ __forceinline__ float softmax_exp(float d) {
    constexpr float kLog2e = 1.44269504088896341f;
    constexpr float kLn2Hi = 0.693147182464599609375f;     // fp32(ln 2)
    constexpr float kLn2Lo = -1.90465429995776804525e-09f;   // ln 2 - kLn2Hi
    d = __builtin_elementwise_maximum(d, -120.f);
    const float t = d * kLog2e;
    const float r = fmaf(-t, kLn2Lo, fmaf(-t, kLn2Hi, d));
    const float e = __builtin_amdgcn_exp2f(t);
    return fmaf(e, r, e);
}

// Reduction over the 2^g lanes of a row group, every lane receiving the result:
// neighbours, quads, halves of 8 and of 16 by DPP (each step joins blocks whose
// lanes already agree, so the mirrored forms pair them as well as an xor
// would), rows of 16 and halves of the wave by the lane swaps.  One VALU
// operation per step, where a shuffle takes five and a trip through the LDS.
template <int CTRL>
__device__ __forceinline__ float softmax_dpp(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}
template <typename Op>
__device__ __forceinline__ float softmax_reduce(float x, int g, Op op) {
    if (g < 1) return x;
    x = op(x, softmax_dpp<0xb1>(x));    // quad_perm 1 0 3 2
    if (g < 2) return x;
    x = op(x, softmax_dpp<0x4e>(x));    // quad_perm 2 3 0 1
    if (g < 3) return x;
    x = op(x, softmax_dpp<0x141>(x));   // row_half_mirror
    if (g < 4) return x;
    x = op(x, softmax_dpp<0x140>(x));   // row_mirror
    if (g < 5) return x;
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = op(__uint_as_float(r[0]), __uint_as_float(r[1]));
    if (g < 6) return x;
    const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return op(__uint_as_float(h[0]), __uint_as_float(h[1]));
}

// RAGGED: rows of any length n >= W at any element alignment.  The row's last
// chunk is moved back to end with the row, so every access stays a whole vector
// inside its row; the `dup` elements that it shares with the chunk before are
// left out of its part of the sum and stored twice with the same bits.  Against
// single elements (2 bytes per lane and load): 151,296 x 197 bf16 67 -> 24 us,
// 60,000 x 999 fp16 92 -> 40, 131,072 x 333 fp32 61 -> 57.  Bound there: about
// 18 VALU clocks per element and 25 of 32 lanes in use at 197; several rows per
// wave, to hoist the row-independent work, ran no faster (2 rows: 25.5 us against 27.1 before the
// shorter exponential, 4: 27.1, 8: 31.2, and slower at every other shape).
template <typename Tin, typename Tout, int W, int C, bool LOG, bool RAGGED>
__global__ __launch_bounds__(kSoftmaxThreads) void softmax_fwd_kernel(SoftmaxParams p) {
    constexpr int AIN = RAGGED ? (int)sizeof(Tin) : W * (int)sizeof(Tin);
    constexpr int AOUT = RAGGED ? (int)sizeof(Tout) : W * (int)sizeof(Tout);
    const int lane = threadIdx.x & 63;
    const int g = p.log2g;
    const int G = 1 << g;
    const int j = lane & (G - 1);
    const int64_t wave = (int64_t)blockIdx.x * (kSoftmaxThreads / 64) + (threadIdx.x >> 6);
    const int64_t row = (wave << (6 - g)) + (lane >> g);
    const bool live = row < p.batch;
    const int64_t base = live ? row * p.stride : 0;
    const Tin *src = static_cast<const Tin *>(p.src) + base;

    // A chunk that a lane does not hold stays -inf: it adds exp(-inf) = 0.
    float x[C][W];
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int e0 = (c * G + j) * W;
        SoftmaxVec<Tin, W> t;
#pragma unroll
        for (int w = 0; w < W; ++w) t.v[w] = static_cast<Tin>(-INFINITY);
        if (live && e0 < p.n)   // then a whole chunk: n % W == 0, or RAGGED
            t = softmax_nt_load<AIN, SoftmaxVec<Tin, W>>(src + (RAGGED ? min(e0, p.n - W) : e0));
#pragma unroll
        for (int w = 0; w < W; ++w) x[c][w] = static_cast<float>(t.v[w]);
    }

    // Row max; a NaN element makes it NaN, and with it every output of the
    // row (as in the reference, through the sum).
    float m = -INFINITY;
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int w = 0; w < W; ++w) m = __builtin_elementwise_maximum(m, x[c][w]);
    m = softmax_reduce(m, g, [](float a, float b) { return __builtin_elementwise_maximum(a, b); });

    // Sum of exp(x - m); softmax keeps the exponentials, log-softmax keeps x.
    float s = 0.f;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int dup = RAGGED ? (c * G + j) * W - (p.n - W) : 0;   // > 0 in the last, moved chunk alone
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const float e = softmax_exp(x[c][w] - m);
            s += RAGGED && w < dup ? 0.f : e;
            if (!LOG) x[c][w] = e;
        }
    }
    s = softmax_reduce(s, g, [](float a, float b) { return a + b; });

    if (!live) return;
    Tout *dst = static_cast<Tout *>(p.dst) + base;
    // softmax: one correctly rounded reciprocal per row, then a multiply per
    // element (the reference divides each element by the sum); s == 0 gives NaN
    // as the reference's explicit check does.  log-softmax: (x - m) - log(s).
    const float k = LOG ? logf(s) : (s == 0.f ? __builtin_nanf("") : 1.f / s);
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int e0 = (c * G + j) * W;
        if (e0 < p.n) {
            SoftmaxVec<Tout, W> t;
#pragma unroll
            for (int w = 0; w < W; ++w) t.v[w] = static_cast<Tout>(LOG ? (x[c][w] - m) - k : x[c][w] * k);
            softmax_nt_store<AOUT>(dst + (RAGGED ? min(e0, p.n - W) : e0), t);
        }
    }
}

}  // namespace pmkl_amd
