// tq_digits.h -- f32 activations as exact integers for the i8 matrix cores: every
// row is a fixed-point number of 31 bits below its own largest magnitude, held as
// four balanced base-256 digits in four int8 rows.  The sums of digits times INT8
// codes are exact int32, so y is the exact sum of the fixed-point values, rounded
// once.  A value is at most 2^(e - 30) off, with 2^e <= the row's largest magnitude:
// over a row that is below 2^-31 of its 2-norm times sqrt(K), less than the f32
// rounding of the result up to K = 16384 (measured: 2.5e-8 of y at K = 64 to 14336,
// against 0.8e-7 to 2.8e-7 for f32 FMAs in a wave).
#pragma once

#include "tq_internal.h"

namespace tq {
namespace {

typedef f32x4 f32x4_a4 __attribute__((aligned(4)));  // a vector at the alignment of its elements

__device__ __forceinline__ uint32_t f32_bits(float v) { return __builtin_bit_cast(uint32_t, v); }

// value = digits * 2^(e - 29) with 2^e <= the row's largest magnitude < 2^(e + 1);
// a row holding an infinity or a NaN has no such e and its outputs are summed
// directly in f32.
constexpr int kNotFinite = INT32_MAX;

__device__ __forceinline__ int64_t join_digits(int d0, int d1, int d2, int d3) {
    return ((static_cast<int64_t>(d3) * 256 + d2) * 256 + d1) * 256 + d0;
}

// y of one output from its digits' sum (x, w: its f32 row and code row)
__device__ __forceinline__ float digit_out(int64_t v, int e, float sw, float b, const float* __restrict__ x,
                                           const int8_t* __restrict__ w, int k) {
    if (e != kNotFinite)
        return static_cast<float>(fma(static_cast<double>(v), ldexp(static_cast<double>(sw), e - 29),
                                      static_cast<double>(b)));
    float sum = 0.0f;
    for (int i = 0; i < k; ++i) sum = fmaf(x[i], static_cast<float>(w[i]), sum);
    return fmaf(sw, sum, b);
}

// x [rows, k] f32 -> digit rows [4 rows, lda] (zeros past k) and the row exponents:
// one block per row; v = x * 2^(29 - e) rounded to an integer (|v| <= 2^30), whose
// balanced base-256 digits are the bytes of (v + 0x808080) ^ 0x808080 (the top one
// signed).  The row stays in registers between its maximum and its digits (up to 4
// kItems kThreads values; longer rows are read again).
template <int kItems, int kThreads>
__global__ __launch_bounds__(kThreads) void k_split_rows(const float* __restrict__ x, int k, int lda,
                                                    int8_t* __restrict__ d, int* __restrict__ ea) {
    __shared__ uint32_t red[kThreads / kWave];
    const int row = blockIdx.x, tid = threadIdx.x;
    const float* src = x + static_cast<int64_t>(row) * k;
    auto load = [&](int j) -> f32x4 {  // values 4 j .. 4 j + 3, zeros past k
        if (4 * j + 4 <= k) return *reinterpret_cast<const f32x4_a4*>(src + 4 * j);
        f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
        if (4 * j < k) v.x = src[4 * j];
        if (4 * j + 1 < k) v.y = src[4 * j + 1];
        if (4 * j + 2 < k) v.z = src[4 * j + 2];
        return v;
    };
    // the largest |x| as bits: above every finite value for an infinity or a NaN
    auto fold = [](uint32_t mx, f32x4 v) {
        const uint32_t a = max(f32_bits(v.x) & 0x7FFFFFFFu, f32_bits(v.y) & 0x7FFFFFFFu);
        const uint32_t b = max(f32_bits(v.z) & 0x7FFFFFFFu, f32_bits(v.w) & 0x7FFFFFFFu);
        return max(mx, max(a, b));
    };
    const int items = lda / 4;
    f32x4 v[kItems];
    uint32_t mx = 0;
#pragma unroll
    for (int i = 0; i < kItems; ++i) v[i] = load(tid + kThreads * i);
#pragma unroll
    for (int i = 0; i < kItems; ++i) mx = fold(mx, v[i]);
    for (int j = tid + kThreads * kItems; j < items; j += kThreads) mx = fold(mx, load(j));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = max(mx, static_cast<uint32_t>(__shfl_xor(static_cast<int>(mx), o, kWave)));
    if ((tid & 63) == 0) red[tid >> 6] = mx;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kThreads / kWave; ++i) mx = max(mx, red[i]);
    const bool finite = mx < 0x7F800000u;
    const int e = max(static_cast<int>(mx >> 23), 1) - 127;
    if (tid == 0) ea[row] = finite ? e : kNotFinite;
    int8_t* dst = d + static_cast<int64_t>(row) * 4 * lda;
    auto digits = [&](float f) -> uint32_t {
        const int i = static_cast<int>(rintf(ldexpf(f, 29 - e)));
        return (static_cast<uint32_t>(i) + 0x00808080u) ^ 0x00808080u;
    };
    auto store = [&](int j, f32x4 f) {
        uint32_t a = 0, b = 0, c = 0, g = 0;
        if (finite) {
            a = digits(f.x);
            b = digits(f.y);
            c = digits(f.z);
            g = digits(f.w);
        }
        // 4 x 4 byte transpose: word r = digit r of the four values
        const uint32_t ab0 = __builtin_amdgcn_perm(b, a, 0x05010400u), ab1 = __builtin_amdgcn_perm(b, a, 0x07030602u);
        const uint32_t cg0 = __builtin_amdgcn_perm(g, c, 0x05010400u), cg1 = __builtin_amdgcn_perm(g, c, 0x07030602u);
        uint32_t* o = reinterpret_cast<uint32_t*>(dst) + j;
        const int step = lda / 4;
        o[0] = __builtin_amdgcn_perm(cg0, ab0, 0x05040100u);
        o[step] = __builtin_amdgcn_perm(cg0, ab0, 0x07060302u);
        o[2 * step] = __builtin_amdgcn_perm(cg1, ab1, 0x05040100u);
        o[3 * step] = __builtin_amdgcn_perm(cg1, ab1, 0x07060302u);
    };
#pragma unroll
    for (int i = 0; i < kItems; ++i)
        if (tid + kThreads * i < items) store(tid + kThreads * i, v[i]);
    for (int j = tid + kThreads * kItems; j < items; j += kThreads) store(j, load(j));
}

// Few rows: 1024 threads a row, for the latency of one pass over it; many: 256.
inline int launch_split_rows(const float* x, int m, int k, int lda, int8_t* d, int* ea, hipStream_t st,
                             const char* what) {
    const unsigned rows = static_cast<unsigned>(m);
    if (m <= 2 * device_cu_count())
        k_split_rows<4, 1024><<<rows, 1024, 0, st>>>(x, k, lda, d, ea);
    else if (lda <= 4096)
        k_split_rows<4, 256><<<rows, 256, 0, st>>>(x, k, lda, d, ea);
    else
        k_split_rows<16, 256><<<rows, 256, 0, st>>>(x, k, lda, d, ea);
    return check_launch(what);
}

}  // namespace
}  // namespace tq
