// tq_gemm_tile.h -- one register-staged MFMA GEMM for the 8-bit Linears the
// LDS-DMA kernels do not serve, over operand traits:
//
//   y[m, n] = epilogue(sum_k A[m, k] * W[n, k])       A, W K-contiguous ("NT")
//
//  * GemmI8: A and W INT8 codes, int32 sums (exact).
//  * GemmF8: A and W e4m3 codes on the fp8 matrix cores.
//  * GemmF8b: the same codes widened to bf16 (exact products, f32 sums).
//  * GemmF32<Val>: A f32, W INT8 or e4m3 codes, on the bf16 matrix cores.  Every f32
//    activation is split exactly into three bf16 planes (8 + 8 + 8 significand
//    bits, by truncation) and every code is exact in bf16, so each product is
//    exact and only the f32 sums round, whatever the spread of a row's values.
//
//  * GemmW4, GemmW4GateUp, GemmW4H: INT4 g128 codes widened to bf16 (exact) against bf16
//    activations (GemmW4H: f32 activations as bf16 hi + lo); every 128-long group's sum
//    is scaled by its f16 scale as it is added to the total.  GemmW4GateUp runs two
//    weight matrices side by side and stores h = SiLU(gate) * up.
//
// The 8-bit bf16 forms add their running sums into a second set of accumulators every
// kFlushStages stages (in f64 for GemmF8b), so that a sum's rounding grows with
// the square root of a run's length and not of K: relative errors at K = 14336 are
// 1.0e-7 (GemmF32) and 4.7e-8 (GemmF8b), against 2.8e-7 and 7.2e-8 for a wave's f32
// FMAs per output.  Runs of 256 k: with 512, rows that hold one value far above the
// rest (1000 times, K = 512 to 4096) end 1.2 to 1.6 times a wave's f32 FMAs' error off,
// with 256 1.0 to 1.25 times, at 2 % more time.
//
// Any M, N, K and any alignment of A, W and their rows (element-aligned
// pointers): global loads are 8 to 32 bytes per lane at byte (codes) or 4-byte
// (f32) alignment, which global memory instructions take on this target; the
// last, partial K stage is loaded apart, with zeros past K; rows past M or N re-read the
// last row and are not stored.
#pragma once

#include <algorithm>

#include "tq_internal.h"

namespace tq {
namespace {

typedef __bf16 tile_bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Vectors at the alignment of their elements.
typedef f32x4 f32x4_a4 __attribute__((aligned(4)));
typedef u32x2 u32x2_a1 __attribute__((aligned(1)));
typedef u32x4 u32x4_a1 __attribute__((aligned(1)));
typedef u32x4 u32x4_a2 __attribute__((aligned(2)));
typedef uint32_t u32_a1 __attribute__((aligned(1)));

__device__ __forceinline__ uint32_t f32_bits(float v) { return __builtin_bit_cast(uint32_t, v); }

typedef __bf16 tile_bf16x2 __attribute__((ext_vector_type(2)));
typedef float tile_f32x2 __attribute__((ext_vector_type(2)));
// a and b rounded to bf16, packed (a low)
__device__ __forceinline__ uint32_t bf16_pair(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((tile_f32x2{a, b}), tile_bf16x2));
}

// high halves of a and b as one dword (a low)
__device__ __forceinline__ uint32_t pack_hi(uint32_t a, uint32_t b) {
    return __builtin_amdgcn_perm(b, a, 0x07060302u);
}

// ---- sources: global elements -> registers (Raw) -> 16-byte LDS chunks ----
// kElems elements make one chunk of each of kPlanes planes.

// f32 -> three bf16 planes.  hi = x truncated to 8 significand bits, then the
// (exact) residual twice more: hi + mid + lo == x.  An infinity is its own hi;
// its residual must be 0, not inf - inf; a NaN stays NaN in mid and lo.  (Bits
// below 2^-133, bf16's last place, are dropped: only values under 2^-109 have any.)
struct SrcF32 {
    typedef float elem_t;
    static constexpr int kElems = 8, kPlanes = 3, kPer = 1;
    struct Raw {
        f32x4 a, b;
    };
    __device__ static Raw load(const elem_t* p) {
        return Raw{*reinterpret_cast<const f32x4_a4*>(p), *reinterpret_cast<const f32x4_a4*>(p + 4)};
    }
    __device__ static Raw load_tail(const elem_t* p, int n, int) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = p[min(i, n - 1)];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = i < n ? v[i] : 0.0f;
        return Raw{f32x4{v[0], v[1], v[2], v[3]}, f32x4{v[4], v[5], v[6], v[7]}};
    }
    __device__ static void planes(const Raw& r, u32x4 (&out)[kPlanes]) {
        const float v[8] = {r.a.x, r.a.y, r.a.z, r.a.w, r.b.x, r.b.y, r.b.z, r.b.w};
        uint32_t h[8], m[8], l[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            h[i] = f32_bits(v[i]) & 0xFFFF0000u;
            const float hf = __uint_as_float(h[i]);
            const float r1 = v[i] == hf ? 0.0f : v[i] - hf;
            m[i] = f32_bits(r1) & 0xFFFF0000u;
            l[i] = f32_bits(r1 - __uint_as_float(m[i]));  // at most 8 significant bits are left
        }
        out[0] = u32x4{pack_hi(h[0], h[1]), pack_hi(h[2], h[3]), pack_hi(h[4], h[5]), pack_hi(h[6], h[7])};
        out[1] = u32x4{pack_hi(m[0], m[1]), pack_hi(m[2], m[3]), pack_hi(m[4], m[5]), pack_hi(m[6], m[7])};
        out[2] = u32x4{pack_hi(l[0], l[1]), pack_hi(l[2], l[3]), pack_hi(l[4], l[5]), pack_hi(l[6], l[7])};
    }
};

// The first `take` (<= 16) bytes from p, zeros after them, where `n` bytes of a row of
// `k` are left from p on (none: n <= 0).  Rows of 16 bytes and more: one load of 16
// bytes that ends where the row does at the latest, shifted into place; shorter rows
// byte by byte.
__device__ __forceinline__ u32x4 bytes_tail(const uint8_t* p, int take, int n, int k) {
    uint64_t lo = 0, hi = 0;
    if (k >= 16) {  // uniform
        const int back = n >= 16 ? 0 : 16 - n;  // bytes before p that the load takes in
        const u32x4 v = *reinterpret_cast<const u32x4_a1*>(p - back);
        lo = v.x | static_cast<uint64_t>(v.y) << 32;
        hi = v.z | static_cast<uint64_t>(v.w) << 32;
        if (back >= 8) {
            lo = hi;
            hi = 0;
        }
        const int s = 8 * (back & 7);
        if (s) {
            lo = (lo >> s) | (hi << (64 - s));
            hi >>= s;
        }
    } else {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const uint64_t b = p[min(i, n - 1)];
            if (i < 8)
                lo |= b << (8 * i);
            else
                hi |= b << (8 * (i - 8));
        }
    }
    // zero what `take` leaves out
    lo = take >= 8 ? lo : take <= 0 ? 0 : lo & (~uint64_t{0} >> (64 - 8 * take));
    hi = take >= 16 ? hi : take <= 8 ? 0 : hi & (~uint64_t{0} >> (128 - 8 * take));
    return u32x4{static_cast<uint32_t>(lo), static_cast<uint32_t>(lo >> 32), static_cast<uint32_t>(hi),
                 static_cast<uint32_t>(hi >> 32)};
}

// 8 byte codes per chunk: the value of each as bf16 (exact).
struct ValI8 {
    typedef int8_t code_t;
    __device__ static float value(uint32_t w, int b) { return static_cast<float>(static_cast<int8_t>(w >> (8 * b))); }
};
struct ValFp8 {
    typedef uint8_t code_t;
    template <int kB>
    __device__ static float get(uint32_t w) { return __builtin_amdgcn_cvt_f32_fp8(static_cast<int>(w), kB); }
    __device__ static float value(uint32_t w, int b) {
        return b == 0 ? get<0>(w) : b == 1 ? get<1>(w) : b == 2 ? get<2>(w) : get<3>(w);
    }
};
template <class Val>
struct SrcBf16 {
    typedef typename Val::code_t elem_t;
    static constexpr int kElems = 8, kPlanes = 1, kPer = 1;
    struct Raw {
        u32x2 v;
    };
    __device__ static Raw load(const elem_t* p) { return Raw{*reinterpret_cast<const u32x2_a1*>(p)}; }
    __device__ static Raw load_tail(const elem_t* p, int n, int k) {
        const u32x4 v = bytes_tail(reinterpret_cast<const uint8_t*>(p), min(n, 8), n, k);
        return Raw{u32x2{v.x, v.y}};
    }
    __device__ static void planes(const Raw& r, u32x4 (&out)[1]) {
        uint32_t f[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) f[i] = f32_bits(Val::value(i < 4 ? r.v.x : r.v.y, i & 3));
        out[0] = u32x4{pack_hi(f[0], f[1]), pack_hi(f[2], f[3]), pack_hi(f[4], f[5]), pack_hi(f[6], f[7])};
    }
};

// 16 byte codes per chunk, as they are.
template <class T>
struct SrcBytes {
    typedef T elem_t;
    static constexpr int kElems = 16, kPlanes = 1, kPer = 1;
    struct Raw {
        u32x4 v;
    };
    __device__ static Raw load(const elem_t* p) { return Raw{*reinterpret_cast<const u32x4_a1*>(p)}; }
    __device__ static Raw load_tail(const elem_t* p, int n, int k) {
        return Raw{bytes_tail(reinterpret_cast<const uint8_t*>(p), min(n, 16), n, k)};
    }
    __device__ static void planes(const Raw& r, u32x4 (&out)[1]) { out[0] = r.v; }
};

// f32 -> bf16 hi and lo (round to nearest: hi + lo keeps 2^-18 of the value); an
// infinity is its own hi.
struct SrcF32HiLo {
    typedef float elem_t;
    static constexpr int kElems = 8, kPlanes = 2, kPer = 1;
    typedef SrcF32::Raw Raw;
    __device__ static Raw load(const elem_t* p) { return SrcF32::load(p); }
    __device__ static Raw load_tail(const elem_t* p, int n, int k) { return SrcF32::load_tail(p, n, k); }
    __device__ static void planes(const Raw& r, u32x4 (&out)[2]) {
        const float v[8] = {r.a.x, r.a.y, r.a.z, r.a.w, r.b.x, r.b.y, r.b.z, r.b.w};
        uint32_t h[4], l[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float a = v[2 * i], b = v[2 * i + 1];
            h[i] = bf16_pair(a, b);
            const float ha = __uint_as_float(h[i] << 16), hb = __uint_as_float(h[i] & 0xFFFF0000u);
            l[i] = bf16_pair(a == ha ? 0.0f : a - ha, b == hb ? 0.0f : b - hb);
        }
        out[0] = u32x4{h[0], h[1], h[2], h[3]};
        out[1] = u32x4{l[0], l[1], l[2], l[3]};
    }
};

// bf16 activations as they are.
struct SrcBf16Raw {
    typedef uint16_t elem_t;
    static constexpr int kElems = 8, kPlanes = 1, kPer = 1;
    struct Raw {
        u32x4 v;
    };
    __device__ static Raw load(const elem_t* p) { return Raw{*reinterpret_cast<const u32x4_a2*>(p)}; }
    __device__ static Raw load_tail(const elem_t* p, int, int) { return load(p); }  // K % 128 == 0: no tails
    __device__ static void planes(const Raw& r, u32x4 (&out)[1]) { out[0] = r.v; }
};

// 8 nibbles (low first) -> bf16 of code / 16, exact (v_cvt_off_f32_i4; the 16 goes into
// the group scale).
struct SrcW4 {
    typedef uint8_t elem_t;
    static constexpr int kElems = 8, kPlanes = 1, kPer = 2;
    struct Raw {
        uint32_t v;
    };
    __device__ static Raw load(const elem_t* p) { return Raw{*reinterpret_cast<const u32_a1*>(p)}; }
    __device__ static Raw load_tail(const elem_t* p, int, int) { return load(p); }
    __device__ static void planes(const Raw& r, u32x4 (&out)[1]) {
        uint32_t f[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) f[i] = f32_bits(__builtin_amdgcn_cvt_off_f32_i4(static_cast<int>(r.v >> (4 * i))));
        out[0] = u32x4{pack_hi(f[0], f[1]), pack_hi(f[2], f[3]), pack_hi(f[4], f[5]), pack_hi(f[6], f[7])};
    }
};

// ---- operand traits ----
// kFragChunks 16-byte chunks per lane and MFMA; an MFMA step covers twice that
// many chunks of a row (one share per lane half).
struct OpBf16 {
    typedef f32x16 Acc;
    static constexpr bool kFlush = true, kGroups = false, kGateUp = false;
    static constexpr int kFragChunks = 1;
    typedef u32x4 Frag;
    __device__ static Frag frag(const u32x4 (&c)[1]) { return c[0]; }
    __device__ static Acc mfma(Frag a, Frag b, Acc c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(tile_bf16x8, a),
                                                       __builtin_bit_cast(tile_bf16x8, b), c, 0, 0, 0);
    }
};
template <class Val>
struct GemmF32 : OpBf16 {
    typedef SrcF32 A;
    typedef SrcBf16<Val> W;
    typedef float part_t;
    static constexpr bool kRowScale = false;
    static constexpr int kFlushStages = 4;
};
typedef GemmF32<ValI8> GemmI8W;
typedef GemmF32<ValFp8> GemmF8W;
struct GemmF8b : OpBf16 {
    typedef SrcBf16<ValFp8> A;
    typedef SrcBf16<ValFp8> W;
    typedef double part_t;
    static constexpr bool kRowScale = true;
    static constexpr int kFlushStages = 4;
};
struct GemmW4 : OpBf16 {
    typedef SrcBf16Raw A;
    typedef SrcW4 W;
    typedef float part_t;
    static constexpr bool kRowScale = false, kGroups = true;
    static constexpr int kFlushStages = 2;  // one group
};
struct GemmW4GateUp : GemmW4 {
    static constexpr bool kGateUp = true;
};
struct GemmW4H : GemmW4 {
    typedef SrcF32HiLo A;
};
struct GemmI8 {
    typedef SrcBytes<int8_t> A;
    typedef SrcBytes<int8_t> W;
    typedef i32x16 Acc;
    typedef int32_t part_t;
    static constexpr bool kRowScale = true, kFlush = false, kGroups = false, kGateUp = false;
    static constexpr int kFragChunks = 1;
    typedef i32x4 Frag;
    __device__ static Frag frag(const u32x4 (&c)[1]) { return __builtin_bit_cast(i32x4, c[0]); }
    __device__ static Acc mfma(Frag a, Frag b, Acc c) {
        return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
    }
};
struct GemmF8 {
    typedef SrcBytes<uint8_t> A;
    typedef SrcBytes<uint8_t> W;
    typedef f32x16 Acc;
    typedef float part_t;
    static constexpr bool kRowScale = true, kFlush = false, kGroups = false, kGateUp = false;
    static constexpr int kFragChunks = 2;
    typedef i32x8 Frag;
    __device__ static Frag frag(const u32x4 (&c)[2]) {
        return i32x8{static_cast<int>(c[0].x), static_cast<int>(c[0].y), static_cast<int>(c[0].z),
                     static_cast<int>(c[0].w), static_cast<int>(c[1].x), static_cast<int>(c[1].y),
                     static_cast<int>(c[1].z), static_cast<int>(c[1].w)};
    }
    __device__ static Acc mfma(Frag a, Frag b, Acc c) {
        // cbsz = blgp = 0: both operands FP8 E4M3; scales 0 select the unscaled MFMA
        return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 0, 0, 0, 0, 0, 0);
    }
};

struct TileArgs {
    const void* a;      // A [m, k]
    const void* w;      // W [n, k]
    const float* sa;    // row scales [m] (kRowScale)
    const float* sw;    // column scales [n]
    const float* bias;  // [n] or null
    const uint16_t* sg;   // f16 group scales [n, k / 128] (kGroups)
    const void* w2;       // kGateUp: w and sg are gate's, w2 and sg2 up's, n both rows' count
    const uint16_t* sg2;  // (n = 2 F: partial sums hold gate's F columns, then up's)
    int m, n, k;
    int tiles_m, tiles_n, split;
    int32_t* acc;  // int32 sums [m, n] or null (GemmI8)
    float* y;      // [m, n]
    void* part;    // split > 1: partial sums [split][m][n]
};

// SiLU(g) * u, as the FFN kernels form it
__device__ __forceinline__ float silu_mul(float g, float u) { return g * (1.0f / (1.0f + __expf(-g))) * u; }

// y[mm, nn] from its sum
template <class T>
__device__ __forceinline__ void tile_store(const TileArgs& p, typename T::part_t v, int mm, int nn, float sw, float b) {
    const int64_t o = static_cast<int64_t>(mm) * p.n + nn;
    if constexpr (T::kGroups) {
        p.y[o] = v + b;
    } else if constexpr (T::kRowScale) {
        if constexpr (__is_same(typename T::part_t, int32_t))
            if (p.acc) p.acc[o] = v;
        p.y[o] = fmaf(static_cast<float>(v) * p.sa[mm], sw, b);
    } else {
        p.y[o] = fmaf(sw, v, b);
    }
}

constexpr int kTileRow = 128;  // bytes of K per row and stage: 8 chunks
__device__ __forceinline__ int tile_swz(int row) { return (row >> 1) & 7; }

template <class T, int BM, int BN>
constexpr int tile_stage_bytes() {
    return (T::A::kPlanes * BM + T::W::kPlanes * BN) * kTileRow;
}

// Block: WM x WN waves (256 threads), each a (BM / WM) x (BN / WN) tile of 32 x
// 32 MFMA tiles.  K runs in stages of 8 chunks (64 bf16 or 128 byte codes) through
// two LDS buffers; while the MFMAs of stage s run, the registers holding stage
// s + 1 are converted and written to the other buffer and refilled from global
// memory with stage s + 2, a share per MFMA step, so that conversion and loads
// hide under the matrix cores.  One barrier per stage.
template <class T, int BM, int BN, int WM, int WN, int kOcc>
__global__ __launch_bounds__(256, kOcc) void k_gemm_tile(TileArgs p) {
    using SA = typename T::A;
    using SW = typename T::W;
    static_assert(WM * WN == 4, "4 waves");
    constexpr int TM = BM / WM / 32, TN = BN / WN / 32, PA = SA::kPlanes;
    constexpr int kAItems = BM * 8 / 256, kWItems = BN * 8 / 256;
    constexpr int kSteps = 4 / T::kFragChunks;
    constexpr int kStage = tile_stage_bytes<T, BM, BN>();
    constexpr int BK = 8 * SA::kElems;
    static_assert(SA::kElems == SW::kElems && SW::kPlanes == 1, "operands advance together");
    static_assert(kAItems >= 1 && kWItems >= 1 && TM >= 1 && TN >= 1, "tile too small");
    __shared__ __attribute__((aligned(1024))) int8_t lds[2 * kStage];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % WM, wn = wave / WM, l32 = lane & 31, lh = lane >> 5;
    // consecutive blocks go to different XCDs: give each XCD a contiguous run of
    // tiles (row tiles fastest) so that blocks sharing weight rows share an L2
    const int total = p.tiles_m * p.tiles_n * p.split;
    const int q8 = total >> 3, r8 = total & 7, xcd = blockIdx.x & 7;
    const int L = xcd * q8 + min(xcd, r8) + (blockIdx.x >> 3);
    const int tm = L % p.tiles_m, tn = (L / p.tiles_m) % p.tiles_n, ks = L / (p.tiles_m * p.tiles_n);
    const int m0 = tm * BM, n0 = tn * BN;
    const int rows_w = T::kGateUp ? p.n / 2 : p.n;
    static_assert(!T::kGateUp || TN == 2, "a wave holds 32 gate and the same 32 up columns");
    const int stages = (p.k + BK - 1) / BK;
    constexpr int kUnit = T::kGroups ? 2 : 1;  // whole groups per split (two stages each)
    const int s_begin = static_cast<int>(static_cast<int64_t>(ks) * (stages / kUnit) / p.split) * kUnit;
    const int s_end = static_cast<int>(static_cast<int64_t>(ks + 1) * (stages / kUnit) / p.split) * kUnit;

    // item i: row (tid + 256 i) / 8, chunk tid % 8
    const int chunk = tid & 7;
    const typename SA::elem_t* asrc[kAItems];
    const typename SW::elem_t* wsrc[kWItems];
    uint32_t adst[kAItems], wdst[kWItems];
#pragma unroll
    for (int i = 0; i < kAItems; ++i) {
        const int r = (tid >> 3) + 32 * i;
        asrc[i] = static_cast<const typename SA::elem_t*>(p.a) + static_cast<int64_t>(min(m0 + r, p.m - 1)) * p.k;
        adst[i] = r * kTileRow + ((chunk ^ tile_swz(r)) << 4);
    }
#pragma unroll
    for (int i = 0; i < kWItems; ++i) {
        const int r = (tid >> 3) + 32 * i;
        const void* w = p.w;
        int row = n0 + r;
        if constexpr (T::kGateUp) {
            // tile row 64 t + i: gate row i of the block's t-th 32, i < 32, then up's
            row = n0 / 2 + 32 * (r >> 6) + (r & 31);
            w = r & 32 ? p.w2 : p.w;
        }
        wsrc[i] = static_cast<const typename SW::elem_t*>(w) +
                  static_cast<int64_t>(min(row, rows_w - 1)) * (p.k / SW::kPer);
        wdst[i] = PA * BM * kTileRow + r * kTileRow + ((chunk ^ tile_swz(r)) << 4);
    }
    // two register sets: stage s of a split goes through set (s - s_begin) & 1
    struct Regs {
        typename SA::Raw a[kAItems];
        typename SW::Raw w[kWItems];
    } rg[2];
    auto store_a = [&](const Regs& r, int i, int8_t* st) {
        u32x4 c[PA];
        SA::planes(r.a[i], c);
#pragma unroll
        for (int pl = 0; pl < PA; ++pl) *reinterpret_cast<u32x4*>(st + pl * BM * kTileRow + adst[i]) = c[pl];
    };
    auto store_w = [&](const Regs& r, int i, int8_t* st) {
        u32x4 c[1];
        SW::planes(r.w[i], c);
        *reinterpret_cast<u32x4*>(st + wdst[i]) = c[0];
    };
    auto load_a = [&](Regs& r, int i, int s) { r.a[i] = SA::load(asrc[i] + s * BK + chunk * SA::kElems); };
    auto load_w = [&](Regs& r, int i, int s) { r.w[i] = SW::load(wsrc[i] + (s * BK + chunk * SW::kElems) / SW::kPer); };
    // output column of the lane in its j-th tile (kGateUp: of gate and of up alike)
    auto column = [&](int j) { return T::kGateUp ? n0 / 2 + wn * 32 + l32 : n0 + (wn * TN + j) * 32 + l32; };
    // the f16 scales of group g of the lane's columns
    uint16_t sc[TN];
    auto load_scales = [&](int g) {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const uint16_t* sg = T::kGateUp && j == 1 ? p.sg2 : p.sg;
            sc[j] = sg[static_cast<int64_t>(min(column(j), rows_w - 1)) * (p.k / 128) + g];
        }
    };
    // fragment of row r (of a plane at `base`) for step `step`
    auto frag = [&](const int8_t* base, int r, int step) -> typename T::Frag {
        u32x4 c[T::kFragChunks];
#pragma unroll
        for (int j = 0; j < T::kFragChunks; ++j) {
            const int ch = (2 * step + lh) * T::kFragChunks + j;
            c[j] = *reinterpret_cast<const u32x4*>(base + r * kTileRow + ((ch ^ tile_swz(r)) << 4));
        }
        return T::frag(c);
    };

    // a plane set's leading plane sums apart from the rest, whose terms are 2^-8 of
    // its own: the leading sums' additions are then a third as many (and mostly
    // exact), the others' rounding negligible
    constexpr int kSets = PA > 1 ? 2 : 1;
    typename T::Acc acc[kSets][TM][TN];
#pragma unroll
    for (int h = 0; h < kSets; ++h)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[h][i][j] = typename T::Acc{};

    // the MFMAs of step `step` of the stage in `st`
    auto step_mfma = [&](const int8_t* st, int step) {
        typename T::Frag fa[TM][PA], fw[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int pl = 0; pl < PA; ++pl)
                fa[i][pl] = frag(st + pl * BM * kTileRow, (wm * TM + i) * 32 + l32, step);
#pragma unroll
        for (int j = 0; j < TN; ++j) fw[j] = frag(st + PA * BM * kTileRow, (wn * TN + j) * 32 + l32, step);
#pragma unroll
        for (int pl = 0; pl < PA; ++pl)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    typename T::Acc& c = acc[pl > 0 ? kSets - 1 : 0][i][j];
                    c = T::mfma(fa[i][pl], fw[j], c);
                }
    };
    // one stage: its MFMAs, the next stage's registers `r` into the other buffer,
    // and the stage after next's successor into those registers
    auto stage = [&](const int8_t* st, int8_t* nst, Regs& r, int s_load) {
#pragma unroll
        for (int step = 0; step < kSteps; ++step) {
            step_mfma(st, step);
#pragma unroll
            for (int i = 0; i < kAItems; ++i)
                if (i * kSteps / kAItems == step) {
                    store_a(r, i, nst);
                    load_a(r, i, s_load);
                }
#pragma unroll
            for (int i = 0; i < kWItems; ++i)
                if (i * kSteps / kWItems == step) {
                    store_w(r, i, nst);
                    load_w(r, i, s_load);
                }
        }
        // the LDS writes have landed and every wave is past its reads of `st`; global
        // loads stay in flight across the barrier
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };
    // whole stages [s_begin, s_full): loads past the last re-read it (never used)
    const int s_full = min(s_end, p.k / BK), s_last = s_full - 1;
    typename T::part_t tot[T::kFlush ? TM : 1][T::kFlush ? TN : 1][16];
    auto flush = [&]() {
        if constexpr (T::kFlush) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    if constexpr (kSets == 2) acc[0][i][j] += acc[1][i][j];
                    if constexpr (T::kGroups) {
                        const float sj = 16.0f * __half2float(__ushort_as_half(sc[j]));
#pragma unroll
                        for (int e = 0; e < 16; ++e) tot[i][j][e] = fmaf(acc[0][i][j][e], sj, tot[i][j][e]);
                    } else {
#pragma unroll
                        for (int e = 0; e < 16; ++e) tot[i][j][e] += acc[0][i][j][e];
                    }
#pragma unroll
                    for (int h = 0; h < kSets; ++h) acc[h][i][j] = typename T::Acc{};
                }
        }
    };
    if constexpr (T::kFlush) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) tot[i][j][e] = 0;
    }
    if (s_begin < s_full) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int i = 0; i < kAItems; ++i) load_a(rg[h], i, min(s_begin + h, s_last));
#pragma unroll
            for (int i = 0; i < kWItems; ++i) load_w(rg[h], i, min(s_begin + h, s_last));
        }
#pragma unroll
        for (int i = 0; i < kAItems; ++i) {
            store_a(rg[0], i, lds);
            load_a(rg[0], i, min(s_begin + 2, s_last));
        }
#pragma unroll
        for (int i = 0; i < kWItems; ++i) {
            store_w(rg[0], i, lds);
            load_w(rg[0], i, min(s_begin + 2, s_last));
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        int s = s_begin;
        for (; s + 1 < s_full; s += 2) {
            if constexpr (T::kGroups) load_scales(s / kUnit);
            stage(lds, lds + kStage, rg[1], min(s + 3, s_last));
            stage(lds + kStage, lds, rg[0], min(s + 4, s_last));
            if constexpr (T::kFlush)
                if (((s + 2 - s_begin) & (T::kFlushStages - 1)) == 0) flush();
        }
        if (s < s_full) stage(lds, lds + kStage, rg[1], s_last);
    }
    if (s_full < s_end) {  // the partial last stage (zeros past K)
        const int k0 = s_full * BK + chunk * SA::kElems;
#pragma unroll
        for (int i = 0; i < kAItems; ++i) {
            rg[0].a[i] = SA::load_tail(asrc[i] + k0, p.k - k0, p.k);
            store_a(rg[0], i, lds);
        }
#pragma unroll
        for (int i = 0; i < kWItems; ++i) {
            rg[0].w[i] = SW::load_tail(wsrc[i] + k0 / SW::kPer, p.k - k0, p.k);
            store_w(rg[0], i, lds);
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int step = 0; step < kSteps; ++step) step_mfma(lds, step);
    }
    if constexpr (!T::kGroups) flush();

    auto sum = [&](int i, int j, int e) {
        if constexpr (T::kFlush)
            return tot[i][j][e];
        else
            return acc[0][i][j][e];
    };
    // lane holds D[m = 8 (e/4) + 4 lh + e % 4][n = l32] of each 32 x 32 tile: a
    // store covers 32 consecutive n of two rows
    if constexpr (T::kGateUp) {
        const int nn = column(0), f = rows_w;
        if (nn >= f) return;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int mm = m0 + (wm * TM + i) * 32 + 8 * (e >> 2) + 4 * lh + (e & 3);
                if (mm >= p.m) continue;
                if (p.split == 1) {
                    p.y[static_cast<int64_t>(mm) * f + nn] = silu_mul(sum(i, 0, e), sum(i, TN - 1, e));
                } else {
                    float* o = static_cast<float*>(p.part) + (static_cast<int64_t>(ks) * p.m + mm) * p.n + nn;
                    o[0] = sum(i, 0, e);
                    o[f] = sum(i, TN - 1, e);
                }
            }
        return;
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int nn = column(j);
        const bool nval = nn < p.n;
        const float sw = !T::kGroups && p.split == 1 && nval ? p.sw[nn] : 0.0f;
        const float bv = p.split == 1 && nval && p.bias ? p.bias[nn] : 0.0f;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int mm = m0 + (wm * TM + i) * 32 + 8 * (e >> 2) + 4 * lh + (e & 3);
                if (!nval || mm >= p.m) continue;
                const typename T::part_t v = sum(i, j, e);
                if (p.split == 1)
                    tile_store<T>(p, v, mm, nn, sw, bv);
                else
                    static_cast<typename T::part_t*>(
                        p.part)[(static_cast<int64_t>(ks) * p.m + mm) * p.n + nn] = v;
            }
    }
}

// Adds the partial sums of a split launch in a fixed order and finishes the outputs.
template <class T>
__global__ __launch_bounds__(256) void k_gemm_tile_finish(TileArgs p) {
    const int64_t mn = static_cast<int64_t>(p.m) * p.n;
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    const int cols = T::kGateUp ? p.n / 2 : p.n;
    if (i >= static_cast<int64_t>(p.m) * cols) return;
    const int mm = static_cast<int>(i / cols), nn = static_cast<int>(i - static_cast<int64_t>(mm) * cols);
    const typename T::part_t* part = static_cast<const typename T::part_t*>(p.part) + static_cast<int64_t>(mm) * p.n + nn;
    typename T::part_t v = part[0];
    for (int s = 1; s < p.split; ++s) v += part[s * mn];
    if constexpr (T::kGateUp) {
        float u = part[cols];
        for (int s = 1; s < p.split; ++s) u += part[s * mn + cols];
        p.y[i] = silu_mul(v, u);
    } else {
        tile_store<T>(p, v, mm, nn, T::kGroups ? 0.0f : p.sw[nn], p.bias ? p.bias[nn] : 0.0f);
    }
}

// ------------------------------------------------------------------ host side
// Tile sizes and a launch's time in ns: of each stage with at most one block on a CU
// (t1) and per block when several share it (t2), and apart from the stages (launch,
// first loads, stores) with one round of blocks (f1) and per round (f2); `split` is the
// finishing launch's.  Fitted to every tile and split at M = 1 to 2048 and 18 weights from
// 64 x 64 to 14336 x 4096, 4096 x 14336, 16384 x 128 and 64 x 16384, read past the caches:
// the chosen one takes 1.01 to 1.03 times the fastest's time on average.  t1 = 0: not built
// (GateUp holds two column tiles per wave; GemmF32's three planes at 128 x 128 were the
// fastest at none of 680 sizes).
struct TileShape {
    int bm, bn, t1, t2, f1, f2;
};
constexpr int kTileShapes = 4;
enum { kTile128x128, kTile64x64, kTile32x128, kTile64x128 };
template <class T>
struct TileCosts;
template <>
struct TileCosts<GemmI8> {
    static constexpr TileShape shape[kTileShapes] = {{128, 128, 600, 640, 8000, 7500}, {64, 64, 270, 250, 4300, 1770}, {32, 128, 290, 250, 4500, 3770}, {64, 128, 430, 360, 6250, 4300}};
    static constexpr int split = 2200;
};
template <>
struct TileCosts<GemmF8> {
    static constexpr TileShape shape[kTileShapes] = {{128, 128, 630, 600, 8000, 7000}, {64, 64, 270, 230, 4600, 1560}, {32, 128, 300, 230, 4760, 4070}, {64, 128, 300, 400, 6870, 2550}};
    static constexpr int split = 2400;
};
template <>
struct TileCosts<GemmF8b> {
    static constexpr TileShape shape[kTileShapes] = {{128, 128, 820, 1060, 8300, 8300}, {64, 64, 390, 260, 4770, 1190}, {32, 128, 550, 330, 4610, 1140}, {64, 128, 640, 500, 6430, 1450}};
    static constexpr int split = 2600;
};
template <class Val>
struct TileCosts<GemmF32<Val>> {
    static constexpr TileShape shape[kTileShapes] = {{128, 128, 0, 0, 0, 0}, {64, 64, 785, 575, 5300, 2200}, {32, 128, 820, 535, 4650, 3150}, {64, 128, 1055, 840, 7200, 2770}};
    static constexpr int split = 3000;
};

template <>
struct TileCosts<GemmW4> {
    static constexpr TileShape shape[kTileShapes] = {{128, 128, 830, 500, 7500, 6850}, {64, 64, 330, 230, 4870, 1170}, {32, 128, 580, 380, 5020, 1020}, {64, 128, 560, 410, 6810, 2460}};
    static constexpr int split = 2200;
};
template <>
struct TileCosts<GemmW4GateUp> {
    static constexpr TileShape shape[kTileShapes] = {{128, 128, 820, 780, 3000, 0}, {64, 64, 0, 0, 0, 0}, {32, 128, 0, 0, 0, 0}, {64, 128, 650, 525, 3000, 0}};
    static constexpr int split = 3000;
};
template <>
struct TileCosts<GemmW4H> {
    static constexpr TileShape shape[kTileShapes] = {{128, 128, 1500, 1900, 3000, 0}, {64, 64, 720, 570, 3000, 0}, {32, 128, 810, 475, 3000, 0}, {64, 128, 1000, 815, 3000, 0}};
    static constexpr int split = 3000;
};

template <class T>
constexpr bool tile_built(int shape) {
    return TileCosts<T>::shape[shape].t1 > 0;
}

// The LDS-DMA kernels' 128 x 256 tiles: a 128-byte stage takes t with up to half of the
// CUs at work and t + busy with all of them (M = 1024, N = K = 4096, 128 blocks: 25.4 us;
// M = 2048, 256 blocks: 37 us).
constexpr int kTileDma = -1;
struct DmaCost {
    int t, busy, f1, f2;
};

inline int64_t dma_ns(const DmaCost& c, int64_t m, int64_t n, int64_t k) {
    const int64_t cus = device_cu_count(), blocks = ((m + 127) / 128) * ((n + 255) / 256);
    const int64_t full = blocks / cus, rest = blocks % cus, rounds = full + (rest > 0);
    int64_t stage = full * (c.t + c.busy);
    if (rest) stage += c.t + c.busy * std::max<int64_t>(0, 2 * rest - cus) / cus;
    const int64_t ns = c.f1 + c.f2 * (rounds - 1) + k / 128 * stage;
    // stores at 3.1 TB/s; weights past 16 MiB hold the loads up by some of their read
    return std::max(ns, m * n * 4 / 3100) + std::max<int64_t>(0, n * k - (16 << 20)) / 6000;
}

struct TilePlan {
    int shape, split, tiles_m, tiles_n;
    int64_t part_bytes, ns;
};

// The shape and K split with the smallest estimate; a split adds the finishing launch
// and its partial sums' traffic (4 TB/s).  `dma`: the LDS-DMA kernel serves these operands.
template <class T>
TilePlan tile_plan(int64_t m, int64_t n, int64_t k, const DmaCost* dma, bool may_split) {
    const int64_t cus = device_cu_count();
    const int64_t stages = (k + 8 * T::A::kElems - 1) / (8 * T::A::kElems);
    TilePlan best{kTile64x128, 1, 0, 0, 0, INT64_MAX};
    if (dma) best = TilePlan{kTileDma, 1, 0, 0, 0, dma_ns(*dma, m, n, k)};
    for (int c = 0; c < kTileShapes; ++c) {
        if (!tile_built<T>(c)) continue;
        const TileShape& t = TileCosts<T>::shape[c];
        const int64_t tm = (m + t.bm - 1) / t.bm, tn = (n + t.bn - 1) / t.bn;
        for (int split : {1, 2, 3, 4, 6, 8, 12, 16}) {
            if (split > 1 && (!may_split || stages < 4 * split || tm * tn * split > 4 * cus)) break;
            const int64_t rounds = (tm * tn * split + cus - 1) / cus, per = (stages + split - 1) / split;
            int64_t ns = rounds == 1 ? t.f1 + t.t1 * per
                                     : std::max<int64_t>(t.f1, rounds * t.f2) + std::max<int64_t>(t.t1, rounds * t.t2) * per;
            const int64_t part = split * m * n * static_cast<int64_t>(sizeof(typename T::part_t));
            if (split > 1) ns += TileCosts<T>::split + 2 * part / 4000;
            if (ns < best.ns) best = TilePlan{c, split, 0, 0, split > 1 ? part : 0, ns};
        }
    }
    if (best.shape != kTileDma) {
        const TileShape& t = TileCosts<T>::shape[best.shape];
        best.tiles_m = static_cast<int>((m + t.bm - 1) / t.bm);
        best.tiles_n = static_cast<int>((n + t.bn - 1) / t.bn);
    }
    return best;
}

// m, n and k fit the kernels' 32-bit indexes
inline bool tile_fits(int64_t m, int64_t n, int64_t k) {
    return m < (int64_t(1) << 31) - 128 && n < (int64_t(1) << 31) - 128 && k < (int64_t(1) << 31) - 1024 &&
           ((m + 31) / 32) * ((n + 63) / 64) < (int64_t(1) << 31);
}

// Launches the plan's tiles (not kTileDma) and, for a split, the finishing kernel.
template <class T>
int launch_tile(const TilePlan& plan, TileArgs p, hipStream_t st, const char* what) {
    p.tiles_m = plan.tiles_m;
    p.tiles_n = plan.tiles_n;
    p.split = plan.split;
    const unsigned grid = static_cast<unsigned>(static_cast<int64_t>(p.tiles_m) * p.tiles_n * p.split);
    switch (plan.shape) {
    case kTile128x128:
        if constexpr (tile_built<T>(kTile128x128)) k_gemm_tile<T, 128, 128, 2, 2, 1><<<grid, 256, 0, st>>>(p);
        break;
    case kTile64x64:
        if constexpr (tile_built<T>(kTile64x64)) k_gemm_tile<T, 64, 64, 2, 2, 2><<<grid, 256, 0, st>>>(p);
        break;
    case kTile32x128:
        if constexpr (tile_built<T>(kTile32x128)) k_gemm_tile<T, 32, 128, 1, 4, 2><<<grid, 256, 0, st>>>(p);
        break;
    default: k_gemm_tile<T, 64, 128, 2, 2, 2><<<grid, 256, 0, st>>>(p);
    }
    if (p.split > 1) {
        const int rc = check_launch(what);
        if (rc != TQ_OK) return rc;
        const int64_t blocks = (static_cast<int64_t>(p.m) * (T::kGateUp ? p.n / 2 : p.n) + 255) / 256;
        k_gemm_tile_finish<T><<<static_cast<unsigned>(blocks), 256, 0, st>>>(p);
    }
    return check_launch(what);
}

}  // namespace
}  // namespace tq
