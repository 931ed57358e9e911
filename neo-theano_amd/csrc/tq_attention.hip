// tq_attention.hip -- the attention core of MultiheadAttention::forward_with_mask
// (crates/theano-nn/src/transformer.rs:95-142) on gfx950, for the quantized
// q/k/v/out projections around it:
//
//   scores = (Q_h K_h^T) * (1 / sqrt(head_dim))       (+ mask, broadcast over heads)
//   P      = softmax(scores, -1)                       (tensor_ops.rs:574-620)
//   O_h    = P V_h,   heads concatenated along the embedding
//
// f32 inputs, outputs, softmax and accumulators.  Q, K and V are row-major [B*S, ld] matrices whose head h
// occupies columns [h*D, (h+1)*D) (the fused QKV projection's output is read in
// place with ld = 3E); O is [B*S, ldo].
//
// One block per (128 queries, head, batch): 4 waves of 32 query rows on the
// bf16 matrix cores (v_mfma_f32_32x32x16_bf16).  Every f32 operand is split
// exactly into bf16 hi = bf16(v) and lo = bf16(v - hi) (|v - hi - lo| <=
// 2^-18 |v|), and each product runs as hi*hi + hi*lo + lo*hi, all bf16 products
// exact in the f32 accumulators; the dropped lo*lo term is below 2^-16 of the
// product.  Keys run in tiles of 32, staged in LDS for the 4 waves as hi and lo
// planes (K row-major, V transposed, both padded against bank conflicts), the
// next tile's loads in flight during the current tile's work.  Scores are kept
// in log2 units (scale * log2(e), the mask likewise), so each probability is
// one v_exp_f32 (2^x).  Per tile a wave computes S^T = K Q^T (lane = query, registers = keys, so the softmax of a
// query row is in-lane plus one partner lane), updates its running max / sum,
// and accumulates O^T += V^T P^T with the probabilities as they came out of the
// first product: lane half g holds keys 8a + 4g + b (a, b < 4), and the
// transposed V tile stores key k at column k with bits 2 and 3 swapped, so the
// 8 keys of a 16-key MFMA step are one contiguous 16-byte read.  The head
// dimension is padded with zeros to 32, 64, 96 or 128.  A running max of -inf
// (every key so far masked) leaves the row untouched; a row masked everywhere
// ends as 0/0 = NaN, as the reference's softmax gives.
//
// With D % 4 == 0 and 16-byte aligned K and V rows (k_attention_vec) a thread
// loads K as 16-byte quads along d and V as four keys at one d (coalesced
// along d across the wave), both stored to LDS as 8-byte runs, with offsets
// fixed per thread and a uniform step per item, so whole tiles load without
// clamps; it fits two waves per SIMD in 256 registers.  Other head dimensions
// keep the per-element loads (k_attention, one wave per SIMD).  Head dims past 64
// run blocks of 3 or 6 waves (96 wide) and 4 or 8 (128 wide; up to 256 queries, each
// key tile loaded and split once for all of them), as tq_attention_f32 picks by the
// rounds of blocks over the CUs.  All forms give the same bits.
#include <cmath>

#include "tq_internal.h"

namespace tq {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef f32x4 f32x4_a4 __attribute__((aligned(4)));

constexpr int kWaves = 4;           // waves per block (8 in the wide form)
constexpr int kQW = 32;              // query rows per wave
constexpr int kKT = 32;              // keys per tile
constexpr int kMaxD = 128;

__device__ __forceinline__ f32x16 mfma_bf16(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
}

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// a, b -> packed bf16 pairs (a low): v = hi + lo (+ < 2^-18 |v|), hi = bf16(v),
// lo = bf16(v - hi).  Both conversions round two values in one instruction, whose
// result is already the packed pair: 3 VALU operations per value.
__device__ __forceinline__ void split2(float a, float b, uint32_t& hi, uint32_t& lo) {
    hi = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{a, b}), bf16x2));
    const float ra = a - __uint_as_float(hi << 16), rb = b - __uint_as_float(hi & 0xFFFF0000u);
    lo = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{ra, rb}), bf16x2));
}

// 8 f32 -> packed bf16 hi and lo
__device__ __forceinline__ void split8(const float* v, u32x4& hi, u32x4& lo) {
    uint32_t h[4], l[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) split2(v[2 * i], v[2 * i + 1], h[i], l[i]);
    hi = u32x4{h[0], h[1], h[2], h[3]};
    lo = u32x4{l[0], l[1], l[2], l[3]};
}

// A lane's value and its partner's 32 lanes away, combined (v_permlane32_swap_b32, a
// vector operation; __shfl_xor is a round trip through LDS).
template <class Op>
__device__ __forceinline__ float with_partner(float v, Op op) {
    const uint32_t u = __float_as_uint(v);
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return op(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

__device__ __forceinline__ int vcol(int key) { return (key & ~12) | ((key & 4) << 1) | ((key & 8) >> 1); }

// kVec: D % 4 == 0 and 16-byte aligned rows of K and V, loaded as whole quads.
// kW waves per block share each key tile (kW x 32 queries).
template <int kDP, bool kVec, int kW>
__device__ __forceinline__ void attention_block(const float* __restrict__ q, int64_t ldq,
                                                              const float* __restrict__ k, int64_t ldk,
                                                              const float* __restrict__ v, int64_t ldv,
                                                              const float* __restrict__ mask, int64_t mask_batch,
                                                              int S, int D, float scale, float* __restrict__ o,
                                                              int64_t ldo) {
    constexpr int kSteps = kDP / 16;   // 16-wide d steps of S^T = K Q^T
    constexpr int kKRow = kDP + 8;     // K plane row (bf16), padded
    constexpr int kVRow = kKT + 8;     // transposed V plane row (bf16), padded
    constexpr int kBlocks = kDP / 32;  // 32-wide d blocks of O^T
    constexpr int kElems = kKT * kDP / (kW * kWave);  // tile elements per thread (K and V each)
    constexpr bool kMaskEarly = kElems * kDP < 16 * 128;  // not the narrow form at 128
    static_assert(!kVec || kElems % 4 == 0, "whole quads per thread");
    __shared__ __attribute__((aligned(16))) uint16_t ksh[2][kKT * kKRow], ksl[2][kKT * kKRow];
    __shared__ __attribute__((aligned(16))) uint16_t vsh[2][kDP * kVRow], vsl[2][kDP * kVRow];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 5, lr = lane & 31;
    const int h = blockIdx.y, b = blockIdx.z;
    const int qrow = blockIdx.x * (kW * kQW) + wave * kQW + lr;  // this lane's query row
    const int64_t base = static_cast<int64_t>(b) * S;
    const int col = h * D;
    constexpr float kLog2e = 1.4426950408889634f;
    const float scale2 = scale * kLog2e;

    // Q operand: step s covers d = 16 s + 8 g + j (rows past S read row S-1; never stored)
    u32x4 qh[kSteps], ql[kSteps];
    {
        const float* qr = q + (base + min(qrow, S - 1)) * ldq + col;
#pragma unroll
        for (int st = 0; st < kSteps; ++st) {
            float qv[8];
            if constexpr (kVec) {  // whole quads (D % 4 == 0), any alignment
#pragma unroll
                for (int j = 0; j < 8; j += 4) {
                    const int d = 16 * st + 8 * g + j;
                    const f32x4 t = *reinterpret_cast<const f32x4_a4*>(qr + min(d, D - 4));
#pragma unroll
                    for (int e = 0; e < 4; ++e) qv[j + e] = d < D ? t[e] : 0.f;
                }
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int d = 16 * st + 8 * g + j;
                    qv[j] = qr[min(d, D - 1)];
                    qv[j] = d < D ? qv[j] : 0.f;
                }
            }
            split8(qv, qh[st], ql[st]);
            // (the raw values of two steps in registers at a time)
            if (st % 2 == 1) __builtin_amdgcn_sched_barrier(0);
        }
    }
    const float* mrow =
        mask ? mask + ((mask_batch == 1 ? 0 : static_cast<int64_t>(b)) * S + min(qrow, S - 1)) * static_cast<int64_t>(S)
             : nullptr;

    // tile loads.  Scalar: element e = tid + 256 i -> key e / kDP, d e % kDP
    // (coalesced along d).  kVec: K item e -> key e / (kDP / 4), the quad of d
    // from 4 (e % (kDP / 4)), one 16-byte load; V item e -> d = e % kDP and keys
    // 4 (e / kDP) .. + 3, four loads coalesced along d across the wave, so that
    // both land in LDS as 8-byte runs (K along d, the transposed V along keys).
    // Rows past S and d past D read clamped addresses and are zeroed.
    constexpr int kQuads = kElems / 4;  // K and V items per thread (kVec)
    float kreg[kElems], vreg[kElems];
    // kVec: the element offsets of item 0 from its tile's first row (the host
    // keeps a tile's offsets below 2^31) and whether its d is inside the head;
    // item i has the same d and keys 256 i / (kDP / 4) (K) or 4 (256 i / kDP)
    // (V) further on
    constexpr int kKeyStepK = kW * kWave / (kDP / 4), kKeyStepV = 4 * (kW * kWave / kDP);
    const int dq = 4 * (tid % (kDP / 4)), dv = tid % kDP;
    const uint32_t koff = static_cast<uint32_t>((tid / (kDP / 4)) * ldk + col + min(dq, D - 4));
    const uint32_t voff = static_cast<uint32_t>(4 * (tid / kDP) * ldv + col + min(dv, D - 1));
    static_assert(!kVec || kW * kWave % kDP == 0, "an item's column does not depend on the item");
    const bool kin = dq < D, vin = dv < D;
    // The loads leave their registers untouched until the tile is stored: zeroing them
    // here made every tile wait for its successor's loads before its own MFMAs.
    auto load_tile = [&](int j0) {
        if constexpr (kVec) {
            if (j0 + kKT <= S) {  // a whole tile (uniform): no row clamps
#pragma unroll
                for (int i = 0; i < kQuads; ++i) {
                    const float* kb = k + (base + j0 + i * kKeyStepK) * ldk;
                    const float4 kv = *reinterpret_cast<const float4*>(kb + koff);
                    kreg[4 * i] = kv.x;
                    kreg[4 * i + 1] = kv.y;
                    kreg[4 * i + 2] = kv.z;
                    kreg[4 * i + 3] = kv.w;
#pragma unroll
                    for (int r = 0; r < 4; ++r) vreg[4 * i + r] = (v + (base + j0 + i * kKeyStepV + r) * ldv)[voff];
                }
                return;
            }
            // the last, partial tile: rows clamped, as 32-bit offsets from its first
            const float* kt = k + (base + j0) * ldk;
            const float* vt = v + (base + j0) * ldv;
            const uint32_t lk = static_cast<uint32_t>(ldk), lv = static_cast<uint32_t>(ldv);
#pragma unroll
            for (int i = 0; i < kQuads; ++i) {
                const int e = tid + i * kW * kWave;
                const uint32_t key = min(e / (kDP / 4), S - 1 - j0);
                const f32x4 kv = *reinterpret_cast<const f32x4*>(kt + (key * lk + col + min(dq, D - 4)));
                kreg[4 * i] = kv.x;
                kreg[4 * i + 1] = kv.y;
                kreg[4 * i + 2] = kv.z;
                kreg[4 * i + 3] = kv.w;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const uint32_t kr = min(4 * (e / kDP) + r, S - 1 - j0);
                    vreg[4 * i + r] = vt[kr * lv + col + min(dv, D - 1)];
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < kElems; ++i) {
                const int e = tid + i * kW * kWave, key = e / kDP, d = e % kDP;
                const int64_t row = base + min(j0 + key, S - 1);
                kreg[i] = k[row * ldk + col + min(d, D - 1)];
                vreg[i] = v[row * ldv + col + min(d, D - 1)];
            }
        }
    };
    // the tile of keys j0 .. j0 + 31 into buffer `buf`, zeros past S and past D
    auto store_tile = [&](int buf, int j0) {
        if constexpr (kVec) {
#pragma unroll
            for (int i = 0; i < kQuads; ++i) {
                const int e = tid + i * kW * kWave;
                const int key = e / (kDP / 4), k4 = 4 * (e / kDP);
                const bool ok = kin && j0 + key < S;
                uint32_t h[2], l[2];
#pragma unroll
                for (int r = 0; r < 2; ++r)
                    split2(ok ? kreg[4 * i + 2 * r] : 0.f, ok ? kreg[4 * i + 2 * r + 1] : 0.f, h[r], l[r]);
                *reinterpret_cast<uint2*>(&ksh[buf][key * kKRow + dq]) = make_uint2(h[0], h[1]);
                *reinterpret_cast<uint2*>(&ksl[buf][key * kKRow + dq]) = make_uint2(l[0], l[1]);
#pragma unroll
                for (int r = 0; r < 2; ++r)
                    split2(vin && j0 + k4 + 2 * r < S ? vreg[4 * i + 2 * r] : 0.f,
                           vin && j0 + k4 + 2 * r + 1 < S ? vreg[4 * i + 2 * r + 1] : 0.f, h[r], l[r]);
                // keys 4a .. 4a + 3 sit at 4 consecutive columns of the transposed tile
                *reinterpret_cast<uint2*>(&vsh[buf][dv * kVRow + vcol(k4)]) = make_uint2(h[0], h[1]);
                *reinterpret_cast<uint2*>(&vsl[buf][dv * kVRow + vcol(k4)]) = make_uint2(l[0], l[1]);
            }
        } else {
#pragma unroll
            for (int i = 0; i < kElems; ++i) {
                const int e = tid + i * kW * kWave, key = e / kDP, d = e % kDP;
                const bool ok = j0 + key < S && d < D;
                uint32_t hi, lo;
                split2(ok ? kreg[i] : 0.f, ok ? vreg[i] : 0.f, hi, lo);
                ksh[buf][key * kKRow + d] = static_cast<uint16_t>(hi);
                ksl[buf][key * kKRow + d] = static_cast<uint16_t>(lo);
                vsh[buf][d * kVRow + vcol(key)] = static_cast<uint16_t>(hi >> 16);
                vsl[buf][d * kVRow + vcol(key)] = static_cast<uint16_t>(lo >> 16);
            }
        }
    };

    f32x16 ot[kBlocks];
#pragma unroll
    for (int c = 0; c < kBlocks; ++c) ot[c] = f32x16{};
    float m = -INFINITY, l = 0.f;  // l: this lane's half of the row's sum

    load_tile(0);
    store_tile(0, 0);
    __syncthreads();
    int buf = 0;
    for (int j0 = 0; j0 < S; j0 += kKT) {
        const bool more = j0 + kKT < S;
        if (more) load_tile(j0 + kKT);  // in flight during this tile

        // the mask's 16 values of this lane: keys 8 a + 4 g .. + 3, as quads (at 4-byte
        // alignment: a mask row is S values) in whole tiles.  In flight during the first
        // product where the registers hold them (kMaskEarly).
        f32x4 mk[4];
        auto load_mask = [&]() {
            if (j0 + kKT <= S) {
                asm volatile("");
#pragma unroll
                for (int a = 0; a < 4; ++a) mk[a] = *reinterpret_cast<const f32x4_a4*>(mrow + j0 + 8 * a + 4 * g);
            } else {
#pragma unroll
                for (int r = 0; r < 16; ++r) mk[r >> 2][r & 3] = mrow[min(j0 + 8 * (r >> 2) + 4 * g + (r & 3), S - 1)];
            }
        };
        if (kMaskEarly && mask) {
            asm volatile("");
            load_mask();
        }
        // S^T[key][q] = sum_d K[key][d] Q[q][d]: lane holds keys 8(r/4) + 4g + r%4 of query lr
        f32x16 st = f32x16{};
        {
            const uint16_t* kh = &ksh[buf][lr * kKRow + 8 * g];
            const uint16_t* kl = &ksl[buf][lr * kKRow + 8 * g];
#pragma unroll
            for (int s2 = 0; s2 < kSteps; ++s2) {
                const u32x4 a_h = *reinterpret_cast<const u32x4*>(kh + 16 * s2);
                const u32x4 a_l = *reinterpret_cast<const u32x4*>(kl + 16 * s2);
                st = mfma_bf16(a_h, qh[s2], st);
                st = mfma_bf16(a_h, ql[s2], st);
                st = mfma_bf16(a_l, qh[s2], st);
            }
        }
        // scores in log2 units: s * scale * log2(e) (+ mask * log2(e)), so that the
        // probabilities are one v_exp_f32 (2^x) each.  Without a mask the scale goes
        // into the exponent's fma, the maximum being taken of the products.
        float p[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) p[r] = st[r];
        float unit = scale2;
        // `mask` (a kernel argument) and the tile are uniform: real branches (the empty
        // statement keeps the compiler from computing both sides)
        if (mask) {
            asm volatile("");
            unit = 1.0f;
            if (!kMaskEarly) load_mask();
#pragma unroll
            for (int r = 0; r < 16; ++r) p[r] = fmaf(mk[r >> 2][r & 3], kLog2e, p[r] * scale2);
        }
        if (j0 + kKT > S) {
            asm volatile("");
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (j0 + 8 * (r >> 2) + 4 * g + (r & 3) >= S) p[r] = -INFINITY;
        }
        float mt = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; ++r) mt = fmaxf(mt, p[r]);
        mt *= unit;
        mt = with_partner(mt, OpMax{});  // the partner lane holds the other 16 keys
        const float mn = fmaxf(m, mt);
        const float base_m = mn == -INFINITY ? 0.f : mn;  // all masked so far: nothing to add
        float ls[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            p[r] = __builtin_amdgcn_exp2f(fmaf(p[r], unit, -base_m));
            ls[r & 3] += p[r];
        }
        const float alpha = __builtin_amdgcn_exp2f(m - base_m);
        l = fmaf(l, alpha, (ls[0] + ls[1]) + (ls[2] + ls[3]));
        m = mn;
        // P^T operand: step t of 16 keys takes registers 8t .. 8t+7 (keys 16t + 8h + 4g + b,
        // slot 4h + b), the order of the transposed V tile's columns
        u32x4 ph[2], pl[2];
        split8(p, ph[0], pl[0]);
        split8(p + 8, ph[1], pl[1]);
        // O^T[d][q] += sum_key V[key][d] P[q][key]
        // alpha is 1 in every lane once the running maxima settle: the rescale is skipped
        if (__ballot(alpha != 1.0f) != 0) {
            // in place: multiplies that the compiler may give other destinations made it
            // hold the running output twice, with as many copies a tile.  It places no wait
            // states for inline asm: the products that wrote ot ended a barrier and this
            // tile's scores ago, the next ones follow the split of p, and
            // tests/test_attention_asm.py counts the distances in every instance (statements
            // with the waits of their own took 3 to 5 % at 128 wide, S = 2048).
#pragma unroll
            for (int c = 0; c < kBlocks; ++c)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    float t = ot[c][e];
                    asm volatile("v_mul_f32 %0, %1, %0" : "+v"(t) : "v"(alpha));
                    ot[c][e] = t;
                }
        }
#pragma unroll
        for (int c = 0; c < kBlocks; ++c) {
            const uint16_t* vh = &vsh[buf][(32 * c + lr) * kVRow + 8 * g];
            const uint16_t* vl = &vsl[buf][(32 * c + lr) * kVRow + 8 * g];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const u32x4 a_h = *reinterpret_cast<const u32x4*>(vh + 16 * t);
                const u32x4 a_l = *reinterpret_cast<const u32x4*>(vl + 16 * t);
                ot[c] = mfma_bf16(a_h, ph[t], ot[c]);
                ot[c] = mfma_bf16(a_h, pl[t], ot[c]);
                ot[c] = mfma_bf16(a_l, ph[t], ot[c]);
            }
        }
        if (more) {
            store_tile(buf ^ 1, j0 + kKT);  // the other buffer: last read before the previous barrier
            __syncthreads();
            buf ^= 1;
        }
    }
    l = with_partner(l, OpAdd{});
    // lane holds O^T[d = 32c + 8(r/4) + 4g + r%4][q = lr]
    // (the row formed again from the thread's index: it would hold registers through the loop)
    int t2 = threadIdx.x;
    asm volatile("" : "+v"(t2));
    const int row = blockIdx.x * (kW * kQW) + (t2 >> 6) * kQW + (t2 & 31);
    if (row < S) {
        float* orow = o + (base + row) * ldo + col;
        const float inv = 1.0f / l;
#pragma unroll
        for (int c = 0; c < kBlocks; ++c)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int d = 32 * c + 8 * (r >> 2) + 4 * g + (r & 3);
                if (d < D) orow[d] = ot[c][r] * inv;
            }
    }
}

// Two waves per SIMD where the quad loads leave the registers for them (256 per
// lane); the scalar form keeps one (its element loads need more).  kW: waves, 32
// queries each.
template <int kDP, int kW>
__global__ __launch_bounds__(kW * kWave) __attribute__((amdgpu_waves_per_eu(2))) void k_attention_vec(
    const float* __restrict__ q, int64_t ldq, const float* __restrict__ k, int64_t ldk, const float* __restrict__ v,
    int64_t ldv, const float* __restrict__ mask, int64_t mask_batch, int S, int D, float scale, float* __restrict__ o,
    int64_t ldo) {
    attention_block<kDP, true, kW>(q, ldq, k, ldk, v, ldv, mask, mask_batch, S, D, scale, o, ldo);
}

template <int kDP>
__global__ __launch_bounds__(kWaves * kWave) void k_attention(const float* __restrict__ q, int64_t ldq,
                                                              const float* __restrict__ k, int64_t ldk,
                                                              const float* __restrict__ v, int64_t ldv,
                                                              const float* __restrict__ mask, int64_t mask_batch,
                                                              int S, int D, float scale, float* __restrict__ o,
                                                              int64_t ldo) {
    attention_block<kDP, false, kWaves>(q, ldq, k, ldk, v, ldv, mask, mask_batch, S, D, scale, o, ldo);
}

}  // namespace
}  // namespace tq

using namespace tq;

extern "C" int tq_attention_f32(const float* q, int64_t ldq, const float* k, int64_t ldk, const float* v,
                                int64_t ldv, const float* mask, int64_t mask_batch, int64_t batch, int64_t seq,
                                int64_t heads, int64_t head_dim, float* out, int64_t ldo, tq_stream_t stream) {
    TQ_REQUIRE(batch >= 0 && seq >= 0 && heads >= 0 && head_dim >= 0, "tq_attention_f32: negative shape");
    if (batch == 0 || seq == 0 || heads == 0) return TQ_OK;
    TQ_REQUIRE(head_dim >= 1 && head_dim <= kMaxD, "tq_attention_f32: head_dim=%lld outside [1, %d]",
               (long long)head_dim, kMaxD);
    TQ_REQUIRE(q && k && v && out, "tq_attention_f32: null pointer");
    const int64_t e = heads * head_dim;
    TQ_REQUIRE(ldq >= e && ldk >= e && ldv >= e && ldo >= e, "tq_attention_f32: row stride below heads * head_dim");
    TQ_REQUIRE(mask_batch == 0 || mask_batch == 1 || mask_batch == batch,
               "tq_attention_f32: mask_batch must be 0 (no mask), 1 or batch");
    TQ_REQUIRE(mask_batch == 0 || mask, "tq_attention_f32: null mask");
    TQ_REQUIRE(seq < (int64_t(1) << 30) && heads < 65536 && batch < 65536, "tq_attention_f32: problem too large");
    TQ_REQUIRE(aligned(q, 4) && aligned(k, 4) && aligned(v, 4) && aligned(out, 4) && (!mask || aligned(mask, 4)),
               "tq_attention_f32: misaligned pointer");
    const float scale = static_cast<float>(1.0 / std::sqrt(static_cast<double>(head_dim)));
    const float* mk = mask_batch ? mask : nullptr;
    const int S = static_cast<int>(seq), D = static_cast<int>(head_dim);
    // whole quads of d where every K and V row is 16-byte aligned
    // (and element offsets within a key tile below 2^31)
    const bool vec = head_dim % 4 == 0 && ldk % 4 == 0 && ldv % 4 == 0 && aligned(k, 16) && aligned(v, 16) &&
                     kKT * std::max(ldk, ldv) + e < (int64_t(1) << 31);
    // Waves per block (32 queries each).  Head dims past 64: 8 (6 at up to 96, where a
    // thread's tile items then share a column), each key tile split once for all of them
    // (S = 2048, 32 heads of 128: 218 us against 247 with 4), unless half as many already
    // give at most one block per CU (S = 129, 16 heads of 80: 18.7 against 21.4).  The
    // 6-wave blocks run one to a CU, of 3/4 of the time of the 8-wave ones padded to 128,
    // which take head dims up to 96 where they need that much fewer rounds over the CUs
    // (S = 2048, 32 heads of 80: 196 us against 290; S = 1500: 138 against 118).
    const int64_t cus = device_cu_count();
    auto blocks = [&](int w) { return (seq + w * kQW - 1) / (w * kQW) * heads * batch; };
    auto rounds = [&](int w) { return (blocks(w) + cus - 1) / cus; };
    const bool pad = head_dim > 96 || 4 * rounds(8) < 3 * rounds(6);
    const int most = pad ? 8 : 6;
    const int waves = !vec || head_dim <= 64 ? kWaves : blocks(most / 2) > cus ? most : most / 2;
    const dim3 grid(static_cast<unsigned>((seq + waves * kQW - 1) / (waves * kQW)), static_cast<unsigned>(heads),
                    static_cast<unsigned>(batch));
#define TQ_ATT(KERNEL, ...)                                                                                     \
    KERNEL<__VA_ARGS__><<<grid, waves * kWave, 0, as_hip(stream)>>>(q, ldq, k, ldk, v, ldv, mk, mask_batch, S, D, \
                                                                    scale, out, ldo)
    if (head_dim <= 32) {
        if (vec) TQ_ATT(k_attention_vec, 32, kWaves); else TQ_ATT(k_attention, 32);
    } else if (head_dim <= 64) {
        if (vec) TQ_ATT(k_attention_vec, 64, kWaves); else TQ_ATT(k_attention, 64);
    } else if (vec && !pad) {
        if (waves == 6) TQ_ATT(k_attention_vec, 96, 6); else TQ_ATT(k_attention_vec, 96, 3);
    } else if (vec) {
        if (waves == 8) TQ_ATT(k_attention_vec, 128, 8); else TQ_ATT(k_attention_vec, 128, kWaves);
    } else {
        TQ_ATT(k_attention, 128);
    }
#undef TQ_ATT
    return check_launch("tq_attention_f32");
}
