// tq_mlp.hip -- prefill-shaped INT4 group-128 Linear (W4A16) and the quantized
// Llama-style FFN on the register-staged tiles of tq_gemm_tile.h, for the shapes and
// alignments that the pipelined kernels of tq_ffn.hip do not take and for the ones
// whose tiles would leave most compute units idle.
//
// Reference composition: Linear::forward (crates/theano-nn/src/linear.rs:111-121)
// over dequantized weights, SiLU (crates/theano-nn/src/activation.rs:66-79,
// x * 1/(1+exp(-x))) and Tensor::mul, all in f64; here f32 accumulation.
//
// The INT4 codes widen to bf16 exactly, so a group's 128 products are exact and its
// f32 sum is scaled once; the down projection takes the f32 h = SiLU(gate) * up as
// bf16 hi + lo planes.  M = 389, N = 5827, K = 256: 8.3 us, against 300 us for a wave
// per output (N % 16 != 0 had no other kernel); FFN at M = 889, D = 4096, F = 384: 44
// us with its weights read past the caches, against 170 us for 128-row tiles that ran K
// unsplit.
#include "tq_gemm_tile.h"

namespace tq {
namespace {

int64_t align256(int64_t v) { return (v + 255) / 256 * 256; }

TileArgs w4_args(const void* a, const uint8_t* packed, const uint16_t* s, const float* bias, int64_t m, int64_t n,
                 int64_t k, float* y, void* part) {
    TileArgs p{};
    p.a = a;
    p.w = packed;
    p.sg = s;
    p.bias = bias;
    p.m = static_cast<int>(m);
    p.n = static_cast<int>(n);
    p.k = static_cast<int>(k);
    p.y = y;
    p.part = part;
    return p;
}

// So little work that a wave per output in one launch is ahead.
bool tiny(int64_t m, int64_t n, int64_t k) { return m * n <= 1 << 22 && m * n * k <= 1 << 20; }

}  // namespace

W4TileCost w4_linear_tile_cost(int64_t m, int64_t n, int64_t k) {
    if (k == 0 || tiny(m, n, k) || !tile_fits(m, n, k)) return W4TileCost{0, 0};
    const TilePlan plan = tile_plan<GemmW4>(m, n, k, nullptr, true);
    return W4TileCost{plan.ns, plan.part_bytes};
}

int launch_w4_linear_tile(const uint16_t* x_bf16, int64_t m, const uint8_t* packed, const uint16_t* s_f16,
                          const float* bias, int64_t n, int64_t k, void* part, float* y, hipStream_t st,
                          const char* what) {
    if (k == 0 || tiny(m, n, k) || !tile_fits(m, n, k))
        return launch_linear_w4_generic(x_bf16, m, packed, s_f16, bias, n, k, y, st);
    const TilePlan plan = tile_plan<GemmW4>(m, n, k, nullptr, part != nullptr);
    return launch_tile<GemmW4>(plan, w4_args(x_bf16, packed, s_f16, bias, m, n, k, y, part), st, what);
}

W4TileCost mlp_tile_cost(int64_t m, int64_t d, int64_t f) {
    if (!tile_fits(m, 2 * f, d) || !tile_fits(m, d, f)) return W4TileCost{INT64_MAX, 0};
    const TilePlan gu = tile_plan<GemmW4GateUp>(m, 2 * f, d, nullptr, true), dn = tile_plan<GemmW4H>(m, d, f, nullptr, true);
    return W4TileCost{gu.ns + dn.ns, align256(4 * m * f) + std::max(gu.part_bytes, dn.part_bytes)};
}

int launch_mlp_tile(const uint16_t* x_bf16, int64_t m, int64_t d, int64_t f, const uint8_t* gate_packed,
                    const uint16_t* gate_s, const uint8_t* up_packed, const uint16_t* up_s, const uint8_t* down_packed,
                    const uint16_t* down_s, void* workspace, bool may_split, float* y, hipStream_t st) {
    TQ_REQUIRE(tile_fits(m, 2 * f, d) && tile_fits(m, d, f), "tq_mlp_w4g128: problem too large");
    float* h = static_cast<float*>(workspace);
    void* part = static_cast<uint8_t*>(workspace) + align256(4 * m * f);
    TileArgs gu = w4_args(x_bf16, gate_packed, gate_s, nullptr, m, 2 * f, d, h, part);
    gu.w2 = up_packed;
    gu.sg2 = up_s;
    const int rc = launch_tile<GemmW4GateUp>(tile_plan<GemmW4GateUp>(m, 2 * f, d, nullptr, may_split), gu, st,
                                             "tq_mlp_w4g128 (gate/up)");
    if (rc != TQ_OK) return rc;
    return launch_tile<GemmW4H>(tile_plan<GemmW4H>(m, d, f, nullptr, may_split),
                                w4_args(h, down_packed, down_s, nullptr, m, d, f, y, part), st,
                                "tq_mlp_w4g128 (down)");
}

}  // namespace tq

using namespace tq;

extern "C" {

int tq_gemm_w4g128_bf16(const uint16_t* x_bf16, int64_t m, const uint8_t* packed,
                        const uint16_t* s_f16, const float* bias, int64_t n, int64_t k, float* y,
                        tq_stream_t stream) {
    TQ_REQUIRE(m >= 0 && n >= 0 && k >= 0, "tq_gemm_w4g128_bf16: negative shape");
    TQ_REQUIRE(k % 128 == 0, "tq_gemm_w4g128_bf16: K=%lld is not a multiple of 128", (long long)k);
    if (m == 0 || n == 0) return TQ_OK;
    TQ_REQUIRE(y && (k == 0 || (x_bf16 && packed && s_f16)), "tq_gemm_w4g128_bf16: null pointer");
    TQ_REQUIRE(aligned(x_bf16, 2) && aligned(s_f16, 2) && aligned(y, 4) && (!bias || aligned(bias, 4)),
               "tq_gemm_w4g128_bf16: misaligned pointer");
    return launch_w4_linear_tile(x_bf16, m, packed, s_f16, bias, n, k, nullptr, y, as_hip(stream),
                                 "tq_gemm_w4g128_bf16");
}

}  // extern "C"
