// tq_gemm_w8.hip -- 8-bit weight-only quantized Linear beyond a few tokens: f32
// activations times per-row INT8 or FP8 (e4m3) codes on the matrix cores,
//
//   y[m, n] = sw[n] * sum_k x[m, k] * value(q[n, k]) (+ b[n]),
//
// the reference's Linear::forward (crates/theano-nn/src/linear.rs:111-121) over
// the dequantized weight.  The GEMV (tq_gemv.hip) reads the weights once per 4
// tokens; here they are read once per 32 to 128.  Which one runs: gemv_runs below.
// The activations go through the tile kernel as three exact bf16 planes (GemmF32).
#include "tq_gemm_tile.h"

namespace tq {
namespace {

// Which calls run the GEMV (passes over the weights of 4 tokens, of 2 past K = 4096)
// and which the matrix cores, whose split and finish launches cost ~6 us: up to 4
// tokens the GEMV (N = K = 4096: 6.9 us at 4; N = 4096, K = 8192: 16 us on both); past
// 8 the matrix cores (13 against 18 us at 9); between, the GEMV while a pass over the
// weights is short (N = K = 4096: 11.5-13.5 us against 13; N = 14336, K = 4096: 29-34
// against 20; N = 4096, K = 4097, 24-33 against 15).  The FP8 form's matrix kernel
// takes longer: the GEMV's aligned form keeps all of its 5 to 8 tokens.
// Long rows of many outputs go over from 2 INT8 tokens on, at x's traffic (N = 14336, K =
// 8960: 36 / 45 / 53 us at 2 / 3 / 4 tokens against 33; N = 4096, K = 16384: 16 / 19 / 21
// against 24).
bool gemv_runs(int64_t m, int64_t n, int64_t k, bool fp8) {
    if (!fp8 && m > 1 && k > 8192 && n * k > 96 << 20) return false;
    if (m <= 4 || m > 8) return m <= 4;
    const bool vec16 = k % 16 == 0 && k <= 8192;
    return vec16 ? fp8 || n * k <= 4096 * 4096 : n * k <= 2 << 20;
}
// So little work that one launch of a wave per output is ahead (N = 1000, K = 100: 3.9
// against 7.1 us at 16 tokens).
bool tiny(int64_t m, int64_t n, int64_t k) { return k < 16 || (m * n <= 1 << 22 && m * n * k <= 4 << 20); }

int launch_gemv(const float* x, int64_t m, const int8_t* q, const float* s, const float* b, int64_t n, int64_t k,
                float* y, tq_stream_t st) {
    return tq_gemv_w8(x, m, q, s, b, n, k, y, st);
}
int launch_gemv(const float* x, int64_t m, const uint8_t* q, const float* s, const float* b, int64_t n, int64_t k,
                float* y, tq_stream_t st) {
    return tq_gemv_fp8(x, m, q, s, b, n, k, y, st);
}

template <class T>
int64_t workspace_bytes(int64_t m, int64_t n, int64_t k) {
    constexpr bool kFp8 = __is_same(T, GemmF8W);
    if (n <= 0 || k <= 0 || gemv_runs(m, n, k, kFp8) || tiny(m, n, k) || !tile_fits(m, n, k)) return 0;
    return tile_plan<T>(m, n, k, 0, true).part_bytes;
}

template <class T>
int weight_only(const float* x, int64_t m, const typename T::W::elem_t* q, const float* s, const float* bias,
                int64_t n, int64_t k, void* workspace, int64_t workspace_bytes, float* y, tq_stream_t stream,
                const char* what) {
    constexpr bool kFp8 = __is_same(T, GemmF8W);
    TQ_REQUIRE(m >= 0 && n >= 0 && k >= 0, "%s: negative shape", what);
    if (m == 0 || n == 0) return TQ_OK;
    TQ_REQUIRE(y && s && (k == 0 || (x && q)), "%s: null pointer", what);
    TQ_REQUIRE(aligned(x, 4) && aligned(s, 4) && (!bias || aligned(bias, 4)) && aligned(y, 4),
               "%s: misaligned f32 pointer", what);
    if (gemv_runs(m, n, k, kFp8)) return launch_gemv(x, m, q, s, bias, n, k, y, stream);
    const hipStream_t st = as_hip(stream);
    if (tiny(m, n, k) || !tile_fits(m, n, k)) return launch_linear_8bit_generic(x, m, q, s, bias, n, k, y, st);
    const TilePlan plan = tile_plan<T>(m, n, k, 0, true);
    TQ_REQUIRE(plan.part_bytes == 0 || (workspace && aligned(workspace, 8) && workspace_bytes >= plan.part_bytes),
               "%s: workspace of %lld bytes, %lld needed", what, (long long)workspace_bytes,
               (long long)plan.part_bytes);
    TileArgs p{};
    p.a = x;
    p.w = q;
    p.sw = s;
    p.bias = bias;
    p.m = static_cast<int>(m);
    p.n = static_cast<int>(n);
    p.k = static_cast<int>(k);
    p.y = y;
    p.part = workspace;
    return launch_tile<T>(plan, p, st, what);
}

}  // namespace
}  // namespace tq

using namespace tq;

extern "C" {

int64_t tq_gemm_w8_workspace_bytes(int64_t m, int64_t n, int64_t k) { return workspace_bytes<GemmI8W>(m, n, k); }

int tq_gemm_w8(const float* x, int64_t m, const int8_t* q, const float* s, const float* bias, int64_t n, int64_t k,
               void* workspace, int64_t workspace_bytes, float* y, tq_stream_t stream) {
    return weight_only<GemmI8W>(x, m, q, s, bias, n, k, workspace, workspace_bytes, y, stream, "tq_gemm_w8");
}

int64_t tq_gemm_fp8_weight_workspace_bytes(int64_t m, int64_t n, int64_t k) {
    return workspace_bytes<GemmF8W>(m, n, k);
}

int tq_gemm_fp8_weight(const float* x, int64_t m, const uint8_t* q, const float* s, const float* bias, int64_t n,
                       int64_t k, void* workspace, int64_t workspace_bytes, float* y, tq_stream_t stream) {
    return weight_only<GemmF8W>(x, m, q, s, bias, n, k, workspace, workspace_bytes, y, stream, "tq_gemm_fp8_weight");
}

}  // extern "C"
