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

// Which calls run the GEMV and which the matrix cores, by the GEMV's passes over the
// weights (us at cold weights, both sides; the two code types alike):
//  * up to 4 tokens the GEMV (N = K = 4096: 7 against 16 at 4; N = 4096, K = 8192, two
//    passes: 16.5 against 22.4), but for wide outputs of rows of 8 K to 10 K, which leave
//    half of the GEMV's lanes idle (N = 14336, K = 8960 at 4 tokens: 54 against 48; N =
//    12288, K = 16384: 51 against 74);
//  * 5 to 8 tokens of aligned rows up to 4096, two passes, while these are short (N = K =
//    4096: 12.1-13.5 against 16; N = 12288: 25-28 against 28; N = 14336: 27-31 against
//    28; N = 8192, K = 512 9.5 against 10; N = 16384, K = 256 14 against 8);
//  * aligned rows up to 8192, three or four passes: N = 4096, K = 6144 at 6 tokens 19.4
//    against 19.5, K = 8192 24 against 22; at 8 N = 1024, K = 8192 16.4 against 17.5, N =
//    2048 22 against 18;
//  * other rows up to 512, a wave per output: N = 15000, K = 300 21 against 9 at 5;
//  * other rows up to 2048, one pass of 8: N = 8000, K = 1000 10.2 against 12.8; longer,
//    two of 4: N = 1024, K = 14336 18.4 against 21.9 at 8, N = 4096, K = 4097 21 against
//    18 at 5;
//  * past 8 the matrix cores (N = K = 4096 at 12: 20 against 16).
bool gemv_runs(int64_t m, int64_t n, int64_t k) {
    if (m > 8) return false;
    if (k <= 4096 && k % 16 == 0) return m <= 4 || (n <= (k < 1024 ? 8192 : 12288) && n * k <= 48 << 20);
    if (k <= 8192 && k % 16 == 0) return m <= 4 || n * k <= (m <= 6 ? 24 << 20 : 8 << 20);
    if (m <= 4) return m < 4 || k > 10240 || n * k <= 96 << 20;
    if (k <= 512) return n * k <= 2 << 20;
    return k <= 2048 ? n * k <= 8 << 20 : n <= 1024;
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
    if (n <= 0 || k <= 0 || gemv_runs(m, n, k) || tiny(m, n, k) || !tile_fits(m, n, k)) return 0;
    return tile_plan<T>(m, n, k, nullptr, true).part_bytes;
}

template <class T>
int weight_only(const float* x, int64_t m, const typename T::W::elem_t* q, const float* s, const float* bias,
                int64_t n, int64_t k, void* workspace, int64_t workspace_bytes, float* y, tq_stream_t stream,
                const char* what) {
    TQ_REQUIRE(m >= 0 && n >= 0 && k >= 0, "%s: negative shape", what);
    if (m == 0 || n == 0) return TQ_OK;
    TQ_REQUIRE(y && s && (k == 0 || (x && q)), "%s: null pointer", what);
    TQ_REQUIRE(aligned(x, 4) && aligned(s, 4) && (!bias || aligned(bias, 4)) && aligned(y, 4),
               "%s: misaligned f32 pointer", what);
    if (gemv_runs(m, n, k)) return launch_gemv(x, m, q, s, bias, n, k, y, stream);
    const hipStream_t st = as_hip(stream);
    if (tiny(m, n, k) || !tile_fits(m, n, k)) return launch_linear_8bit_generic(x, m, q, s, bias, n, k, y, st);
    const TilePlan plan = tile_plan<T>(m, n, k, nullptr, true);
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
