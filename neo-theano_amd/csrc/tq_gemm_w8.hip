// tq_gemm_w8.hip -- 8-bit weight-only quantized Linear beyond a few tokens: f32
// activations times per-row INT8 or FP8 (e4m3) codes on the matrix cores,
//
//   y[m, n] = sw[n] * sum_k x[m, k] * value(q[n, k]) (+ b[n]),
//
// the reference's Linear::forward (crates/theano-nn/src/linear.rs:111-121) over
// the dequantized weight.  The GEMV (tq_gemv.hip) reads the weights once per 4
// tokens; here they are read once per 16 to 32 (digit rows) or 64 tokens.  Which one
// runs: gemv_runs below.
//
// INT8: the activations become digit rows (tq_digits.h, one small launch) and the
// product is the W8A8 GEMM's with four digit rows per token: the LDS-DMA kernel's
// 128 x 256 tiles or the register-staged ones (tq_gemm_tile.h).  At M = 512, N = K
// = 4096 the three bf16 planes of the FP8 form take 69 us on INT8 codes, the digits
// 5 + 36 us, and are the more exact ones.
// FP8: e4m3 values span 18 bits, so the activations are split into three bf16
// planes inside the tile kernel instead (GemmF8W).
#include "tq_gemm_dma.h"
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

constexpr int kDmaStageW8 = 1000;  // ns per stage of the DMA kernel's tiles

int64_t align256(int64_t v) { return (v + 255) / 256 * 256; }

struct W8Workspace {
    int64_t lda, ea, part;  // digit row length, byte offsets
};
W8Workspace w8_workspace(int64_t m, int64_t k) {
    W8Workspace w{};
    w.lda = (k + 127) / 128 * 128;
    w.ea = align256(4 * m * w.lda);
    w.part = w.ea + align256(4 * m);
    return w;
}

// sizes the matrix-core kernels take (the digits need room in their int32 sums)
bool w8_fits(int64_t m, int64_t n, int64_t k) { return k <= 65536 && tile_fits(4 * m, n, k); }
bool f8w_fits(int64_t m, int64_t n, int64_t k) { return tile_fits(m, n, k); }

int check_args(const void* x, int64_t m, const void* q, const float* s, const float* bias, int64_t n, int64_t k,
               const float* y, const char* what) {
    TQ_REQUIRE(m >= 0 && n >= 0 && k >= 0, "%s: negative shape", what);
    if (m == 0 || n == 0) return TQ_OK;
    TQ_REQUIRE(y && s && (k == 0 || (x && q)), "%s: null pointer", what);
    TQ_REQUIRE(aligned(x, 4) && aligned(s, 4) && (!bias || aligned(bias, 4)) && aligned(y, 4),
               "%s: misaligned f32 pointer", what);
    return TQ_OK;
}

}  // namespace
}  // namespace tq

using namespace tq;

extern "C" {

int64_t tq_gemm_w8_workspace_bytes(int64_t m, int64_t n, int64_t k) {
    if (n <= 0 || k <= 0 || gemv_runs(m, n, k, false) || tiny(m, n, k) || !w8_fits(m, n, k)) return 0;
    return w8_workspace(m, k).part + tile_plan<GemmW8>(m, n, k, 0, true).part_bytes;
}

int tq_gemm_w8(const float* x, int64_t m, const int8_t* q, const float* s, const float* bias, int64_t n, int64_t k,
               void* workspace, int64_t workspace_bytes, float* y, tq_stream_t stream) {
    const int rc = check_args(x, m, q, s, bias, n, k, y, "tq_gemm_w8");
    if (rc != TQ_OK || m == 0 || n == 0) return rc;
    if (gemv_runs(m, n, k, false)) return tq_gemv_w8(x, m, q, s, bias, n, k, y, stream);
    const hipStream_t st = as_hip(stream);
    if (tiny(m, n, k) || !w8_fits(m, n, k)) return launch_linear_8bit_generic(x, m, q, s, bias, n, k, y, st);
    const int64_t need = tq_gemm_w8_workspace_bytes(m, n, k);
    TQ_REQUIRE(workspace && aligned(workspace, 256) && workspace_bytes >= need,
               "tq_gemm_w8: workspace of %lld bytes (256-byte aligned), %lld needed", (long long)workspace_bytes,
               (long long)need);
    const W8Workspace w = w8_workspace(m, k);
    int8_t* digits = static_cast<int8_t*>(workspace);
    int* ea = reinterpret_cast<int*>(digits + w.ea);
    const int ki = static_cast<int>(k), lda = static_cast<int>(w.lda);
    const int rs = launch_split_rows(x, static_cast<int>(m), ki, lda, digits, ea, st, "tq_gemm_w8 (split)");
    if (rs != TQ_OK) return rs;
    const bool vec = n % 16 == 0 && k % kDmaBK == 0 && aligned(q, 16) && aligned(s, 16) && aligned(y, 16) &&
                     (!bias || aligned(bias, 16));
    const TilePlan plan = tile_plan<GemmW8>(m, n, k, vec ? kDmaStageW8 : 0, true);
    if (plan.shape == kTileDma) {
        const int tm = static_cast<int>((4 * m + kDmaBM - 1) / kDmaBM), tn = static_cast<int>((n + kDmaBN - 1) / kDmaBN);
        k_gemm_w8a8_dma<false, true><<<static_cast<unsigned>(tm * tn), 256, 0, st>>>(
            digits, nullptr, q, s, bias, static_cast<int>(4 * m), static_cast<int>(n), ki, nullptr, y, tm, tn, nullptr,
            DigitArgs{x, ea, static_cast<int>(m)});
        return check_launch("tq_gemm_w8");
    }
    TileArgs p{};
    p.a = digits;
    p.w = q;
    p.ea = ea;
    p.x = x;
    p.sw = s;
    p.bias = bias;
    p.m = static_cast<int>(m);
    p.n = static_cast<int>(n);
    p.k = ki;
    p.lda = lda;
    p.y = y;
    p.part = digits + w.part;
    return launch_tile<GemmW8>(plan, p, st, "tq_gemm_w8");
}

int64_t tq_gemm_fp8_weight_workspace_bytes(int64_t m, int64_t n, int64_t k) {
    if (n <= 0 || k <= 0 || gemv_runs(m, n, k, true) || tiny(m, n, k) || !f8w_fits(m, n, k)) return 0;
    return tile_plan<GemmF8W>(m, n, k, 0, true).part_bytes;
}

int tq_gemm_fp8_weight(const float* x, int64_t m, const uint8_t* q, const float* s, const float* bias, int64_t n,
                       int64_t k, void* workspace, int64_t workspace_bytes, float* y, tq_stream_t stream) {
    const int rc = check_args(x, m, q, s, bias, n, k, y, "tq_gemm_fp8_weight");
    if (rc != TQ_OK || m == 0 || n == 0) return rc;
    if (gemv_runs(m, n, k, true)) return tq_gemv_fp8(x, m, q, s, bias, n, k, y, stream);
    const hipStream_t st = as_hip(stream);
    if (tiny(m, n, k) || !f8w_fits(m, n, k)) return launch_linear_8bit_generic(x, m, q, s, bias, n, k, y, st);
    const TilePlan plan = tile_plan<GemmF8W>(m, n, k, 0, true);
    TQ_REQUIRE(plan.part_bytes == 0 || (workspace && aligned(workspace, 8) && workspace_bytes >= plan.part_bytes),
               "tq_gemm_fp8_weight: workspace of %lld bytes, %lld needed", (long long)workspace_bytes,
               (long long)plan.part_bytes);
    TileArgs p{};
    p.a = x;
    p.w = q;
    p.sw = s;
    p.bias = bias;
    p.m = static_cast<int>(m);
    p.n = static_cast<int>(n);
    p.k = static_cast<int>(k);
    p.lda = p.k;
    p.y = y;
    p.part = workspace;
    return launch_tile<GemmF8W>(plan, p, st, "tq_gemm_fp8_weight");
}

}  // extern "C"
