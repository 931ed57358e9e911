// C++ tests of the host layer (neo-theano_amd/host/theano_quantize.hpp).
//
// The first groups restate the reference crate's own unit tests with the same
// inputs and asserts (crates/theano-quantize/src/{qconfig,quantize,observer}.rs
// and crates/theano-nn/src/linear.rs), run on the GPU through the C++ API.
// The parity group compares the API's results with the C oracle (oracle/,
// test infrastructure) on seeded inputs: f64 results bit-exact, Linear outputs
// within 1e-3 relative / 1e-4 absolute of the oracle's f64 result.
//
// Usage: test_theano_quantize [--cpu]   (--cpu: only the tests that need no GPU)
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <memory>
#include <cstring>
#include <functional>
#include <random>
#include <string>
#include <vector>

#include "../../oracle/tq_oracle.h"
#include "theano_quantize.hpp"
#include "theano_rocm.hpp"
#include "theano_serialize.hpp"

#include <fstream>
#include <map>
#include <unistd.h>

using namespace theano;
using namespace theano::quantize;
using theano::nn::QuantizedLinear;
using theano::nn::QuantizedMLP;
using theano::nn::QuantizedMultiheadAttention;
namespace ser = theano::serialize;

namespace {

struct Case {
    const char* name;
    bool gpu;
    std::function<void()> fn;
};
std::vector<Case>& registry() {
    static std::vector<Case> r;
    return r;
}
struct Reg {
    Reg(const char* n, bool gpu, std::function<void()> f) { registry().push_back({n, gpu, std::move(f)}); }
};

struct Failure : std::runtime_error {
    using std::runtime_error::runtime_error;
};

#define TEST_CPU(name)                                     \
    void name();                                           \
    static Reg reg_##name(#name, false, name);             \
    void name()
#define TEST_GPU(name)                                     \
    void name();                                           \
    static Reg reg_##name(#name, true, name);              \
    void name()
#define ASSERT(cond)                                                                                    \
    do {                                                                                                \
        if (!(cond)) throw Failure(std::string(__FILE__) + ":" + std::to_string(__LINE__) + ": " #cond); \
    } while (0)
#define ASSERT_EQ(a, b) ASSERT((a) == (b))

// bitwise equality of f64 vectors (signed zeros included); any NaN equals any NaN
bool same_bits(const std::vector<double>& a, const std::vector<double>& b) {
    if (a.size() != b.size()) return false;
    for (size_t i = 0; i < a.size(); ++i) {
        if (std::isnan(a[i]) && std::isnan(b[i])) continue;
        if (std::memcmp(&a[i], &b[i], 8) != 0) return false;
    }
    return true;
}

std::vector<double> randn(size_t n, double std, uint64_t seed) {
    std::mt19937_64 g(seed);
    std::normal_distribution<double> d(0.0, std);
    std::vector<double> v(n);
    for (auto& x : v) x = d(g);
    return v;
}

void assert_close(const std::vector<double>& got, const std::vector<double>& ref, const char* what) {
    ASSERT_EQ(got.size(), ref.size());
    for (size_t i = 0; i < got.size(); ++i)
        if (!(std::fabs(got[i] - ref[i]) <= 1e-4 + 1e-3 * std::fabs(ref[i])))
            throw Failure(std::string(what) + ": element " + std::to_string(i) + " got " + std::to_string(got[i]) +
                          " ref " + std::to_string(ref[i]));
}

// ------------------------------------------------------------ qconfig.rs:82-148

TEST_CPU(test_quant_dtype_bits) {
    ASSERT_EQ(QuantDType::Int8.bits(), 8u);
    ASSERT_EQ(QuantDType::UInt8.bits(), 8u);
    ASSERT_EQ(QuantDType::Int4.bits(), 4u);
    ASSERT_EQ(QuantDType::FP8.bits(), 8u);
}

TEST_CPU(test_quant_dtype_signed) {
    ASSERT(QuantDType::Int8.is_signed());
    ASSERT(!QuantDType::UInt8.is_signed());
    ASSERT(QuantDType::Int4.is_signed());
    ASSERT(!QuantDType::FP8.is_signed());
}

TEST_CPU(test_quant_dtype_range) {
    ASSERT_EQ(QuantDType::Int8.qmin(), -128.0);
    ASSERT_EQ(QuantDType::Int8.qmax(), 127.0);
    ASSERT_EQ(QuantDType::UInt8.qmin(), 0.0);
    ASSERT_EQ(QuantDType::UInt8.qmax(), 255.0);
    ASSERT_EQ(QuantDType::Int4.qmin(), -8.0);
    ASSERT_EQ(QuantDType::Int4.qmax(), 7.0);
    ASSERT_EQ(QuantDType::FP8.qmin(), -448.0);
    ASSERT_EQ(QuantDType::FP8.qmax(), 448.0);
}

TEST_CPU(test_qconfig_default_int8) {
    const QConfig cfg = QConfig::default_int8();
    ASSERT(cfg.weight_dtype == QuantDType::Int8);
    ASSERT(cfg.activation_dtype == QuantDType::UInt8);
    ASSERT(cfg.symmetric);
    ASSERT(!cfg.per_channel);
}

TEST_CPU(test_qconfig_default_int4) {
    const QConfig cfg = QConfig::default_int4();
    ASSERT(cfg.weight_dtype == QuantDType::Int4);
    ASSERT(cfg.activation_dtype == QuantDType::Int8);
    ASSERT(cfg.symmetric);
    ASSERT(cfg.per_channel);
}

TEST_CPU(test_qconfig_default_trait) { ASSERT(QConfig::default_().weight_dtype == QuantDType::Int8); }

TEST_CPU(test_quant_dtype_equality) {
    ASSERT(QuantDType::Int8 == QuantDType::Int8);
    ASSERT(QuantDType::Int8 != QuantDType::UInt8);
}

TEST_CPU(test_qconfig_clone) {
    const QConfig cfg = QConfig::default_int8();
    const QConfig cloned = cfg;
    ASSERT(cloned.weight_dtype == cfg.weight_dtype);
    ASSERT(cloned.activation_dtype == cfg.activation_dtype);
    ASSERT_EQ(cloned.symmetric, cfg.symmetric);
    ASSERT_EQ(cloned.per_channel, cfg.per_channel);
}

TEST_CPU(test_tensor_from_slice_checks_shape) {
    bool threw = false;
    try {
        Tensor::from_slice({1.0, 2.0, 3.0}, {2, 2});
    } catch (const TheanoError& e) {
        threw = e.kind() == TheanoError::Kind::ShapeMismatch;
    }
    ASSERT(threw);
    ASSERT_EQ(Tensor::scalar(2.5).item().unwrap(), 2.5);
    ASSERT(Tensor::ones({2, 3}).item().is_err());
}

// ------------------------------------------------------------ quantize.rs:61-136

TEST_GPU(test_quantize_dequantize_roundtrip) {
    const Tensor tensor = Tensor::from_slice({0.0, 0.5, 1.0, -0.5, -1.0}, {5});
    auto [quantized, scale, zp] = quantize_per_tensor(tensor, QuantDType::Int8).unwrap();
    const auto dequantized = dequantize_tensor(quantized, scale, zp);
    const auto original = tensor.to_vec_f64().unwrap();
    for (size_t i = 0; i < original.size(); ++i) ASSERT(std::fabs(original[i] - dequantized[i]) < 0.05);
}

TEST_GPU(test_fake_quantize) {
    const Tensor tensor = Tensor::from_slice({0.1, 0.5, 0.9}, {3});
    const Tensor result = fake_quantize(tensor, 0.01, 0.0, QuantDType::Int8).unwrap();
    ASSERT(result.shape() == std::vector<size_t>{3});
}

TEST_GPU(test_quantize_tensor_clamps) {
    const Tensor tensor = Tensor::from_slice({1000.0, -1000.0}, {2});
    const auto quantized = quantize_tensor(tensor, 1.0, 0.0, QuantDType::Int8).unwrap();
    ASSERT_EQ(quantized[0], 127.0);
    ASSERT_EQ(quantized[1], -128.0);
}

TEST_GPU(test_dequantize_tensor) {
    const std::vector<double> quantized = {0.0, 64.0, 127.0};
    const auto result = dequantize_tensor(quantized, 0.01, 0.0);
    ASSERT_EQ(result.size(), 3u);
    ASSERT(std::fabs(result[0] - 0.0) < 1e-10);
    ASSERT(std::fabs(result[1] - 0.64) < 1e-10);
    ASSERT(std::fabs(result[2] - 1.27) < 1e-10);
}

TEST_GPU(test_quantize_per_tensor_int4) {
    const Tensor tensor = Tensor::from_slice({0.0, 0.5, 1.0}, {3});
    auto [quantized, scale, zp] = quantize_per_tensor(tensor, QuantDType::Int4).unwrap();
    ASSERT_EQ(quantized.size(), 3u);
    for (double q : quantized) ASSERT(q >= -8.0 && q <= 7.0);
    (void)scale;
    (void)zp;
}

TEST_GPU(test_quantize_per_tensor_uint8) {
    const Tensor tensor = Tensor::from_slice({0.0, 0.5, 1.0}, {3});
    auto r = quantize_per_tensor(tensor, QuantDType::UInt8).unwrap();
    for (double q : std::get<0>(r)) ASSERT(q >= 0.0 && q <= 255.0);
}

TEST_GPU(test_fake_quantize_preserves_shape) {
    const Tensor tensor = Tensor::from_slice({1.0, 2.0, 3.0, 4.0, 5.0, 6.0}, {2, 3});
    const Tensor result = fake_quantize(tensor, 0.1, 0.0, QuantDType::Int8).unwrap();
    ASSERT((result.shape() == std::vector<size_t>{2, 3}));
}

TEST_GPU(test_quantize_single_value) {
    const Tensor tensor = Tensor::from_slice({0.5, -0.5}, {2});
    auto [quantized, scale, zp] = quantize_per_tensor(tensor, QuantDType::Int8).unwrap();
    const auto dequantized = dequantize_tensor(quantized, scale, zp);
    ASSERT(std::fabs(0.5 - dequantized[0]) < 0.05);
    ASSERT(std::fabs(-0.5 - dequantized[1]) < 0.05);
}

// ------------------------------------------------------------ observer.rs:142-223

TEST_GPU(test_minmax_observer_basic) {
    MinMaxObserver obs;
    obs.observe({1.0, 2.0, 3.0, -1.0});
    ASSERT_EQ(obs.min_val(), -1.0);
    ASSERT_EQ(obs.max_val(), 3.0);
}

TEST_GPU(test_minmax_observer_multiple_observations) {
    MinMaxObserver obs;
    obs.observe({1.0, 2.0});
    obs.observe({-5.0, 10.0});
    ASSERT_EQ(obs.min_val(), -5.0);
    ASSERT_EQ(obs.max_val(), 10.0);
}

TEST_GPU(test_minmax_observer_uninitialized) {
    const MinMaxObserver obs;
    auto [scale, zp] = obs.compute_scale_zero_point(QuantDType::Int8);
    ASSERT_EQ(scale, 1.0);
    ASSERT_EQ(zp, 0.0);
}

TEST_GPU(test_minmax_observer_scale_zero_point) {
    MinMaxObserver obs;
    obs.observe({0.0, 1.0});
    auto [scale, zp] = obs.compute_scale_zero_point(QuantDType::UInt8);
    ASSERT(std::fabs(scale - 1.0 / 255.0) < 1e-6);
    (void)zp;
}

TEST_GPU(test_minmax_observer_reset) {
    MinMaxObserver obs;
    obs.observe({1.0, 2.0});
    obs.reset();
    ASSERT_EQ(obs.min_val(), INFINITY);
    ASSERT_EQ(obs.max_val(), -INFINITY);
    auto [scale, zp] = obs.compute_scale_zero_point(QuantDType::Int8);
    ASSERT_EQ(scale, 1.0);
    ASSERT_EQ(zp, 0.0);
}

TEST_GPU(test_per_channel_observer) {
    PerChannelMinMaxObserver obs(2);
    obs.observe({1.0, 2.0, 3.0, -1.0, 0.0, 1.0});
    ASSERT_EQ(obs.scales_and_zero_points(QuantDType::Int8).size(), 2u);
}

TEST_GPU(test_per_channel_observer_reset) {
    PerChannelMinMaxObserver obs(3);
    obs.observe({1.0, 2.0, 3.0});
    obs.reset();
    auto [scale, zp] = obs.compute_scale_zero_point(QuantDType::Int8);
    ASSERT(scale > 0.0);
    (void)zp;
}

TEST_GPU(test_minmax_observer_default) {
    const MinMaxObserver obs = MinMaxObserver::default_();
    ASSERT_EQ(obs.min_val(), INFINITY);
    ASSERT_EQ(obs.max_val(), -INFINITY);
}

TEST_GPU(test_per_channel_compute_global_scale) {
    PerChannelMinMaxObserver obs(2);
    obs.observe({0.0, 1.0, 0.0, 2.0});
    auto [scale, zp] = obs.compute_scale_zero_point(QuantDType::Int8);
    ASSERT(scale > 0.0);
    (void)zp;
}

// ------------------------------------------------------------ linear.rs:145-174 (quantized)

TEST_GPU(test_quantized_linear_shape) {
    const Tensor w = Tensor::from_slice(randn(5 * 10, 0.5, 1), {5, 10});
    const Tensor b = Tensor::from_slice(randn(5, 0.1, 2), {5});
    const QuantizedLinear layer = QuantizedLinear::from_tensors(w, b).unwrap();
    ASSERT_EQ(layer.in_features(), 10u);
    ASSERT_EQ(layer.out_features(), 5u);
    ASSERT((layer.parameters()[0].shape() == std::vector<size_t>{5, 10}));
    ASSERT_EQ(layer.parameters().size(), 3u);  // codes, scales, bias
    ASSERT_EQ(layer.num_parameters(), 55u);
}

TEST_GPU(test_quantized_linear_forward_shape) {
    const Tensor w = Tensor::from_slice(randn(2 * 3, 0.5, 3), {2, 3});
    const QuantizedLinear layer = QuantizedLinear::from_tensors(w, std::nullopt).unwrap();
    const Tensor out = layer.forward(Tensor::ones({4, 3}));
    ASSERT((out.shape() == std::vector<size_t>{4, 2}));
    ASSERT((layer.forward(Tensor::ones({3})).shape() == std::vector<size_t>{2}));
}

TEST_GPU(test_quantized_linear_errors) {
    const Tensor w = Tensor::from_slice(randn(4 * 8, 0.5, 4), {4, 8});
    const QuantizedLinear layer = QuantizedLinear::from_tensors(w, std::nullopt).unwrap();
    auto r = layer.try_forward(Tensor::ones({2, 7}));
    ASSERT(r.is_err() && r.unwrap_err().kind() == TheanoError::Kind::ShapeMismatch);
    // INT4 g128 needs K % 128 == 0
    auto r4 = QuantizedLinear::from_tensors(Tensor::ones({4, 100}), std::nullopt, QConfig::default_int4());
    ASSERT(r4.is_err() && r4.unwrap_err().kind() == TheanoError::Kind::InvalidArgument);
    auto rb = QuantizedLinear::from_tensors(w, Tensor::ones({3}));
    ASSERT(rb.is_err() && rb.unwrap_err().kind() == TheanoError::Kind::ShapeMismatch);
}

// ------------------------------------------------------------ parity with the oracle

TEST_GPU(test_parity_primitives_f64) {
    // f64 inputs, including values no f32 holds, and exact ties
    std::vector<double> x = randn(4099, 3.0, 11);
    x[0] = 2.5;
    x[1] = -2.5;
    x[2] = 0.1 + 1e-12;
    x[3] = NAN;
    x[4] = -0.3;
    x[5] = 1e300;
    const Tensor t = Tensor::from_slice(x, {x.size()});
    for (QuantDType dt : {QuantDType::Int8, QuantDType::UInt8, QuantDType::Int4, QuantDType::FP8}) {
        const double s = 0.037, zp = dt == QuantDType::UInt8 ? 128.0 : 0.0;
        std::vector<double> ref(x.size());
        tqo_quantize_tensor(x.data(), static_cast<int64_t>(x.size()), s, zp, dt.abi(), ref.data());
        const auto q = quantize_tensor(t, s, zp, dt).unwrap();
        ASSERT(same_bits(q, ref));
        std::vector<double> dref(x.size());
        tqo_dequantize_tensor(ref.data(), static_cast<int64_t>(x.size()), s, zp, dref.data());
        ASSERT(same_bits(dequantize_tensor(q, s, zp), dref));
        std::vector<double> fref(x.size());
        tqo_fake_quantize(x.data(), static_cast<int64_t>(x.size()), s, zp, dt.abi(), fref.data());
        ASSERT(same_bits(fake_quantize(t, s, zp, dt).unwrap().to_vec_f64().unwrap(), fref));
    }
    std::vector<double> y = randn(1000, 2.0, 12);
    y[7] = NAN;
    const Tensor ty = Tensor::from_slice(y, {y.size()});
    for (QuantDType dt : {QuantDType::Int8, QuantDType::UInt8, QuantDType::Int4}) {
        std::vector<double> ref(y.size());
        double rs = 0, rz = 0;
        tqo_quantize_per_tensor(y.data(), static_cast<int64_t>(y.size()), dt.abi(), ref.data(), &rs, &rz);
        auto [q, s, z] = quantize_per_tensor(ty, dt).unwrap();
        ASSERT(same_bits(q, ref));
        ASSERT_EQ(s, rs);
        ASSERT_EQ(z, rz);
    }
}

TEST_GPU(test_parity_observers_f64) {
    const std::vector<double> a = randn(777, 1.5, 21), b = randn(333, 4.0, 22);
    MinMaxObserver obs;
    obs.observe(a);
    obs.observe(b);
    double st[3] = {INFINITY, -INFINITY, 0.0};
    tqo_minmax_observe(st, a.data(), static_cast<int64_t>(a.size()));
    tqo_minmax_observe(st, b.data(), static_cast<int64_t>(b.size()));
    ASSERT_EQ(obs.min_val(), st[0]);
    ASSERT_EQ(obs.max_val(), st[1]);
    for (QuantDType dt : {QuantDType::Int8, QuantDType::UInt8, QuantDType::Int4}) {
        double rs, rz;
        tqo_minmax_scale_zp(st, dt.abi(), &rs, &rz);
        auto [s, z] = obs.compute_scale_zero_point(dt);
        ASSERT_EQ(s, rs);
        ASSERT_EQ(z, rz);
    }
    const size_t ch = 7;
    PerChannelMinMaxObserver pc(ch);
    std::vector<double> mins(ch, INFINITY), maxs(ch, -INFINITY);
    pc.observe(a);  // 777 = 7 x 111, no remainder
    tqo_perchannel_observe(mins.data(), maxs.data(), ch, a.data(), static_cast<int64_t>(a.size()));
    pc.observe(b);  // 333 = 7 x 47 + 4: the remainder is ignored
    tqo_perchannel_observe(mins.data(), maxs.data(), ch, b.data(), static_cast<int64_t>(b.size()));
    std::vector<double> rs(ch), rz(ch);
    tqo_perchannel_scales_zps(mins.data(), maxs.data(), ch, TQ_QINT8, rs.data(), rz.data());
    const auto sz = pc.scales_and_zero_points(QuantDType::Int8);
    for (size_t c = 0; c < ch; ++c) {
        ASSERT_EQ(sz[c].first, rs[c]);
        ASSERT_EQ(sz[c].second, rz[c]);
    }
    double gs, gz;
    tqo_perchannel_global_scale_zp(mins.data(), maxs.data(), ch, TQ_QINT8, &gs, &gz);
    auto [s, z] = pc.compute_scale_zero_point(QuantDType::Int8);
    ASSERT_EQ(s, gs);
    ASSERT_EQ(z, gz);
}

// weights as the f32 values the device formats hold
std::vector<float> f32(const std::vector<double>& v) { return std::vector<float>(v.begin(), v.end()); }

TEST_GPU(test_parity_quantized_linear_w8) {
    const size_t n = 300, k = 512, m = 3;
    const auto wv = randn(n * k, 0.02, 31), xv = randn(m * k, 1.0, 32), bv = randn(n, 0.1, 33);
    const QuantizedLinear layer =
        QuantizedLinear::from_tensors(Tensor::from_slice(wv, {n, k}), Tensor::from_slice(bv, {n})).unwrap();
    ASSERT(layer.mode() == QuantizedLinear::Mode::W8);
    const auto y = layer.forward(Tensor::from_slice(xv, {m, k})).to_vec_f64().unwrap();
    const auto w32 = f32(wv), x32 = f32(xv), b32 = f32(bv);
    std::vector<int8_t> q(n * k);
    std::vector<float> s(n);
    tqo_quantize_i8_rowwise(w32.data(), n, k, q.data(), s.data());
    std::vector<double> ref(m * n);
    tqo_linear_w8(x32.data(), m, q.data(), s.data(), b32.data(), n, k, ref.data());
    assert_close(y, ref, "w8 linear");
}

TEST_GPU(test_quantized_linear_w8_needs_no_workspace_where_it_asks_for_none) {
    // sizes that the matrix cores run unsplit: no workspace asked for, none needed
    const size_t m = 100, n = 1000, k = 384;
    const auto wv = randn(n * k, 0.02, 34), xv = randn(m * k, 1.0, 35);
    const auto w32 = f32(wv), x32 = f32(xv);
    rocm::DeviceBuffer<float> x(m * k), y(m * n), y2(m * n), s(n);
    x.upload(x32.data(), m * k, nullptr);
    std::vector<float> got(m * n), want(m * n), sv(n);
    for (bool fp8 : {false, true}) {
        const QConfig cfg = fp8 ? QConfig{QuantDType::FP8, QuantDType::UInt8, true, true} : QConfig::default_int8();
        const QuantizedLinear layer =
            QuantizedLinear::from_tensors(Tensor::from_slice(wv, {n, k}), std::nullopt, cfg).unwrap();
        ASSERT(layer.workspace_bytes(m) == 0);
        ASSERT(layer.forward_device(x.data(), m, y.data(), nullptr).is_ok());
        rocm::DeviceBuffer<uint8_t> q(n * k);
        std::vector<uint8_t> qv(n * k);
        if (fp8)
            tqo_quantize_fp8_rowwise(w32.data(), n, k, qv.data(), sv.data());
        else
            tqo_quantize_i8_rowwise(w32.data(), n, k, reinterpret_cast<int8_t*>(qv.data()), sv.data());
        q.upload(qv.data(), n * k, nullptr);
        s.upload(sv.data(), n, nullptr);
        ASSERT((fp8 ? tq_gemm_fp8_weight(x.data(), m, q.data(), s.data(), nullptr, n, k, nullptr, 0, y2.data(), nullptr)
                    : tq_gemm_w8(x.data(), m, reinterpret_cast<int8_t*>(q.data()), s.data(), nullptr, n, k, nullptr, 0,
                                 y2.data(), nullptr)) == TQ_OK);
        y.download(got.data(), m * n, nullptr);
        y2.download(want.data(), m * n, nullptr);
        ASSERT(std::memcmp(got.data(), want.data(), m * n * sizeof(float)) == 0);
    }
}

TEST_GPU(test_parity_quantized_linear_w4) {
    const size_t n = 200, k = 1024;
    const auto wv = randn(n * k, 0.02, 41);
    const QuantizedLinear layer =
        QuantizedLinear::from_tensors(Tensor::from_slice(wv, {n, k}), std::nullopt, QConfig::default_int4()).unwrap();
    const auto w32 = f32(wv);
    std::vector<uint8_t> p(n * k / 2);
    std::vector<uint16_t> s(n * k / 128);
    tqo_quantize_i4_g128(w32.data(), n, k, p.data(), s.data());
    for (size_t m : {1u, 3u, 9u, 32u, 40u}) {  // tiled GEMV (1-16, 2 passes at 32), W4A16 GEMM (40)
        const auto xv = randn(m * k, 1.0, 42 + m);
        const auto y = layer.forward(Tensor::from_slice(xv, {m, k})).to_vec_f64().unwrap();
        std::vector<uint16_t> xb(m * k);
        for (size_t i = 0; i < xb.size(); ++i) xb[i] = tqo_f32_to_bf16_bits(static_cast<float>(xv[i]));
        std::vector<double> ref(m * n);
        tqo_linear_w4g128_bf16(xb.data(), m, p.data(), s.data(), nullptr, n, k, ref.data());
        assert_close(y, ref, "w4 linear");
    }
}

TEST_GPU(test_parity_quantized_linear_w4_prefill) {
    // N % 256 == 0 and K % 256 == 0, M > 32: the pipelined kernels (64-row tiles
    // with K split in two for the small grids at M = 64 and 100), with bias
    const size_t n = 512, k = 2048;
    const auto wv = randn(n * k, 0.02, 71), bv = randn(n, 0.1, 72);
    const QuantizedLinear layer = QuantizedLinear::from_tensors(Tensor::from_slice(wv, {n, k}),
                                                                Tensor::from_slice(bv, {n}), QConfig::default_int4())
                                      .unwrap();
    ASSERT(layer.workspace_bytes(100) > 0 && layer.workspace_bytes(64) > 0 && layer.workspace_bytes(32) == 0);
    const auto w32 = f32(wv), b32 = f32(bv);
    std::vector<uint8_t> p(n * k / 2);
    std::vector<uint16_t> s(n * k / 128);
    tqo_quantize_i4_g128(w32.data(), n, k, p.data(), s.data());
    for (size_t m : {64u, 100u, 300u}) {
        const auto xv = randn(m * k, 1.0, 73 + m);
        const auto y = layer.forward(Tensor::from_slice(xv, {m, k})).to_vec_f64().unwrap();
        std::vector<uint16_t> xb(m * k);
        for (size_t i = 0; i < xb.size(); ++i) xb[i] = tqo_f32_to_bf16_bits(static_cast<float>(xv[i]));
        std::vector<double> ref(m * n);
        tqo_linear_w4g128_bf16(xb.data(), m, p.data(), s.data(), b32.data(), n, k, ref.data());
        assert_close(y, ref, "w4 prefill linear");
    }
}

TEST_GPU(test_parity_quantized_linear_w8a8) {
    // m = 2: the fused GEMV; 5, 16: quantize + the skinny GEMM; 37: the tiled GEMM
    const size_t n = 272, k = 1024;
    const auto wv = randn(n * k, 0.02, 51);
    const QConfig cfg{QuantDType::Int8, QuantDType::Int8, true, true};
    const QuantizedLinear layer = QuantizedLinear::from_tensors(Tensor::from_slice(wv, {n, k}), std::nullopt, cfg).unwrap();
    ASSERT(layer.mode() == QuantizedLinear::Mode::W8A8);
    const auto w32 = f32(wv);
    std::vector<int8_t> qw(n * k);
    std::vector<float> sw(n);
    tqo_quantize_i8_rowwise(w32.data(), n, k, qw.data(), sw.data());
    for (size_t m : {2u, 5u, 16u, 37u}) {
        const auto xv = randn(m * k, 1.0, 52 + m);
        const auto y = layer.forward(Tensor::from_slice(xv, {m, k})).to_vec_f64().unwrap();
        const auto x32 = f32(xv);
        std::vector<int8_t> qa(m * k);
        std::vector<float> sa(m);
        tqo_quantize_i8_rowwise(x32.data(), m, k, qa.data(), sa.data());
        std::vector<double> ref(m * n);
        tqo_linear_w8a8(qa.data(), sa.data(), qw.data(), sw.data(), nullptr, m, n, k, ref.data());
        assert_close(y, ref, "w8a8 linear");
    }
}

TEST_GPU(test_parity_quantized_linear_fp8) {
    const size_t n = 272, k = 1024;
    const auto wv = randn(n * k, 0.02, 53), bv = randn(n, 0.1, 55);
    const QConfig cfg{QuantDType::FP8, QuantDType::FP8, true, true};
    const QuantizedLinear layer =
        QuantizedLinear::from_tensors(Tensor::from_slice(wv, {n, k}), Tensor::from_slice(bv, {n}), cfg).unwrap();
    ASSERT(layer.mode() == QuantizedLinear::Mode::FP8);
    const auto w32 = f32(wv), b32 = f32(bv);
    std::vector<uint8_t> qw(n * k);
    std::vector<float> sw(n);
    tqo_quantize_fp8_rowwise(w32.data(), n, k, qw.data(), sw.data());
    for (size_t m : {3u, 37u}) {  // decode GEMV and prefill GEMM
        const auto xv = randn(m * k, 1.0, 54 + m);
        const auto y = layer.forward(Tensor::from_slice(xv, {m, k})).to_vec_f64().unwrap();
        const auto x32 = f32(xv);
        std::vector<uint8_t> qa(m * k);
        std::vector<float> sa(m);
        tqo_quantize_fp8_rowwise(x32.data(), m, k, qa.data(), sa.data());
        std::vector<double> ref(m * n);
        tqo_linear_fp8(qa.data(), sa.data(), qw.data(), sw.data(), b32.data(), m, n, k, ref.data());
        assert_close(y, ref, "fp8 linear");
    }
    // weight-only: f32 activations against Linear over the dequantized weight
    const QuantizedLinear wo =
        QuantizedLinear::from_tensors(Tensor::from_slice(wv, {n, k}), std::nullopt,
                                      QConfig{QuantDType::FP8, QuantDType::UInt8, true, true})
            .unwrap();
    ASSERT(wo.mode() == QuantizedLinear::Mode::FP8Weight);
    const size_t m = 20;
    const auto xv = randn(m * k, 1.0, 56);
    const auto y = wo.forward(Tensor::from_slice(xv, {m, k})).to_vec_f64().unwrap();
    std::vector<float> wh(n * k);
    tqo_dequantize_fp8_rowwise(qw.data(), sw.data(), n, k, wh.data());
    std::vector<double> x64(m * k), w64(wh.begin(), wh.end()), ref(m * n);
    for (size_t i = 0; i < x64.size(); ++i) x64[i] = static_cast<float>(xv[i]);
    tqo_linear(x64.data(), m, w64.data(), nullptr, n, k, ref.data());
    assert_close(y, ref, "fp8 weight-only linear");
}

TEST_GPU(test_parity_quantized_mlp) {
    // M = 1, 2, 4, 5, 9, 16 run the decode kernels (M = 4: one K-split down launch;
    // M >= 5: one gate/up launch, D <= 4096), M = 17, 28 two passes of them, M = 29
    // and 33 the prefill FFN
    const size_t d = 256, f = 384;
    const auto gv = randn(f * d, 0.02, 61), uv = randn(f * d, 0.02, 62), dv = randn(d * f, 0.02, 63);
    const QuantizedMLP mlp = QuantizedMLP::from_tensors(Tensor::from_slice(gv, {f, d}), Tensor::from_slice(uv, {f, d}),
                                                        Tensor::from_slice(dv, {d, f}))
                                 .unwrap();
    std::vector<uint8_t> pg(f * d / 2), pu(f * d / 2), pd(d * f / 2);
    std::vector<uint16_t> sg(f * d / 128), su(f * d / 128), sd(d * f / 128);
    const auto g32 = f32(gv), u32 = f32(uv), d32 = f32(dv);
    tqo_quantize_i4_g128(g32.data(), f, d, pg.data(), sg.data());
    tqo_quantize_i4_g128(u32.data(), f, d, pu.data(), su.data());
    tqo_quantize_i4_g128(d32.data(), d, f, pd.data(), sd.data());
    for (size_t m : {1, 2, 4, 5, 9, 16, 17, 28, 29, 33}) {
        ASSERT(mlp.decode_path(static_cast<int64_t>(m)) == (m <= 28));
        const auto xv = randn(m * d, 1.0, 64 + m);
        const auto y = mlp.forward(Tensor::from_slice(xv, {m, d})).to_vec_f64().unwrap();
        std::vector<uint16_t> xb(m * d);
        for (size_t i = 0; i < xb.size(); ++i) xb[i] = tqo_f32_to_bf16_bits(static_cast<float>(xv[i]));
        std::vector<double> ref(m * d);
        tqo_mlp_w4g128(xb.data(), m, d, f, pg.data(), sg.data(), pu.data(), su.data(), pd.data(), sd.data(),
                       ref.data());
        assert_close(y, ref, m <= 28 ? "mlp decode" : "mlp prefill");
    }
}

TEST_GPU(test_parity_weight_formats) {
    const size_t n = 33, k = 384;
    auto wv = randn(n * k, 0.02, 71);
    wv[5] = 0.0;
    const Tensor w = Tensor::from_slice(wv, {n, k});
    const auto w32 = f32(wv);
    auto i8 = quantize_per_channel_i8(w).unwrap();
    std::vector<int8_t> q(n * k);
    std::vector<float> s(n);
    tqo_quantize_i8_rowwise(w32.data(), n, k, q.data(), s.data());
    ASSERT(i8.codes.to_host(nullptr) == q);
    ASSERT(i8.scales.to_host(nullptr) == s);
    auto i4 = quantize_i4_g128(w).unwrap();
    std::vector<uint8_t> p(n * k / 2);
    std::vector<uint16_t> s4(n * k / 128);
    tqo_quantize_i4_g128(w32.data(), n, k, p.data(), s4.data());
    ASSERT(i4.packed.to_host(nullptr) == p);
    ASSERT(i4.scales.to_host(nullptr) == s4);
    auto f8 = quantize_per_channel_fp8(w).unwrap();
    std::vector<uint8_t> q8(n * k);
    std::vector<float> s8(n);
    tqo_quantize_fp8_rowwise(w32.data(), n, k, q8.data(), s8.data());
    ASSERT(f8.codes.to_host(nullptr) == q8);
    ASSERT(f8.scales.to_host(nullptr) == s8);
    std::vector<float> wh8(n * k);
    tqo_dequantize_fp8_rowwise(q8.data(), s8.data(), n, k, wh8.data());
    const auto got8 = dequantize(f8).unwrap().to_vec_f64().unwrap();
    for (size_t i = 0; i < wh8.size(); ++i) ASSERT_EQ(got8[i], static_cast<double>(wh8[i]));
    std::vector<float> wh(n * k);
    tqo_dequantize_i4_g128(p.data(), s4.data(), n, k, wh.data());
    const auto got = dequantize(i4).unwrap().to_vec_f64().unwrap();
    for (size_t i = 0; i < wh.size(); ++i) ASSERT_EQ(got[i], static_cast<double>(wh[i]));
}

}  // namespace


// ------------------------------------------------- safetensors.rs:240-286

TEST_CPU(test_safetensors_roundtrip) {
    std::map<std::string, Tensor> tensors;
    tensors.emplace("weight", Tensor::from_slice({1.0, 2.0, 3.0, 4.0}, {2, 2}));
    tensors.emplace("bias", Tensor::from_slice({5.0, 6.0}, {2}));
    const auto bytes = ser::save_safetensors(tensors);
    const auto loaded = ser::load_safetensors(bytes).unwrap();
    ASSERT_EQ(loaded.size(), 2u);
    ASSERT(loaded.at("weight").shape() == (std::vector<size_t>{2, 2}));
    ASSERT(loaded.at("weight").to_vec_f64().unwrap() == (std::vector<double>{1.0, 2.0, 3.0, 4.0}));
    ASSERT(loaded.at("bias").to_vec_f64().unwrap() == (std::vector<double>{5.0, 6.0}));
}

TEST_CPU(test_safetensors_file_api) {
    ser::SafeTensorsFile file;
    file.add_tensor("x", Tensor::ones({3, 3}));
    ASSERT_EQ(file.tensor_names().size(), 1u);
    const Tensor t = file.get_tensor("x").unwrap();
    ASSERT(t.shape() == (std::vector<size_t>{3, 3}));
}

TEST_CPU(test_safetensors_empty) {
    const auto bytes = ser::save_safetensors({});
    ASSERT_EQ(ser::load_safetensors(bytes).unwrap().size(), 0u);
}

// The reference's own bytes: f64 payloads under DType names, header keys sorted,
// data in insertion order (safetensors.rs:36-54, 83-135).
TEST_CPU(test_safetensors_reference_dialect) {
    const std::vector<double> w = {1.0, 2.0, 3.0, 4.0}, b = {5.0, 6.0};
    std::vector<uint8_t> data(48);
    std::memcpy(data.data(), b.data(), 16);       // bias inserted first
    std::memcpy(data.data() + 16, w.data(), 32);
    const std::string h = "{\"bias\":{\"dtype\":\"float32\",\"shape\":[2],\"data_offsets\":[0,16]},"
                          "\"weight\":{\"dtype\":\"float64\",\"shape\":[2,2],\"data_offsets\":[16,48]}}";
    std::vector<uint8_t> bytes(8);
    const uint64_t n = h.size();
    std::memcpy(bytes.data(), &n, 8);
    bytes.insert(bytes.end(), h.begin(), h.end());
    bytes.insert(bytes.end(), data.begin(), data.end());
    const auto loaded = ser::load_safetensors(bytes).unwrap();
    ASSERT(loaded.at("weight").to_vec_f64().unwrap() == w);
    ASSERT(loaded.at("bias").to_vec_f64().unwrap() == b);
}

TEST_CPU(test_safetensors_raw_payloads) {
    ser::SafeTensorsFile f;
    const int8_t i8[4] = {-128, -1, 0, 127};
    const uint16_t f16[2] = {0x3800, 0xBC00};  // 0.5, -1.0
    ASSERT(f.add_raw("a", "I8", {2, 2}, i8, 4).is_ok());
    ASSERT(f.add_raw("b", "F16", {2}, f16, 4).is_ok());
    ASSERT(f.add_raw("c", "F32", {3}, i8, 4).is_err());      // size mismatch
    ASSERT(f.add_raw("d", "float32", {1}, i8, 4).is_err());  // not a standard code
    f.metadata["a.quant"] = "int8_per_channel";
    const auto bytes = f.to_bytes();
    uint64_t hl;
    std::memcpy(&hl, bytes.data(), 8);
    ASSERT_EQ(hl % 8, 0u);
    const auto g = ser::SafeTensorsFile::from_bytes(bytes).unwrap();
    ASSERT(g.metadata.at("a.quant") == "int8_per_channel");
    const auto raw = g.get_raw("a", "I8", {2, 2}).unwrap();
    ASSERT(std::memcmp(raw.data(), i8, 4) == 0);
    ASSERT(g.get_raw("a", "U8", {2, 2}).is_err());
    ASSERT(g.get_tensor("a").unwrap().to_vec_f64().unwrap() == (std::vector<double>{-128, -1, 0, 127}));
    ASSERT(g.get_tensor("b").unwrap().to_vec_f64().unwrap() == (std::vector<double>{0.5, -1.0}));
    // F8_E4M3 codes: 1.0, -448, smallest subnormal 2^-9, NaN
    ser::SafeTensorsFile h;
    const uint8_t f8[4] = {0x38, 0xFE, 0x01, 0x7F};
    ASSERT(h.add_raw("e", "F8_E4M3", {4}, f8, 4).is_ok());
    const auto hb = ser::SafeTensorsFile::from_bytes(h.to_bytes()).unwrap();
    ASSERT(hb.get_raw("e", "F8_E4M3", {4}).is_ok());
    const auto ev = hb.get_tensor("e").unwrap().to_vec_f64().unwrap();
    ASSERT(ev[0] == 1.0 && ev[1] == -448.0 && ev[2] == std::ldexp(1.0, -9) && std::isnan(ev[3]));
}

TEST_CPU(test_safetensors_malformed) {
    ASSERT(ser::SafeTensorsFile::from_bytes({1, 0}).is_err());
    std::vector<uint8_t> b(8);
    const uint64_t big = 100;
    std::memcpy(b.data(), &big, 8);
    ASSERT(ser::SafeTensorsFile::from_bytes(b).is_err());  // truncated header
    auto make = [](const std::string& h, size_t data) {
        std::vector<uint8_t> v(8);
        const uint64_t n = h.size();
        std::memcpy(v.data(), &n, 8);
        v.insert(v.end(), h.begin(), h.end());
        v.resize(v.size() + data);
        return v;
    };
    ASSERT(ser::SafeTensorsFile::from_bytes(make("[]", 0)).is_err());
    ASSERT(ser::SafeTensorsFile::from_bytes(make("{\"t\":{\"dtype\":\"F32\",\"shape\":[2],\"data_offsets\":[0,12]}}", 8))
               .is_err());  // offsets past the data
    ASSERT(ser::SafeTensorsFile::from_bytes(make("{\"t\":{\"dtype\":\"F32\",\"shape\":[3],\"data_offsets\":[0,8]}}", 8))
               .is_err());  // size != shape x element
    ASSERT(ser::SafeTensorsFile::from_bytes(make("{\"t\":{\"dtype\":\"X9\",\"shape\":[1],\"data_offsets\":[0,4]}}", 4))
               .is_err());  // unknown dtype
    ASSERT(ser::SafeTensorsFile::from_bytes(make("{\"t\":{\"dtype\":\"F32\",\"shape\":[1]", 4)).is_err());
}

// tests/golden/ beside the executable's directory, or $TQ_GOLDEN_DIR (a build elsewhere)
std::vector<uint8_t> golden_checkpoint() {
    std::string dir;
    if (const char* g = std::getenv("TQ_GOLDEN_DIR")) {
        dir = g;
    } else {
        char exe[4096];
        const ssize_t n = readlink("/proc/self/exe", exe, sizeof exe - 1);
        ASSERT(n > 0);
        dir = std::string(exe, static_cast<size_t>(n));
        dir = dir.substr(0, dir.rfind('/')) + "/../golden";
    }
    std::ifstream in(dir + "/checkpoint_int4_16x256.safetensors", std::ios::binary);
    ASSERT(in.good());
    return std::vector<uint8_t>((std::istreambuf_iterator<char>(in)), std::istreambuf_iterator<char>());
}

// written by the independent `safetensors` package (tests/golden/make_golden.py)
TEST_CPU(test_safetensors_independent_writer) {
    const auto f = ser::SafeTensorsFile::from_bytes(golden_checkpoint()).unwrap();
    ASSERT(f.get_tensor("const.f64").unwrap().to_vec_f64().unwrap() == (std::vector<double>{1.5, -2.0, 3.25}));
    ASSERT(f.get_tensor("const.i8").unwrap().to_vec_f64().unwrap() == (std::vector<double>{-128, 0, 127}));
    ASSERT(f.get_tensor("const.f16").unwrap().to_vec_f64().unwrap() == (std::vector<double>{0.5, -1.0, 65504.0}));
    const Tensor u8 = f.get_tensor("const.u8").unwrap();
    ASSERT(u8.shape() == (std::vector<size_t>{2, 2}));
    ASSERT(u8.to_vec_f64().unwrap() == (std::vector<double>{0, 255, 7, 128}));
    ASSERT(f.metadata.at("proj.quant") == "int4_g128");
    ASSERT(f.get_raw("proj.weight", "U8", {16, 128}).is_ok());
    ASSERT(f.get_raw("proj.weight_scale", "F16", {16, 2}).is_ok());
}

TEST_GPU(test_checkpoint_linear_and_mlp_roundtrip) {
    const size_t n = 256, k = 512;
    const auto wv = randn(n * k, 0.02, 91), bv = randn(n, 0.1, 92);
    const QConfig a8{QuantDType::Int8, QuantDType::Int8, true, true};
    const QConfig fp8{QuantDType::FP8, QuantDType::FP8, true, true};
    const QConfig fp8w{QuantDType::FP8, QuantDType::Int8, true, true};
    const std::vector<std::pair<std::string, QConfig>> cfgs = {{"l4", QConfig::default_int4()},
                                                              {"l8", QConfig::default_int8()},
                                                              {"l8a8", a8},
                                                              {"lfp8", fp8},
                                                              {"lfp8w", fp8w}};
    ser::SafeTensorsFile file;
    std::vector<QuantizedLinear> layers;
    for (const auto& [name, cfg] : cfgs) {
        layers.push_back(QuantizedLinear::from_tensors(Tensor::from_slice(wv, {n, k}),
                                                       name == "l8a8" ? std::optional<Tensor>{}
                                                                      : std::optional<Tensor>{Tensor::from_slice(bv, {n})},
                                                       cfg)
                             .unwrap());
        ASSERT(layers.back().save(file, name).is_ok());
    }
    const QuantizedMLP mlp = QuantizedMLP::from_tensors(Tensor::from_slice(randn(512 * 256, 0.02, 93), {512, 256}),
                                                        Tensor::from_slice(randn(512 * 256, 0.02, 94), {512, 256}),
                                                        Tensor::from_slice(randn(256 * 512, 0.02, 95), {256, 512}))
                                 .unwrap();
    ASSERT(mlp.save(file, "mlp").is_ok());
    const auto back = ser::SafeTensorsFile::from_bytes(file.to_bytes()).unwrap();
    for (size_t i = 0; i < cfgs.size(); ++i) {
        const QuantizedLinear l = QuantizedLinear::load(back, cfgs[i].first).unwrap();
        ASSERT(l.mode() == layers[i].mode() && l.in_features() == k && l.out_features() == n);
        for (size_t m : {1u, 5u, 40u}) {
            const Tensor x = Tensor::from_slice(randn(m * k, 1.0, 96 + m), {m, k});
            ASSERT(same_bits(l.forward(x).to_vec_f64().unwrap(), layers[i].forward(x).to_vec_f64().unwrap()));
        }
    }
    const QuantizedMLP m2 = QuantizedMLP::load(back, "mlp").unwrap();
    const Tensor x = Tensor::from_slice(randn(7 * 256, 1.0, 97), {7, 256});
    ASSERT(same_bits(m2.forward(x).to_vec_f64().unwrap(), mlp.forward(x).to_vec_f64().unwrap()));
    ASSERT(QuantizedLinear::load(back, "missing").is_err());
}

// the independent writer's checkpoint through QuantizedLinear::load vs the oracle
TEST_GPU(test_checkpoint_independent_writer_forward) {
    const auto f = ser::SafeTensorsFile::from_bytes(golden_checkpoint()).unwrap();
    const QuantizedLinear l = QuantizedLinear::load(f, "proj").unwrap();
    const size_t n = 16, k = 256, m = 3;
    const auto p = f.get_raw("proj.weight", "U8", {n, k / 2}).unwrap();
    const auto sraw = f.get_raw("proj.weight_scale", "F16", {n, k / 128}).unwrap();
    const auto braw = f.get_raw("proj.bias", "F32", {n}).unwrap();
    std::vector<uint16_t> s(n * k / 128);
    std::memcpy(s.data(), sraw.data(), sraw.size());
    std::vector<float> b(n);
    std::memcpy(b.data(), braw.data(), braw.size());
    const auto xv = randn(m * k, 1.0, 98);
    const auto y = l.forward(Tensor::from_slice(xv, {m, k})).to_vec_f64().unwrap();
    std::vector<uint16_t> xb(m * k);
    for (size_t i = 0; i < xb.size(); ++i) xb[i] = tqo_f32_to_bf16_bits(static_cast<float>(xv[i]));
    std::vector<double> ref(m * n);
    tqo_linear_w4g128_bf16(xb.data(), m, p.data(), s.data(), b.data(), n, k, ref.data());
    assert_close(y, ref, "checkpoint linear");
}

// ------------------------------------- allocator.rs:249-348 (host-memory backend)

struct HostMem {
    size_t limit = SIZE_MAX, used = 0;
    int mallocs = 0, frees = 0;
    std::map<void*, size_t> live;
};

rocm::MemoryBackend host_backend(std::shared_ptr<HostMem> h) {
    rocm::MemoryBackend b;
    b.malloc = [h](void** p, size_t n) {
        if (h->used + n > h->limit) return false;
        *p = std::malloc(n);
        h->used += n;
        h->live[*p] = n;
        ++h->mallocs;
        return true;
    };
    b.free = [h](void* p) {
        h->used -= h->live.at(p);
        h->live.erase(p);
        std::free(p);
        ++h->frees;
    };
    b.synchronize = []() {};
    return b;
}

TEST_CPU(test_allocator_basic) {
    auto h = std::make_shared<HostMem>();
    rocm::CachingAllocator alloc(0, host_backend(h));
    const rocm::Block b1 = alloc.allocate(1024).unwrap();
    ASSERT(b1.ptr != nullptr && b1.size >= 1024);
    auto st = alloc.stats();
    ASSERT_EQ(st.num_cache_misses, 1u);
    ASSERT(st.allocated_bytes > 0);
    alloc.free(b1);
    st = alloc.stats();
    ASSERT_EQ(st.allocated_bytes, 0u);
    ASSERT(st.cached_bytes > 0);
}

TEST_CPU(test_allocator_cache_reuse) {
    auto h = std::make_shared<HostMem>();
    rocm::CachingAllocator alloc(0, host_backend(h));
    const rocm::Block b1 = alloc.allocate(1024).unwrap();
    const size_t size1 = b1.size;
    alloc.free(b1);
    const rocm::Block b2 = alloc.allocate(1024).unwrap();
    ASSERT_EQ(b2.size, size1);
    ASSERT(b2.ptr == b1.ptr);
    const auto st = alloc.stats();
    ASSERT_EQ(st.num_cache_hits, 1u);
    ASSERT_EQ(st.num_mallocs, 1u);  // only one real malloc
    alloc.free(b2);
}

TEST_CPU(test_allocator_empty_cache) {
    auto h = std::make_shared<HostMem>();
    rocm::CachingAllocator alloc(0, host_backend(h));
    const rocm::Block b1 = alloc.allocate(1024).unwrap(), b2 = alloc.allocate(2048).unwrap();
    alloc.free(b1);
    alloc.free(b2);
    ASSERT(alloc.stats().cached_bytes > 0);
    alloc.empty_cache();
    ASSERT_EQ(alloc.stats().cached_bytes, 0u);
    ASSERT_EQ(alloc.stats().num_frees, 2u);
    ASSERT(h->live.empty() && h->frees == 2);  // the driver got both segments back
}

TEST_CPU(test_allocator_large_pool) {
    auto h = std::make_shared<HostMem>();
    rocm::CachingAllocator alloc(0, host_backend(h));
    const rocm::Block b = alloc.allocate(2 * 1024 * 1024).unwrap();
    ASSERT(b.size >= 2u * 1024 * 1024);
    alloc.free(b);
    ASSERT(alloc.stats().cached_bytes > 0);
    ASSERT_EQ(rocm::CachingAllocator::round_size(2 * 1024 * 1024 + 1), 4u * 1024 * 1024);
    ASSERT_EQ(rocm::CachingAllocator::round_size(1000), 1024u);
}

TEST_CPU(test_allocator_zero_size) {
    auto h = std::make_shared<HostMem>();
    rocm::CachingAllocator alloc(0, host_backend(h));
    const rocm::Block b = alloc.allocate(0).unwrap();
    ASSERT_EQ(b.size, 0u);
    ASSERT(b.ptr == nullptr);
    alloc.free(b);
    ASSERT_EQ(h->mallocs, 0);
}

TEST_CPU(test_allocator_stats) {
    auto h = std::make_shared<HostMem>();
    rocm::CachingAllocator alloc(0, host_backend(h));
    const rocm::Block b1 = alloc.allocate(512).unwrap(), b2 = alloc.allocate(1024).unwrap();
    const auto st = alloc.stats();
    ASSERT_EQ(st.num_mallocs, 2u);
    ASSERT(st.peak_allocated_bytes >= 512 + 1024);
    alloc.free(b1);
    alloc.free(b2);
}

TEST_CPU(test_allocator_device_ordinal) {
    auto h = std::make_shared<HostMem>();
    rocm::CachingAllocator alloc(3, host_backend(h));
    ASSERT_EQ(alloc.device(), 3);
}

TEST_CPU(test_allocator_split_merge_streams) {
    auto h = std::make_shared<HostMem>();
    rocm::CachingAllocator alloc(0, host_backend(h));
    const size_t MB = 1u << 20;
    const rocm::Block big = alloc.allocate(2 * MB + 1).unwrap();  // one 4 MB segment
    ASSERT_EQ(big.size, 4 * MB);
    alloc.free(big);
    const rocm::Block a = alloc.allocate(MB + 1).unwrap();  // 2 MB from the 4 MB piece; 2 MB stays cached
    const rocm::Block b = alloc.allocate(2 * MB).unwrap();  // the remainder
    ASSERT_EQ(h->mallocs, 1);
    ASSERT(static_cast<char*>(b.ptr) == static_cast<char*>(a.ptr) + 2 * MB);
    auto st = alloc.stats();
    ASSERT_EQ(st.allocated_bytes, 4 * MB);
    ASSERT_EQ(st.cached_bytes, 0u);
    alloc.free(a);
    alloc.free(b);  // merges back into one free 4 MB piece
    st = alloc.stats();
    ASSERT_EQ(st.allocated_bytes, 0u);
    ASSERT_EQ(st.cached_bytes, 4 * MB);
    alloc.empty_cache();
    ASSERT_EQ(h->frees, 1);
    ASSERT(h->live.empty());
    // stream order: a block freed on one stream is not handed to another
    hipStream_t s1 = reinterpret_cast<hipStream_t>(0x10), s2 = reinterpret_cast<hipStream_t>(0x20);
    const rocm::Block c = alloc.allocate(4096, s1).unwrap();
    alloc.free(c);
    const rocm::Block d = alloc.allocate(4096, s2).unwrap();
    ASSERT(d.ptr != c.ptr);
    const rocm::Block e = alloc.allocate(4096, s1).unwrap();
    ASSERT(e.ptr == c.ptr);
    alloc.free(d);
    alloc.free(e);
}

TEST_CPU(test_allocator_oom_recovery) {
    auto h = std::make_shared<HostMem>();
    const size_t MB = 1u << 20;
    h->limit = 5 * MB;
    rocm::CachingAllocator alloc(0, host_backend(h));
    const rocm::Block a = alloc.allocate(4 * MB, reinterpret_cast<hipStream_t>(0x10)).unwrap();
    alloc.free(a);  // cached, not usable by the other stream
    const rocm::Block b = alloc.allocate(4 * MB, reinterpret_cast<hipStream_t>(0x20)).unwrap();  // frees the cache, retries
    ASSERT_EQ(h->frees, 1);
    auto r = alloc.allocate(4 * MB, reinterpret_cast<hipStream_t>(0x20));
    ASSERT(r.is_err() && r.unwrap_err().kind() == TheanoError::Kind::OutOfMemory);
    alloc.free(b);
}

// ------------------------------------------- device.rs / storage.rs on the GPU

TEST_GPU(test_rocm_device_properties) {
    auto dev = rocm::DeviceManager::global().get_device(0).unwrap();
    ASSERT(dev == rocm::DeviceManager::global().get_device(0).unwrap());  // one handle per ordinal
    const auto& p = dev->properties();
    ASSERT_EQ(p.gcn_arch, 950u);
    ASSERT_EQ(p.warp_size, 64u);
    ASSERT(p.multiprocessor_count >= 256u);
    ASSERT(p.total_memory > (200ull << 30));
    std::printf("[%s gfx%u, %u CUs, %zu GiB, %u threads/block, %zu B LDS/block] ", p.name.c_str(), p.gcn_arch,
                p.multiprocessor_count, p.total_memory >> 30, p.max_threads_per_block, p.max_shared_memory_per_block);
    ASSERT(p.max_threads_per_block >= 1024u);
    ASSERT(p.max_shared_memory_per_block >= 32u * 1024);
    const auto mi = dev->memory_info().unwrap();
    ASSERT(mi.second > 0 && mi.first <= mi.second);
    ASSERT(rocm::DeviceManager::global().get_device(99).is_err());
    ASSERT(rocm::DeviceManager::global().device_count() >= 1);
    ASSERT(dev->synchronize().is_ok());
}

TEST_GPU(test_rocm_storage_roundtrip_dtypes) {
    auto dev = rocm::DeviceManager::global().get_device(0).unwrap();
    std::vector<double> v = randn(100000, 1e3, 101);
    const double special[] = {0.0, -0.0, INFINITY, -INFINITY, NAN, 65520.0, 3.4e38, 1e-40, 127.5, -128.5,
                              300.0, -3e9, 9.3e18, 2.5, -2.5, 1e-8};
    for (double x : special) v.push_back(x);
    for (int t = 0; t < 10; ++t) {
        const DType dt = static_cast<DType>(t);
        const auto s = rocm::RocmStorage::from_host_f64(dev, v.data(), v.size(), dt).unwrap();
        ASSERT_EQ(s.byte_size(), v.size() * dtype_size(dt));
        const auto back = s.to_host_f64().unwrap();
        // oracle: the conversion, then its source decode back to f64
        std::vector<uint8_t> conv(v.size() * dtype_size(dt));
        tqo_convert(v.data(), 3, conv.data(), t, static_cast<int64_t>(v.size()));
        std::vector<double> ref(v.size());
        tqo_convert(conv.data(), t, ref.data(), 3, static_cast<int64_t>(v.size()));
        ASSERT(same_bits(back, ref));
    }
    // more than two staging chunks (f64 and f32 payloads)
    std::vector<double> big = randn(10u << 20, 1.0, 102);
    const auto s64 = rocm::RocmStorage::from_host_f64(dev, big.data(), big.size(), DType::F64).unwrap();
    ASSERT(same_bits(s64.to_host_f64().unwrap(), big));
    const auto s32 = s64.to_dtype(DType::F32).unwrap();
    const auto b32 = s32.to_host_f64().unwrap();
    for (size_t i = 0; i < big.size(); i += 997) ASSERT_EQ(b32[i], static_cast<double>(static_cast<float>(big[i])));
}

TEST_GPU(test_rocm_storage_returns_blocks_to_the_pool) {
    auto dev = rocm::DeviceManager::global().get_device(0).unwrap();
    { auto warm = rocm::RocmStorage::allocate(dev, 12345, DType::F32).unwrap(); }
    const auto before = dev->allocator().stats();
    for (int i = 0; i < 5; ++i) {
        auto s = rocm::RocmStorage::allocate(dev, 12345, DType::F32).unwrap();
        ASSERT(s.device_ptr() != nullptr);
    }
    const auto after = dev->allocator().stats();
    ASSERT_EQ(after.num_mallocs, before.num_mallocs);
    ASSERT_EQ(after.num_cache_hits, before.num_cache_hits + 5);
    ASSERT_EQ(after.allocated_bytes, before.allocated_bytes);
}

// Tensor::to(Device) round trip and quantized modules chained on the device give
// the host path's results bit for bit, without driver allocations once warm.
TEST_GPU(test_device_tensor_chain_matches_host_path) {
    auto dev = rocm::DeviceManager::global().get_device(0).unwrap();
    const size_t m = 24, d = 256, f = 384;
    const QConfig a8{QuantDType::Int8, QuantDType::Int8, true, true};
    const QConfig fp8{QuantDType::FP8, QuantDType::FP8, true, true};
    const QuantizedLinear l1 =
        QuantizedLinear::from_tensors(Tensor::from_slice(randn(f * d, 0.05, 111), {f, d}), std::nullopt, a8).unwrap();
    const QuantizedLinear l2 = QuantizedLinear::from_tensors(Tensor::from_slice(randn(d * f, 0.05, 112), {d, f}),
                                                             Tensor::from_slice(randn(d, 0.1, 113), {d}),
                                                             QConfig::default_int4())
                                   .unwrap();
    const QuantizedLinear l3 =
        QuantizedLinear::from_tensors(Tensor::from_slice(randn(d * d, 0.05, 114), {d, d}), std::nullopt, fp8).unwrap();
    const QuantizedMLP mlp = QuantizedMLP::from_tensors(Tensor::from_slice(randn(f * d, 0.02, 115), {f, d}),
                                                        Tensor::from_slice(randn(f * d, 0.02, 116), {f, d}),
                                                        Tensor::from_slice(randn(d * f, 0.02, 117), {d, f}))
                                 .unwrap();
    const Tensor x = Tensor::from_slice(randn(m * d, 1.0, 118), {m, d});
    const Tensor ref = mlp.forward(l3.forward(l2.forward(l1.forward(x))));
    const DeviceTensor xd = DeviceTensor::from_host(x, dev, DType::F32).unwrap();
    ASSERT(same_bits(xd.to_host().unwrap().to_vec_f64().unwrap(),
                     [&] {
                         std::vector<double> v = x.to_vec_f64().unwrap();
                         for (auto& e : v) e = static_cast<float>(e);
                         return v;
                     }()));
    auto run = [&]() {
        const DeviceTensor h1 = nn::forward(l1, xd).unwrap();
        const DeviceTensor h2 = nn::forward(l2, h1).unwrap();  // F32 -> BF16 on the device
        const DeviceTensor h3 = nn::forward(l3, h2).unwrap();
        return nn::forward(mlp, h3).unwrap();
    };
    const DeviceTensor y = run();
    ASSERT(y.shape() == (std::vector<size_t>{m, d}) && y.dtype() == DType::F32);
    ASSERT(same_bits(y.to_host().unwrap().to_vec_f64().unwrap(), ref.to_vec_f64().unwrap()));
    const auto warm = dev->allocator().stats();
    for (int i = 0; i < 3; ++i) (void)run();
    ASSERT_EQ(dev->allocator().stats().num_mallocs, warm.num_mallocs);  // served from the pool
    ASSERT(dev->synchronize().is_ok());
}

// ------------------------------------------------------------ multi-head attention (transformer.rs)

namespace {

struct MhaWeights {
    std::vector<std::vector<double>> w, b;  // q, k, v, out: [E, E] and [E]
};

MhaWeights mha_weights(size_t e, uint64_t seed) {
    MhaWeights r;
    for (uint64_t i = 0; i < 4; ++i) {
        r.w.push_back(randn(e * e, 0.05, seed + i));
        r.b.push_back(randn(e, 0.1, seed + 10 + i));
    }
    return r;
}

QuantizedMultiheadAttention make_mha(const MhaWeights& p, size_t e, size_t h, const QConfig& cfg) {
    auto t = [&](size_t i) { return Tensor::from_slice(p.w[i], {e, e}); };
    auto b = [&](size_t i) { return std::optional<Tensor>(Tensor::from_slice(p.b[i], {e})); };
    return QuantizedMultiheadAttention::from_tensors(h, t(0), t(1), t(2), t(3), b(0), b(1), b(2), b(3), cfg).unwrap();
}

std::vector<double> causal_mask(size_t s) {
    std::vector<double> m(s * s, 0.0);
    for (size_t i = 0; i < s; ++i)
        for (size_t j = i + 1; j < s; ++j) m[i * s + j] = -INFINITY;
    return m;
}

}  // namespace

TEST_CPU(test_mha_construction_errors) {
    // embed_dim % num_heads != 0 and non-square weights fail before any device work
    const Tensor w10 = Tensor::ones({10, 10});
    auto r = QuantizedMultiheadAttention::from_tensors(3, w10, w10, w10, w10);
    ASSERT(r.is_err() && r.unwrap_err().kind() == TheanoError::Kind::InvalidArgument);
    const Tensor w = Tensor::ones({8, 4});
    auto r2 = QuantizedMultiheadAttention::from_tensors(2, w, w, w, w);
    ASSERT(r2.is_err() && r2.unwrap_err().kind() == TheanoError::Kind::ShapeMismatch);
    auto r3 = QuantizedMultiheadAttention::from_tensors(0, w10, w10, w10, w10);
    ASSERT(r3.is_err() && r3.unwrap_err().kind() == TheanoError::Kind::InvalidArgument);
}

TEST_GPU(test_mha_reference_shapes_and_names) {
    // transformer.rs:188-268: output shape, parameter names and counts, masked forward
    const QuantizedMultiheadAttention mha = make_mha(mha_weights(64, 200), 64, 8, QConfig::default_int8());
    ASSERT(mha.embed_dim() == 64 && mha.num_heads() == 8 && mha.head_dim() == 8);
    ASSERT(mha.forward(Tensor::ones({2, 10, 64})).shape() == (std::vector<size_t>{2, 10, 64}));
    const auto named = mha.named_parameters();
    ASSERT_EQ(named.size(), size_t{12});
    ASSERT(named[0].first == "q_proj.weight" && named[1].first == "q_proj.weight_scale" && named[2].first == "q_proj.bias");
    ASSERT(named[3].first == "k_proj.weight" && named[6].first == "v_proj.weight" && named[11].first == "out_proj.bias");
    ASSERT(named[0].second.shape() == (std::vector<size_t>{64, 64}) && named[2].second.shape() == (std::vector<size_t>{64}));
    ASSERT_EQ(mha.parameters().size(), size_t{12});
    const QuantizedMultiheadAttention m16 = make_mha(mha_weights(16, 210), 16, 4, QConfig::default_int8());
    const Tensor x = Tensor::ones({1, 4, 16});
    const Tensor mask = Tensor::from_slice(causal_mask(4), {1, 4, 4});
    ASSERT(m16.forward_with_mask(x, x, x, mask).unwrap().shape() == (std::vector<size_t>{1, 4, 16}));
    ASSERT(m16.forward_qkv(x, x, x).shape() == (std::vector<size_t>{1, 4, 16}));
    ASSERT_EQ(m16.num_parameters(), size_t{4 * (16 * 16 + 16)});
    auto bad = m16.forward_with_mask(x, x, x, Tensor::ones({1, 3, 4}));
    ASSERT(bad.is_err() && bad.unwrap_err().kind() == TheanoError::Kind::ShapeMismatch);
    auto bad2 = m16.forward_with_mask(Tensor::ones({1, 4, 8}), Tensor::ones({1, 4, 8}), Tensor::ones({1, 4, 8}),
                                      std::nullopt);
    ASSERT(bad2.is_err() && bad2.unwrap_err().kind() == TheanoError::Kind::ShapeMismatch);
}

TEST_GPU(test_parity_mha_w8) {
    // INT8 weight-only projections + attention against the oracle chain in f64
    const size_t b = 2, s = 40, e = 256, h = 4, m = b * s;
    const MhaWeights p = mha_weights(e, 220);
    const QuantizedMultiheadAttention mha = make_mha(p, e, h, QConfig::default_int8());
    const auto xv = randn(m * e, 1.0, 230), kv = randn(m * e, 1.0, 231), vv = randn(m * e, 1.0, 232);
    const auto mask = causal_mask(s);
    auto proj = [&](size_t i, const std::vector<double>& x) {
        const auto w32 = f32(p.w[i]), b32 = f32(p.b[i]), x32 = f32(x);
        std::vector<int8_t> q(e * e);
        std::vector<float> sc(e);
        tqo_quantize_i8_rowwise(w32.data(), e, e, q.data(), sc.data());
        std::vector<double> y(x.size() / e * e);
        tqo_linear_w8(x32.data(), static_cast<int64_t>(x.size() / e), q.data(), sc.data(), b32.data(), e, e, y.data());
        return y;
    };
    auto chain = [&](const std::vector<double>& xq, const std::vector<double>& xk, const std::vector<double>& xw,
                     const double* mk) {
        const auto q = proj(0, xq), k = proj(1, xk), v = proj(2, xw);
        std::vector<double> att(m * e);
        tqo_attention(q.data(), k.data(), v.data(), mk, mk ? 1 : 0, b, s, h, e / h, att.data());
        return proj(3, att);
    };
    const Tensor x = Tensor::from_slice(xv, {b, s, e});
    assert_close(mha.forward_with_mask(x, x, x, Tensor::from_slice(mask, {1, s, s})).unwrap().to_vec_f64().unwrap(),
                 chain(xv, xv, xv, mask.data()), "mha w8 self, causal");
    assert_close(mha.forward(x).to_vec_f64().unwrap(), chain(xv, xv, xv, nullptr), "mha w8 self");
    assert_close(mha.forward_qkv(x, Tensor::from_slice(kv, {b, s, e}), Tensor::from_slice(vv, {b, s, e}))
                     .to_vec_f64()
                     .unwrap(),
                 chain(xv, kv, vv, nullptr), "mha w8 cross");
}

TEST_GPU(test_mha_device_tensor_matches_host_path) {
    // the device-resident forward gives the host API's bits, for each activation format
    auto dev = rocm::DeviceManager::global().get_device(0).unwrap();
    const size_t b = 2, s = 33, e = 256, h = 8;
    const MhaWeights p = mha_weights(e, 240);
    const QConfig a8{QuantDType::Int8, QuantDType::Int8, true, true};
    const QConfig fp8{QuantDType::FP8, QuantDType::FP8, true, true};
    const Tensor x = Tensor::from_slice(randn(b * s * e, 1.0, 250), {b, s, e});
    const Tensor xk = Tensor::from_slice(randn(b * s * e, 1.0, 251), {b, s, e});
    const Tensor mask = Tensor::from_slice(causal_mask(s), {1, 1, s, s});
    const DeviceTensor xd = DeviceTensor::from_host(x, dev, DType::F32).unwrap();
    const DeviceTensor xkd = DeviceTensor::from_host(xk, dev, DType::F32).unwrap();
    const DeviceTensor md = DeviceTensor::from_host(mask, dev, DType::F32).unwrap();
    for (const QConfig& cfg : {QConfig::default_int8(), QConfig::default_int4(), a8, fp8}) {
        const QuantizedMultiheadAttention mha = make_mha(p, e, h, cfg);
        const Tensor ref = mha.forward_with_mask(x, x, x, mask).unwrap();
        const DeviceTensor y = nn::forward_with_mask(mha, xd, xd, xd, md).unwrap();
        ASSERT(y.shape() == (std::vector<size_t>{b, s, e}) && y.dtype() == DType::F32);
        ASSERT(same_bits(y.to_host().unwrap().to_vec_f64().unwrap(), ref.to_vec_f64().unwrap()));
        const Tensor ref2 = mha.forward_qkv(x, xk, xk);
        ASSERT(same_bits(nn::forward_with_mask(mha, xd, xkd, xkd, std::nullopt).unwrap().to_host().unwrap().to_vec_f64().unwrap(),
                         ref2.to_vec_f64().unwrap()));
        ASSERT(same_bits(nn::forward(mha, xd).unwrap().to_host().unwrap().to_vec_f64().unwrap(),
                         mha.forward(x).to_vec_f64().unwrap()));
    }
    ASSERT(dev->synchronize().is_ok());
}

int main(int argc, char** argv) {
    const bool cpu_only = argc > 1 && std::strcmp(argv[1], "--cpu") == 0;
    int failed = 0, run = 0;
    for (const Case& c : registry()) {
        if (cpu_only && c.gpu) continue;
        ++run;
        std::printf("%-45s ", c.name);
        std::fflush(stdout);
        try {
            c.fn();
            std::printf("ok\n");
        } catch (const std::exception& e) {
            ++failed;
            std::printf("FAILED: %s\n", e.what());
        }
        std::fflush(stdout);
    }
    std::printf("%d of %d tests passed\n", run - failed, run);
    return failed ? 1 : 0;
}
