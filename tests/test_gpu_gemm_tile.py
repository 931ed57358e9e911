"""The register-staged tile GEMM behind the 8-bit Linears (tq_gemm_tile.h): odd and
tile-edge sizes, codes at odd addresses, K split over blocks, against the same
product in float64 (exact for INT8 codes: every partial sum is an integer below
2^53)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (m, n, k): below, at and past the 32/64/128 tile edges; K below one 64- or 128-byte
# stage, at and past stage edges, odd; few tiles of long K (split over blocks)
SHAPES = [(1, 1, 1), (3, 5, 17), (17, 64, 63), (31, 33, 64), (33, 65, 129), (64, 128, 255), (65, 129, 1000),
          (77, 1003, 1000), (128, 131, 128), (200, 257, 384), (40, 70, 8193), (16, 100, 14336), (129, 48, 4099)]


def _codes(torch, shape, seed, fp8):
    g = torch.Generator(device="cuda").manual_seed(seed)
    if fp8:
        x = (torch.randn(shape, generator=g, device="cuda") * 60).clamp(-448, 448)
        return x.to(torch.float8_e4m3fn)
    return torch.randint(-128, 128, shape, generator=g, device="cuda", dtype=torch.int8)


def _at_offset(torch, t, off):
    """`t`'s bytes at an address `off` past a 16-byte boundary."""
    b = t.view(torch.uint8).reshape(-1)
    buf = torch.empty(b.numel() + 64, dtype=torch.uint8, device="cuda")
    v = buf[off:off + b.numel()]
    v.copy_(b)
    return buf, v


def _run(torch, fp8, qa, qw, m, n, k, bias, off, with_ws):
    from theano_quantize import _abi
    from theano_quantize._tensor import ptr, stream

    g = torch.Generator(device="cuda").manual_seed(m * 31 + n)
    sa = torch.rand(m, generator=g, device="cuda") + 0.5
    sw = torch.rand(n, generator=g, device="cuda") + 0.5
    b = torch.randn(n, generator=g, device="cuda") if bias else None
    ka, va = _at_offset(torch, qa, off)
    kw, vw = _at_offset(torch, qw, off)
    y = torch.full((m, n), float("nan"), device="cuda")
    acc = torch.full((m, n), -7, dtype=torch.int32, device="cuda")
    name = "tq_gemm_fp8" if fp8 else "tq_gemm_w8a8"
    nb = int(getattr(_abi.lib(), name + "_workspace_bytes")(m, n, k))
    ws = torch.empty(max(nb, 8), dtype=torch.uint8, device="cuda").fill_(0xA5)
    args = [ptr(va), ptr(sa), ptr(vw), ptr(sw), ptr(b), m, n, k] + ([] if fp8 else [ptr(acc)])
    if with_ws:
        _abi.call(name + "_ws", *args, ptr(ws), nb, ptr(y), stream())
    else:
        _abi.call(name, *args, ptr(y), stream())
    torch.cuda.synchronize()
    prod = qa.double() @ qw.double().t().contiguous()
    ref = prod * sa.double()[:, None] * sw.double()
    if b is not None:
        ref = ref + b.double()
    return y.double(), acc, prod, ref


# with a workspace, each tile form unsplit and with K split (the estimates' choices on 256
# CUs: 128 x 128, 32 x 128, 64 x 128, 64 x 64), for INT8 and for codes widened to bf16
I8_FORMS = [(1980, 1553, 257), (69, 6035, 10460), (67, 8784, 34), (9, 4100, 1937), (297, 10913, 699), (38, 9416, 11275),
            (9, 37, 453), (10, 33, 1828)]
F8B_FORMS = [(1579, 1958, 1083), (99, 8692, 5231), (75, 8718, 32), (9, 1428, 3068), (521, 9749, 33), (258, 4029, 8036),
             (12, 1381, 33), (9, 35, 1256)]


@pytest.mark.parametrize("m,n,k,with_ws", [(*s, ws) for s in SHAPES for ws in (False, True)] +
                         [(*s, True) for s in I8_FORMS])
def test_w8a8_any_shape_exact(tq, m, n, k, with_ws):
    import torch

    for off in (0, 3):
        y, acc, prod, ref = _run(torch, False, _codes(torch, (m, k), 1, False), _codes(torch, (n, k), 2, False), m, n, k,
                                 off == 0, off, with_ws)
        assert torch.equal(acc.double(), prod)
        # f32 of the sum, the product with sa and the fma: three roundings of 2^-24 each
        bound = 4 * 2.0 ** -24 * (ref.abs() + 1.0)
        assert bool(((y - ref).abs() <= bound).all())


@pytest.mark.parametrize("m,n,k,with_ws", [(*s, ws) for s in SHAPES for ws in (False, True)] +
                         [(*s, True) for s in F8B_FORMS])
def test_fp8_any_shape(tq, m, n, k, with_ws):
    import torch

    qa, qw = _codes(torch, (m, k), 3, True), _codes(torch, (n, k), 4, True)
    y, _, _, ref = _run(torch, True, qa, qw, m, n, k, True, 5, with_ws)
    # exact bf16 products; every f32 addition of a run of 256 rounds by at most 2^-23 (twice
    # half an ulp, for an adder that truncates) of the largest partial sum, bounded by the
    # sum of magnitudes; measured errors are a hundred times smaller
    mag = (qa.double().abs() @ qw.double().abs().t().contiguous()) * 1.5 * 1.5
    bound = 2.0 ** -23 * min(k, 256) ** 0.5 * mag + 4 * 2.0 ** -24 * (ref.abs() + 4.0)
    assert bool(((y - ref).abs() <= bound).all())
    rel = ((y - ref).norm() / ref.norm()).item()
    assert rel < 1e-6, rel  # the fp8 matrix instructions' own sums would be 1.5e-5 off


@pytest.mark.parametrize("m,n,k", [(1, 1000, 1000), (1, 5000, 777), (64, 64, 64), (200, 64, 64), (3, 17, 100)])
@pytest.mark.parametrize("with_ws", [False, True])
def test_a8_smallest_calls(tq, m, n, k, with_ws):
    """The smallest products, a wave per output: exact sums for INT8, FP8 summed in f64."""
    import torch

    y, acc, prod, _ = _run(torch, False, _codes(torch, (m, k), 17, False), _codes(torch, (n, k), 18, False), m, n, k,
                           True, 1, with_ws)
    assert torch.equal(acc.double(), prod)
    y, _, _, ref = _run(torch, True, _codes(torch, (m, k), 19, True), _codes(torch, (n, k), 20, True), m, n, k, False, 1,
                        with_ws)
    # the sum to f32 and the products with the two scales: three roundings
    assert bool(((y - ref).abs() <= 3.01 * 2.0 ** -24 * ref.abs()).all())


@pytest.mark.parametrize("m,n,k", [(700, 4096, 256), (700, 4096, 384), (256, 16384, 128), (1024, 1008, 256),
                                   (130, 2064, 512), (512, 528, 2048), (265, 9808, 128), (306, 10528, 2560),
                                   (67, 8528, 256), (10, 1392, 9344), (642, 10880, 128), (33, 8256, 6016), (17, 32, 896),
                                   (21, 32, 1792), (64, 4096, 14336)])
@pytest.mark.parametrize("with_ws", [False, True])
def test_a8_aligned_shapes(tq, m, n, k, with_ws):
    """Sizes that the LDS-DMA kernels and the tiles share (K % 128, N % 16, 16-byte aligned),
    among them every tile form of the fp8 matrix instructions, unsplit and with K split."""
    import torch

    y, acc, prod, ref = _run(torch, False, _codes(torch, (m, k), 17, False), _codes(torch, (n, k), 18, False), m, n, k,
                             True, 0, with_ws)
    assert torch.equal(acc.double(), prod)
    assert bool(((y - ref).abs() <= 4 * 2.0 ** -24 * (ref.abs() + 1.0)).all())
    y, _, _, ref = _run(torch, True, _codes(torch, (m, k), 19, True), _codes(torch, (n, k), 20, True), m, n, k, True, 0,
                        with_ws)
    assert ((y - ref).norm() / ref.norm()).item() < 6e-5  # the fp8 matrix instructions' own sums, 1.5e-5 measured


@pytest.mark.parametrize("m,n,k", [(3, 5, 17), (17, 1003, 1000), (77, 130, 4099), (33, 528, 2048), (64, 4096, 14336),
                                   (12, 272, 1024), (300, 4112, 256)])
@pytest.mark.parametrize("mode", ["w8a8", "fp8"])
def test_linear_in_one_call(tq, m, n, k, mode):
    """Quantize and GEMM of one call: the bits of the two calls, nothing past the workspace
    that it asks for."""
    import torch

    from theano_quantize import _abi
    from theano_quantize._tensor import ptr, stream

    fp8 = mode == "fp8"
    x = torch.randn(m, k, generator=torch.Generator(device="cuda").manual_seed(m), device="cuda")
    qw = _codes(torch, (n, k), 15, fp8)
    sw, b = torch.rand(n, device="cuda") + 0.5, torch.randn(n, device="cuda")
    need = int(getattr(_abi.lib(), f"tq_linear_{mode}_workspace_bytes")(m, n, k))
    ws = torch.empty(need + 256, dtype=torch.uint8, device="cuda").fill_(0xA5)
    y, y2 = (torch.full((m, n), float("nan"), device="cuda") for _ in range(2))
    _abi.call(f"tq_linear_{mode}", ptr(x), m, ptr(qw), ptr(sw), ptr(b), n, k, ptr(ws), need, ptr(y), stream())
    assert bool((ws[need:] == 0xA5).all())
    qa = torch.empty(m, k, dtype=torch.uint8, device="cuda")
    sa = torch.empty(m, device="cuda")
    _abi.call("tq_quantize_fp8_rowwise" if fp8 else "tq_quantize_i8_rowwise", ptr(x), m, k, ptr(qa), ptr(sa), stream())
    nb = int(getattr(_abi.lib(), f"tq_gemm_{mode}_workspace_bytes")(m, n, k))
    part = torch.empty(max(nb, 8) + 256, dtype=torch.uint8, device="cuda").fill_(0xA5)
    args = [ptr(qa), ptr(sa), ptr(qw), ptr(sw), ptr(b), m, n, k] + ([] if fp8 else [None])
    _abi.call(f"tq_gemm_{mode}_ws", *args, ptr(part), nb, ptr(y2), stream())
    assert bool((part[nb:] == 0xA5).all())
    assert torch.equal(y, y2)
    with pytest.raises(tq.InvalidArgument):
        _abi.call(f"tq_linear_{mode}", ptr(x), m, ptr(qw), ptr(sw), ptr(b), n, k, ptr(ws), need - 1, ptr(y), stream())


def test_fp8_nan_code_stays_in_its_row_and_column(tq):
    import torch

    m, n, k = 35, 67, 200
    qa, qw = _codes(torch, (m, k), 5, True), _codes(torch, (n, k), 6, True)
    qa.view(torch.uint8)[4, k - 1] = 0x7F
    qw.view(torch.uint8)[9, 0] = 0xFF
    y, _, _, _ = _run(torch, True, qa, qw, m, n, k, False, 1, False)
    nan = torch.zeros(m, n, dtype=torch.bool, device="cuda")
    nan[4] = True
    nan[:, 9] = True
    assert torch.equal(y.isnan(), nan)


def _weight_only(torch, fp8, x, qw, m, n, k, bias, off):
    from theano_quantize import _abi
    from theano_quantize._tensor import ptr, stream

    g = torch.Generator(device="cuda").manual_seed(m + 7 * n)
    sw = torch.rand(n, generator=g, device="cuda") + 0.5
    b = torch.randn(n, generator=g, device="cuda") if bias else None
    kw, vw = _at_offset(torch, qw, off)
    name = "tq_gemm_fp8_weight" if fp8 else "tq_gemm_w8"
    nb = int(getattr(_abi.lib(), name + "_workspace_bytes")(m, n, k))
    ws = torch.empty(max(nb, 8), dtype=torch.uint8, device="cuda").fill_(0xA5)
    y = torch.full((m, n), float("nan"), device="cuda")
    _abi.call(name, ptr(x), m, ptr(vw), ptr(sw), ptr(b), n, k, ptr(ws), nb, ptr(y), stream())
    torch.cuda.synchronize()
    return y, sw, b


# the same edges with enough work (more than 4 Mi products) for the matrix-core kernels;
# the smaller shapes above run a wave per output, summed in f32
WEIGHT_SHAPES = [(17, 4160, 63), (31, 2200, 64), (33, 1025, 129), (64, 300, 255), (128, 300, 128), (65, 129, 1023),
                 (9, 4096, 4096), (6, 1003, 4100), (512, 512, 1024), (300, 4096, 256), (39, 310, 347), (18, 426, 547),
                 (266, 9904, 34), (33, 4359, 4395), (74, 11047, 34), (543, 34, 4051)]


@pytest.mark.parametrize("m,n,k", [s for s in SHAPES if s[0] > 8] + WEIGHT_SHAPES)
@pytest.mark.parametrize("fp8", [False, True])
def test_weight_only_any_shape(tq, m, n, k, fp8):
    """f32 activations with rows of very different magnitudes (and zero, subnormal and
    huge ones) times 8-bit codes against float64."""
    import torch

    g = torch.Generator(device="cuda").manual_seed(k)
    x = torch.randn(m, k, generator=g, device="cuda")
    x *= (10.0 ** torch.linspace(-8, 8, m, device="cuda"))[:, None]
    x[1] = 0
    x[2] *= 1e-36
    x[3, k // 2] *= 1e4  # one value far above its row
    qw = _codes(torch, (n, k), 8, fp8)
    for off, bias in ((0, False), (0, True), (1, True)):
        y, sw, b = _weight_only(torch, fp8, x, qw, m, n, k, bias, off)
        ref = x.double() @ qw.double().t().contiguous() * sw.double()
        scale = (x.double().abs() @ qw.double().abs().t().contiguous()) * sw.double()
        if b is not None:
            ref = ref + b.double()
        # the matrix cores' sums as in test_fp8_any_shape, over runs of 256; bits of x below
        # 2^-133 have no place in a bf16 plane; the final rounding below 2^-126 at its least
        tiny = 2.0 ** -126
        wsum = qw.double().abs().sum(1) * sw.double()
        if m * n * k > 4 << 20:
            bound = 2.0 ** -23 * min(k, 256) ** 0.5 * scale + 2.0 ** -23 * ref.abs() + 2.0 ** -133 * wsum + tiny
        else:  # f32: K / 64 additions per lane and a tree, over rounded products
            bound = 2.0 ** -23 * (k / 64 + 16) ** 0.5 * scale + 2.0 ** -23 * ref.abs() + tiny
        err = (y.double() - ref).abs()
        assert bool((err <= bound).all()), (err / bound).max().item()
        rows = torch.arange(m, device="cuda") > 2
        rel = (err[rows].norm(dim=1) / ref[rows].norm(dim=1)).max().item()
        assert rel < 4e-7 * (1 + 64 / (n * k) ** 0.5), rel


@pytest.mark.parametrize("m,k", [(13, 4096), (40, 1000), (6, 14336)])
@pytest.mark.parametrize("fp8", [False, True])
def test_weight_only_rows_of_wide_range(tq, m, k, fp8):
    """Rows that hold a few values far above the rest, against outputs whose codes there
    are zero, small or large, and outputs of one code alone: each output to f32 accuracy
    of its own sum |x| |w|, whatever the row's largest value is.  (At the least those of
    one code alone and those whose large values meet zeros were off by up to their whole
    value in a fixed-point form of x.)"""
    import torch

    n = 1500
    g = torch.Generator(device="cuda").manual_seed(k)
    x = torch.randn(m, k, generator=g, device="cuda")
    qw = _codes(torch, (n, k), 13, fp8)
    one = torch.tensor(1.0, device="cuda").to(qw.dtype)
    cols = torch.randperm(k, generator=g, device="cuda")[:100]
    raw, unit = qw.view(torch.uint8), one.view(torch.uint8)
    raw[:300, cols] = 0  # outputs that do not see the large values
    raw[300:500, cols] = unit  # or see them with the smallest whole code
    raw[500:700] = 0  # one code alone: y is that x, times a whole number
    raw[torch.arange(500, 700, device="cuda"), torch.arange(200, device="cuda") * (k // 200)] = unit
    raw[:, cols[0]] = 0  # a column that no output uses
    large = [(c, r) for r in (1e3, 1e5, 1e9, 1e30) for c in (1, 3, 100)]
    for i in range(m):
        c, r = large[i % len(large)]
        x[i, cols[:c]] *= r
    y, sw, b = _weight_only(torch, fp8, x, qw, m, n, k, False, 0)
    ref = x.double() @ qw.double().t().contiguous() * sw.double()
    mag = (x.double().abs() @ qw.double().abs().t().contiguous()) * sw.double()
    # up to 64 additions in a run of 256 k and K / 256 runs, each rounding by 2^-24 of its
    # partial sum at most, uniformly: five standard deviations
    bound = 5 / 3 ** 0.5 * 2.0 ** -24 * (64 + k / 256) ** 0.5 * mag + 2.0 ** -23 * ref.abs() + 2.0 ** -126
    err = (y.double() - ref).abs() / bound
    assert err.max().item() <= 1, (err.max().item(), err.argmax().item())


@pytest.mark.parametrize("n,k", [(5, 17), (9, 700), (33, 1023), (40, 1041), (130, 2049), (70, 4097), (35, 8200),
                                 (12, 16384), (4, 16385), (1003, 1000)])
@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 8, 11])
@pytest.mark.parametrize("fp8", [False, True])
def test_gemv_any_row_length(tq, m, n, k, fp8):
    """The GEMV over rows that end inside a lane's 16 codes and over K slices, at odd
    code addresses; the GEMV and the entry that chooses among the kernels."""
    import torch

    from theano_quantize import _abi
    from theano_quantize._tensor import ptr, stream

    g = torch.Generator(device="cuda").manual_seed(m * k)
    buf = torch.empty(m * k + 8, device="cuda")
    x = buf[1:1 + m * k].view(m, k).normal_(generator=g)  # 4-byte aligned rows
    qw = _codes(torch, (n, k), 11, fp8)
    y, sw, b = _weight_only(torch, fp8, x, qw, m, n, k, True, 3)
    kw, vw = _at_offset(torch, qw, 7)
    y2 = torch.full((m, n), float("nan"), device="cuda")
    _abi.call("tq_gemv_fp8" if fp8 else "tq_gemv_w8", ptr(x), m, ptr(vw), ptr(sw), ptr(b), n, k, ptr(y2), stream())
    ref = x.double() @ qw.double().t().contiguous() * sw.double() + b.double()
    mag = (x.double().abs() @ qw.double().abs().t().contiguous()) * sw.double() + b.double().abs()
    # chains of at most K / 64 (a wave per output) f32 additions and a tree of 6 + 8
    bound = 2.0 ** -24 * (k / 64 + 16) ** 0.5 * mag + 2.0 ** -22 * ref.abs()
    for out in (y, y2):
        assert bool(((out.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("m,n,k", [(1, 1031, 8195), (4, 513, 14336), (3, 1025, 16384), (2, 11183, 9001),
                                   (2, 11184, 9001)])
def test_w8_long_rows(tq, m, n, k):
    """Runs of several rows per block of the long-row GEMV, up to 96 Mi weights."""
    import torch

    x = torch.randn(m, k, generator=torch.Generator(device="cuda").manual_seed(m + k), device="cuda")
    qw = _codes(torch, (n, k), 12, False)
    y, sw, b = _weight_only(torch, False, x, qw, m, n, k, True, 1)
    ref = x.double() @ qw.double().t().contiguous() * sw.double() + b.double()
    mag = (x.double().abs() @ qw.double().abs().t().contiguous()) * sw.double() + b.double().abs()
    # as test_gemv_any_row_length
    bound = 2.0 ** -24 * (k / 64 + 16) ** 0.5 * mag + 2.0 ** -22 * ref.abs()
    assert bool(((y.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("m,n,k,gemv", [(8, 12288, 1024, True), (8, 12304, 1024, False), (8, 8192, 512, True),
                                        (8, 8208, 512, False), (5, 8192, 250, True), (5, 8400, 250, False), (9, 512, 1024, False),
                                        (6, 4096, 6144, True), (6, 4112, 6144, False), (8, 1024, 8192, True),
                                        (7, 1040, 8192, False), (8, 8388, 1000, True), (5, 8389, 1000, False),
                                        (8, 1024, 8208, True), (5, 1025, 8208, False), (4, 11183, 9001, True),
                                        (4, 11184, 9001, False), (3, 11184, 9001, True), (4, 12288, 10241, True)])
@pytest.mark.parametrize("fp8", [False, True])
def test_weight_only_few_tokens(tq, m, n, k, gemv, fp8):
    """Both sides of each line between the GEMV and the matrix cores."""
    import torch

    from theano_quantize import _abi
    from theano_quantize._tensor import ptr, stream

    x = torch.randn(m, k, generator=torch.Generator(device="cuda").manual_seed(n), device="cuda")
    qw = _codes(torch, (n, k), 14, fp8)
    y, sw, b = _weight_only(torch, fp8, x, qw, m, n, k, True, 0)
    ref = x.double() @ qw.double().t().contiguous() * sw.double() + b.double()
    mag = (x.double().abs() @ qw.double().abs().t().contiguous()) * sw.double() + b.double().abs()
    # as test_gemv_any_row_length
    bound = 2.0 ** -24 * (k / 64 + 16) ** 0.5 * mag + 2.0 ** -22 * ref.abs()
    assert bool(((y.double() - ref).abs() <= bound).all())
    y2 = torch.empty_like(y)
    _abi.call("tq_gemv_fp8" if fp8 else "tq_gemv_w8", ptr(x), m, ptr(qw), ptr(sw), ptr(b), n, k, ptr(y2), stream())
    assert torch.equal(y, y2) == gemv  # the GEMV's bits where it runs; other sums elsewhere


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("n,k", [(48, 384), (33, 130), (1033, 130), (512, 2048)])
def test_weight_only_rows_that_are_not_finite(tq, fp8, n, k):
    import torch

    m = 40
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn(m, k, generator=g, device="cuda")
    x[5, 3] = float("inf")
    x[6, k - 1] = float("-inf")
    x[7, 0] = float("nan")
    x.view(torch.int32)[8, 1] = 0x7F800001  # a NaN whose high half is an infinity's
    x[9, 2], x[9, 4] = float("inf"), float("-inf")
    x[10, 1] = 3.0e38
    qw = _codes(torch, (n, k), 9, fp8)
    y, sw, _ = _weight_only(torch, fp8, x, qw, m, n, k, False, 0)
    ref = x.double() @ qw.double().t().contiguous() * sw.double()
    # every class as the exact sum has it, in every row (3e38 times a code past 1 overflows f32)
    f32 = ref.float()
    assert torch.equal(y.isnan(), f32.isnan())
    rows = [i for i in range(m) if i != 10]
    assert torch.equal(y[rows].isinf(), f32[rows].isinf())
    inf = f32[rows].isinf()
    assert torch.equal(y[rows][inf], f32[rows][inf])
    # the row of 3e38: infinite where that product overflows f32, else to f32 accuracy of its sum
    p = x[10, 1].double() * qw[:, 1].double()
    over = p.abs() * sw.double().clamp(min=1) > torch.finfo(torch.float32).max
    assert torch.equal(y[10][over], (p[over].sign() * float("inf")).float())
    mag = x[10].double().abs() @ qw.double().abs().t().contiguous() * sw.double()
    err = (y[10].double() - ref[10]).abs()
    assert bool((err <= 2.0 ** -24 * (k / 64 + 16) ** 0.5 * mag + 2.0 ** -23 * ref[10].abs())[~over].all())
    fin = torch.tensor([i for i in range(m) if i not in (5, 6, 7, 8, 9, 10)], device="cuda")
    assert ((y[fin].double() - ref[fin]).norm() / ref[fin].norm()).item() < 4e-7


def test_workspace_too_small_is_refused(tq):
    import torch

    from theano_quantize import _abi
    from theano_quantize._tensor import ptr, stream

    m, n, k = 64, 100, 14336
    nb = int(_abi.lib().tq_gemm_w8a8_workspace_bytes(m, n, k))
    assert nb > 0  # two 64 x 64 tiles: K is split
    t = torch.zeros(m * k, dtype=torch.int8, device="cuda")
    f = torch.zeros(m * n, device="cuda")
    with pytest.raises(tq.InvalidArgument):
        _abi.call("tq_gemm_w8a8_ws", ptr(t), ptr(f), ptr(torch.zeros(n * k, dtype=torch.int8, device="cuda")), ptr(f),
                  None, m, n, k, None, ptr(f), nb - 1, ptr(f), stream())
    assert np.isfinite(f.cpu().numpy()).all()


def _w4(torch, tq, rows, k, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    q, s = tq.quantize_i4_g128(torch.randn(rows, k, generator=g, device="cuda") * 0.02)
    return q, s, tq.dequantize_i4_g128(q, s).double()


@pytest.mark.parametrize("m,n,k", [(33, 1000, 128), (40, 130, 14336), (65, 129, 4096), (100, 515, 384), (389, 5827, 256),
                                   (64, 4096, 2048), (300, 33, 1024), (129, 128, 8192), (35, 20, 256)])
def test_w4_linear_tiles(tq, m, n, k):
    """The INT4 Linear's tiles at edges of M and N, odd and even group counts, K split
    over blocks; packed bytes, scales and x at their elements' alignment."""
    import torch

    from theano_quantize import _abi
    from theano_quantize._tensor import ptr, stream

    q, s, w = _w4(torch, tq, n, k, 21)
    g = torch.Generator(device="cuda").manual_seed(22)
    x = torch.empty(m * k + 1, dtype=torch.bfloat16, device="cuda")[1:].view(m, k)
    x.copy_(torch.randn(m, k, generator=g, device="cuda"))
    b = torch.randn(n, generator=g, device="cuda")
    kq, vq = _at_offset(torch, q, 3)
    ks, vs = _at_offset(torch, s, 2)
    ref = x.double() @ w.t().contiguous() + b.double()
    mag = x.double().abs() @ w.abs().t().contiguous() + b.double().abs()
    nb = int(_abi.lib().tq_linear_w4g128_workspace_bytes(m, n, k))
    ws = torch.empty(max(nb, 8), dtype=torch.uint8, device="cuda").fill_(0xA5)
    for name, extra in (("tq_linear_w4g128", [ptr(ws), nb]), ("tq_gemm_w4g128_bf16", [])):
        y = torch.full((m, n), float("nan"), device="cuda")
        _abi.call(name, ptr(x), m, ptr(vq), ptr(vs), ptr(b), n, k, *extra, ptr(y), stream())
        # eight MFMA additions of 16 exact products per group, each within 2^-23 of the largest
        # partial sum, then one per group; the pipelined kernels' offset form (K % 256, N % 128)
        # adds 24 times the activations' sum and takes it away again
        off = 24.0 if nb and k % 256 == 0 and n % 128 == 0 else 1.0
        bound = 2.0 ** -23 * off * (8 + k / 128) ** 0.5 * mag + 2.0 ** -22 * ref.abs()
        assert bool(((y.double() - ref).abs() <= bound).all()), name


@pytest.mark.parametrize("m,d,f", [(33, 128, 128), (48, 640, 1408), (100, 384, 128), (65, 128, 3200), (200, 1152, 384),
                                   (300, 256, 2432), (64, 2048, 256), (130, 4096, 384)])
def test_w4_mlp_tiles(tq, m, d, f):
    """The FFN's tiles, with their own workspace (K split) and with the least one."""
    import torch

    (g, gs, gw), (u, us, uw), (dn, ds, dw) = (_w4(torch, tq, r, c, 30 + i)
                                              for i, (r, c) in enumerate([(f, d), (f, d), (d, f)]))
    mlp = tq.QuantizedMLP(d, f, (g, gs), (u, us), (dn, ds), tiled=False)
    gen = torch.Generator(device="cuda").manual_seed(d + f)
    x = torch.randn(m, d, generator=gen, device="cuda").to(torch.bfloat16)
    a = x.double() @ gw.t().contiguous()
    h = a / (1 + torch.exp(-a)) * (x.double() @ uw.t().contiguous())
    ref = h @ dw.t().contiguous()
    least = torch.empty(mlp.workspace_bytes(m), dtype=torch.uint8, device="cuda").fill_(0xA5)
    for ws in (None, least):
        y = mlp.forward(x, ws).double()
        rel = ((y - ref).norm() / ref.norm()).item()
        assert rel < 2e-5, rel  # h is handed over as bf16 hi + lo, 2^-17 of each
        assert bool(((y - ref).abs() <= 1e-4 + 1e-3 * ref.abs()).all())
