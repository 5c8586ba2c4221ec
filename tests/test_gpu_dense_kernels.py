"""The dense weights' GEMV and split-part GEMM at the edges of their tiles and plans.

Against float64 of the exactly widened weights: an f32 sum over k rounds at most once a
product, so 1e-6 normwise up to k 4096 (an f32 GEMM measures 5.8e-7 there).  Non-finite
operands are compared with the f32 product of the same rows.
"""
import pytest
import torch

from unillm_amd import QuantLinear

pytestmark = pytest.mark.gpu

TOL = 1e-6
DTYPES = [torch.float32, torch.float16, torch.bfloat16]


def _err(y, ref):
    return ((y.double() - ref).norm() / ref.norm()).item()


def _make(m, n, k, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    w = (torch.randn(n, k, device="cuda", generator=g) * 0.05).to(dtype)
    return w, torch.randn(m, k, device="cuda", generator=g)


# m: the GEMV's token counts (1, 2, 4, 8) and past its LDS limit (3 x 11008, 8 x 4104),
# tiles of 64 and 128 rows with remainders; n: 1, and around the 128 / 256 column tiles;
# k: one element, odd, around the padding to 64, split and unsplit
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (1, 255, 511), (2, 257, 4096), (3, 40, 11008),
                                   (7, 130, 520), (8, 129, 4096), (8, 129, 4104), (9, 1, 63),
                                   (63, 256, 64), (64, 257, 65), (65, 127, 2048), (129, 300, 4096),
                                   (400, 129, 200)])
def test_dense_edges(dtype, m, n, k):
    print(f"dense edges {dtype} m={m} n={n} k={k}", flush=True)
    w, x = _make(m, n, k, dtype, 31 * m + n + k)
    ql = QuantLinear.from_dense(w)
    ref = x.double() @ w.double().t()
    y = ql.forward(x)
    assert _err(y, ref) < TOL
    assert torch.equal(ql.forward(x), y)
    r = torch.randn_like(y)
    want = r.double() + ref
    assert _err(ql.forward_add(x, r), want) < TOL
    # x at a 4-byte offset
    buf = torch.empty(m * k + 1, device="cuda")
    buf[1:] = x.reshape(-1)
    assert torch.equal(ql.forward(buf[1:].view(m, k)), y)


# the GEMV's row pairs (4096 waves on 256 CUs): one wave with a second row, all of them,
# a single third row, one fewer; x rows that can and cannot be staged 16 bytes a lane
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,n,k", [(3, 4097, 264), (4, 8192, 511), (8, 8193, 130), (5, 12287, 64)])
def test_dense_gemv_row_pairs(dtype, m, n, k):
    print(f"dense row pairs {dtype} m={m} n={n} k={k}", flush=True)
    w, x = _make(m, n, k, dtype, n)
    ql = QuantLinear.from_dense(w)
    y = ql.forward(x)
    assert _err(y, x.double() @ w.double().t()) < TOL
    for t in range(m):  # a token's bits do not depend on how many share the call
        assert torch.equal(ql.forward(x[t:t + 1].contiguous())[0], y[t])


# rows of very different size, and weights in the subnormal range of f16
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m", [2, 40])
def test_dense_wide_ranges(dtype, m):
    n, k = 200, 512
    w, x = _make(m, n, k, dtype, 5)
    w[::3] = (w[::3].float() * 1e-4).to(dtype)
    x *= torch.logspace(-12, 12, m, device="cuda")[:, None]
    x[:, 7] *= 1e4  # one outlier a row
    ql = QuantLinear.from_dense(w)
    y, ref = ql.forward(x), x.double() @ w.double().t()
    # an f32 dot's own bound, element by element: its error is relative to sum |x w|
    size = x.double().abs() @ w.double().abs().t()
    assert ((y.double() - ref).abs() / size).max().item() < TOL


# infinities and NaNs go where the f32 product takes them, and nowhere else
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,n,k", [(4, 100, 256), (70, 300, 256), (40, 64, 2048)])
def test_dense_non_finite(dtype, m, n, k):
    w, x = _make(m, n, k, dtype, 9)
    w = w.abs().clamp_min(0.0078125).to(dtype)  # no zeros: inf * w stays inf
    w[:, 4] = 1.0  # exact in one part: the lower parts are zero
    x[0, 4] = float("inf")
    x[1, 9] = float("-inf")
    x[2, 11] = float("nan")
    w[5, 20] = float("inf")
    ql = QuantLinear.from_dense(w)
    y, ref = ql.forward(x), (x.double() @ w.double().t()).float()
    assert torch.equal(y.isnan(), ref.isnan())
    assert torch.equal(y.isinf(), ref.isinf())
    assert torch.equal(y[y.isinf()], ref[ref.isinf()])
    fin = ref.isfinite()
    assert ((y - ref)[fin].norm() / ref[fin].norm()).item() < TOL


# sums of few terms, where a product's own rounding shows: within f32's bound, each FMA one
# rounding (k 2^-24 of sum |x w|), and no worse than the f32 library product of the widened
# weights (5 % for the draw)
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 8, 31, 32, 33, 64, 100])
def test_dense_short_k(dtype, k):
    m, n = 130, 300
    w, x = _make(m, n, k, dtype, 77 + k)
    if k == 1:  # a product whose parts cut off, not rounded, would lose the most
        w[0], x[0] = 1 + 2 ** -7, 1 + 2 ** -7 - 2 ** -23
        if dtype == torch.float32:
            w[0] = 1 + 2 ** -7 - 2 ** -23
    ql = QuantLinear.from_dense(w)
    y, ref = ql.forward(x), x.double() @ w.double().t()
    size = x.double().abs() @ w.double().abs().t()
    assert ((y.double() - ref).abs() / size).max().item() <= k * 2 ** -24
    assert _err(y, ref) <= 1.05 * _err(x @ w.float().t(), ref)
    r = torch.randn_like(y)
    assert _err(ql.forward_add(x, r.clone()), r.double() + ref) < TOL


# an x far larger than the rest of its row, in a column of zero weights: the rest keeps f32's
# precision on every path (GEMV, GEMM, split k)
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,n,k", [(8, 300, 512), (40, 300, 512), (40, 300, 4096), (200, 64, 512)])
@pytest.mark.parametrize("outlier", [1e6, 1e9, 1e13, 1e30])
def test_dense_outlier_behind_zero_weights(dtype, m, n, k, outlier):
    w, x = _make(m, n, k, dtype, 21)
    w[:, 9] = 0
    x[:, 9] = outlier
    x[::2, 20] = -outlier
    w[:, 20] = 0
    ql = QuantLinear.from_dense(w)
    assert _err(ql.forward(x), x.double() @ w.double().t()) < TOL


# rows of x that hold a NaN at their end, and an infinity at their start: right, and soon (the
# first without a dot; m300 k4096 n2048 measured under 0.1 and 2 ms: the bars leave room for a
# busy machine)
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,n,k", [(300, 2048, 4096), (40, 300, 1040), (30, 200, 71)])
def test_dense_non_finite_rows(dtype, m, n, k):
    w, x = _make(m, n, k, dtype, 3)
    ql = QuantLinear.from_dense(w)
    clean = ql.forward(x)
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(4)]
    bad = x.clone()
    bad[::2, k - 1] = float("nan")
    inf = x.clone()
    inf[1::2, 0] = float("inf")
    torch.cuda.synchronize()
    ev[0].record()
    y = ql.forward(bad)
    ev[1].record()
    ev[2].record()
    z = ql.forward(inf)
    ev[3].record()
    torch.cuda.synchronize()
    assert y[::2].isnan().all() and torch.equal(y[1::2], clean[1::2])
    ref = inf.double() @ w.double().t()
    assert torch.equal(z.isnan(), ref.isnan()) and torch.equal(z[z.isinf()].double(), ref[ref.isinf()])
    assert torch.equal(z[::2], clean[::2])
    assert ev[0].elapsed_time(ev[1]) < 4.0
    assert ev[2].elapsed_time(ev[3]) < 30.0


# calls that run in several chunks of rows (k 65536: 640 rows each), and more rows than a
# launch of one workgroup each holds (2^24): of x, and of a weight whose k is padded
@pytest.mark.parametrize("dtype", DTYPES)
def test_dense_row_chunks(dtype):
    m, n, k = 1300, 70, 65536
    w, x = _make(m, n, k, dtype, 4)
    ql = QuantLinear.from_dense(w)
    y, ref = ql.forward(x), x.double() @ w.double().t()
    assert _err(y, ref) < 4 * TOL  # (f32 rounds once a k: 4 times the sum length of TOL's)
    for r in (0, 640, 1280):
        assert torch.equal(ql.forward(x[r:r + 640].contiguous()), y[r:r + 640])


def test_dense_very_many_rows():
    m, n, k = (1 << 24) + 300, 3, 6
    w, x = _make(m, n, k, torch.bfloat16, 6)
    y = QuantLinear.from_dense(w).forward(x)
    assert _err(y[-1000:], x[-1000:].double() @ w.double().t()) < TOL
    assert _err(y[::4099], x[::4099].double() @ w.double().t()) < TOL
    del x, y
    w, x = _make(2, m, 2, torch.float16, 7)
    ql = QuantLinear.from_dense(w)
    assert _err(ql.forward(x), x.double() @ w.double().t()) < TOL
    assert torch.equal(ql.dequantize()[-5000:], w[-5000:].float())
