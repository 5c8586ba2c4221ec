"""Prefill tiles of 64, 128 and 256 rows, split and unsplit, and SwiGLU inside the prefill.

Against float64 of the device's own dequantized weights (bit-exact by the dequant tests);
the bar is the prefill's 1e-3 normwise (f16 operands; Q4_K, Q5_K measure 6.8e-4).
"""
import numpy as np
import pytest
import torch

from unillm_amd import (PATH_DECODE_MFMA, PATH_PREFILL_MFMA, Q4_0, Q4_K, Q5_0, Q5_K, Q6_K, Q8_0,
                        QuantLinear, _capi)

pytestmark = pytest.mark.gpu

TOL = 1e-3
# (block bytes, weights, offsets of the f16 scales)
BLOCK = {Q4_0: (18, 32, [0]), Q5_0: (22, 32, [0]), Q8_0: (34, 32, [0]),
         Q4_K: (144, 256, [0, 2]), Q5_K: (176, 256, [0, 2]), Q6_K: (210, 256, [208])}


def _weight(qtype, n, k, seed):
    size, elems, scales = BLOCK[qtype]
    rng = np.random.default_rng(seed)
    b = rng.integers(0, 256, (n * k // elems, size), dtype=np.uint8)
    for off in scales:
        d = rng.uniform(0.5e-3, 2e-3, b.shape[0]).astype(np.float16)
        b[:, off:off + 2] = d.view(np.uint8).reshape(-1, 2)
    return QuantLinear.from_blocks(qtype, n, k, b.tobytes())


def _err(y, ref):
    return ((y.double() - ref).norm() / ref.norm()).item()


def _norm64(x, gamma, beta, eps):
    d = x.double() - x.double().mean(-1, keepdim=True)
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + eps) * gamma.double() + beta.double()


# m around the tile heights; n that leaves a ragged last tile; k of a few steps, an odd
# block count (not the K-quants), and a deep one that splits
@pytest.mark.parametrize("qtype", list(BLOCK))
@pytest.mark.parametrize("m,n,k", [(33, 300, 2048), (64, 257, 8192), (65, 1000, 1024),
                                   (127, 255, 512), (129, 520, 4096), (200, 4096, 768),
                                   (257, 130, 2048), (300, 2049, 256)])
def test_prefill_plans(qtype, m, n, k):
    if qtype in (Q4_0, Q5_0, Q8_0):
        k += 32  # an odd number of blocks: the last k step is half full
    print(f"prefill plan qtype={qtype} m={m} n={n} k={k}", flush=True)
    ql = _weight(qtype, n, k, m + n)
    w = ql.dequantize().double()
    x = torch.randn(m, k, device="cuda", generator=torch.Generator("cuda").manual_seed(m))
    ref = x.double() @ w.t()
    y = ql.forward(x, path=PATH_PREFILL_MFMA)
    assert _err(y, ref) < TOL
    assert torch.equal(ql.forward(x, path=PATH_PREFILL_MFMA), y)
    if m > 64:
        r = torch.randn_like(y)
        want = r.double() + ref
        assert _err(ql.forward_add(x, r), want) < TOL


# I: not a multiple of a column tile (16), a workgroup's 128 outputs, or 4; unsplit (many
# columns or a short k) and split
@pytest.mark.parametrize("qtype", [Q4_0, Q8_0, Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("m,I,k", [(65, 30, 256), (100, 129, 2048), (130, 1000, 512),
                                   (256, 4100, 256), (520, 2061, 768), (300, 8200, 512)])
def test_prefill_swiglu(qtype, m, I, k):
    print(f"prefill swiglu qtype={qtype} m={m} I={I} k={k}", flush=True)
    ql = _weight(qtype, 2 * I, k, m + I)
    w = ql.dequantize().double()
    g = torch.Generator("cuda").manual_seed(m)
    x = 0.1 * torch.randn(m, k, device="cuda", generator=g)
    gate, up = (x.double() @ w.t()).chunk(2, -1)
    assert ql.select_path(m) == PATH_PREFILL_MFMA
    act = ql.forward_swiglu(x)
    assert _err(act, gate * torch.sigmoid(gate) * up) < 4 * TOL  # a product of two
    # an output that is not 16-byte aligned takes the scalar sums: the same bits
    buf = torch.empty(m * I + 1, device="cuda")
    assert torch.equal(ql.forward_swiglu(x, out=buf[1:].view(m, I)), act)
    gam, bet = torch.rand(k, device="cuda"), 0.1 * torch.rand(k, device="cuda")
    gate, up = (_norm64(x, gam, bet, 1e-6) @ w.t()).chunk(2, -1)
    act = ql.forward_swiglu(x, norm=(gam, bet, 1e-6))
    assert _err(act, gate * torch.sigmoid(gate) * up) < 4 * TOL


# the rows of a batch that run on the prefill's tiles (the same bits every call, unlike the
# batched decode's own kernels): right, with SwiGLU, inside a reserved capture and through
# the no-allocation entry point; and their neighbours that do not
@pytest.mark.parametrize("qtype,m,n,k,tiles", [
    (Q8_0, 33, 4096, 11008, True), (Q8_0, 32, 4096, 11008, False),
    (Q4_K, 49, 4096, 14336, True), (Q4_K, 48, 4096, 14336, False),
    (Q6_K, 64, 3000, 14336, True), (Q4_0, 64, 2048, 8192, False),
    (Q4_0, 64, 1024, 491520, False)])  # 60 MiB of x: slabs beside it would not fit the scratch
def test_batch_on_the_prefill(qtype, m, n, k, tiles):
    print(f"batch on the prefill qtype={qtype} m={m} n={n} k={k}", flush=True)
    ql = _weight(qtype, n, k, 3)
    assert ql.select_path(m) == PATH_DECODE_MFMA
    x = torch.randn(m, k, device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    y = ql.forward(x)
    assert _err(y, x.double() @ ql.dequantize().double().t()) < TOL
    # (the batched decode adds its slices in any order)
    close = (lambda a: torch.equal(a, y)) if tiles else (lambda a: _err(a, y.double()) < 1e-5)
    gate, up = y.double().chunk(2, -1)
    assert _err(ql.forward_swiglu(x), gate * torch.sigmoid(gate) * up) < 1e-5
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    ql.reserve(m, swiglu=True, stream=s)
    out = torch.empty_like(y)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s, capture_error_mode="thread_local"):
        ql.forward(x, out=out, stream=s)
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            g.replay()
        s.synchronize()
        assert close(out)
    del g
    z = torch.empty_like(y)
    _capi.check(_capi.lib().unillm_hip_qmatmul_noalloc(
        ql._h, x.data_ptr(), m, z.data_ptr(), int(torch.cuda.current_stream().cuda_stream)))
    torch.cuda.synchronize()
    assert close(z)


# a batch's x is scaled by slices of at most 1024 k on the prefill's tiles too: a value far
# larger than the rest of its row (behind 1024 zero weights) costs the other slices nothing
@pytest.mark.parametrize("qtype", [Q4_0, Q8_0, Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("m,n,k", [(64, 4096, 14336), (50, 2900, 14592), (64, 28672, 4096)])
def test_batch_outlier_keeps_the_other_slices(qtype, m, n, k):
    print(f"batch outlier qtype={qtype} m={m} n={n} k={k}", flush=True)
    size, elems, scales = BLOCK[qtype]
    rng = np.random.default_rng(5)
    b = rng.integers(0, 256, (n, k // elems, size), dtype=np.uint8)
    for off in scales:
        d = rng.uniform(0.5e-3, 2e-3, b.shape[:2]).astype(np.float16)
        d[:, : 1024 // elems] = 0
        b[:, :, off:off + 2] = d.view(np.uint8).reshape(n, -1, 2)
    ql = QuantLinear.from_blocks(qtype, n, k, b.tobytes())
    x = torch.randn(m, k, device="cuda", generator=torch.Generator("cuda").manual_seed(m))
    x[:, 3] = 1e13
    x[::2, 3] = 1e30
    w = ql.dequantize()
    assert not w[:, :1024].any()
    ref = x[:, 1024:].double() @ w[:, 1024:].double().t()
    y = ql.forward(x)
    assert _err(y, ref) < TOL
    r = torch.randn_like(y)
    want = r.double() + ref
    assert _err(ql.forward_add(x, r), want) < TOL


# a batch takes the faster of the batched decode and the prefill's tiles: sizes where the tiles
# (asked for by path) lose a fifth to a third, and one where the decode does
@pytest.mark.parametrize("qtype,m,n,k,tiles", [(Q6_K, 64, 24576, 9216, False),
                                               (Q4_0, 56, 24576, 11008, False),
                                               (Q8_0, 40, 24576, 11008, False),
                                               (Q4_0, 64, 3072, 14336, False),
                                               (Q8_0, 64, 4096, 14336, True)])
def test_batch_takes_the_faster_kernels(qtype, m, n, k, tiles):
    print(f"batch speed qtype={qtype} m={m} n={n} k={k}", flush=True)
    # (in turn over weights that together outgrow the 256 MiB cache, as a model meets them: one
    # weight that stays in the cache measures even at 24576 columns)
    qls = [_weight(qtype, n, k, i) for i in range(2 if n * k > 1 << 27 else 6)]
    x = torch.randn(m, k, device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    out = torch.empty(m, n, device="cuda")

    def timed(**path):
        best = 1e9
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for i in range(24):
                qls[i % len(qls)].forward(x, out=out, **path)
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b))
        return best

    timed()
    auto, asked = timed(), timed(path=PATH_PREFILL_MFMA)
    assert auto < asked * (1.1 if tiles else 0.95)
