"""The prompt attention kernel over its plans: block heights, pairing, key splits, tails.

Against float64 attention with RoPE at the reference's f32 angles (positions times f32
frequencies, llama.rs:827-883).  The products keep f32's 24 bits and sum in f32: 1e-6
normwise (the f32 matrix cores measured 3.8e-7 at the same shapes).
"""
import math

import pytest
import torch

from unillm_amd import KvCache

pytestmark = pytest.mark.gpu

TOL = 1e-6


def _rope(t, pos, hd):
    e = torch.arange(0, hd, 2, device="cuda", dtype=torch.float32) / hd
    inv = 1.0 / torch.pow(torch.tensor(10000.0, dtype=torch.float64, device="cuda"),
                          e.double()).float()
    ang = (pos.float()[:, None] * inv).double()[:, None, :]
    a, b = t[..., : hd // 2], t[..., hd // 2:]
    return torch.cat([a * ang.cos() - b * ang.sin(), a * ang.sin() + b * ang.cos()], -1)


def _reference(x, H, KVH, hd, past):
    """x: every token's qkv row; the outputs of tokens past .. (each from its own keys only)."""
    n = x.shape[0]
    q, k, v = x.double().split([H * hd, KVH * hd, KVH * hd], -1)
    pos = torch.arange(n, device="cuda")
    q, k = _rope(q.view(n, H, hd), pos, hd), _rope(k.view(n, KVH, hd), pos, hd)
    v = v.view(n, KVH, hd)
    out = torch.empty(n - past, H, hd, dtype=torch.float64, device="cuda")
    seen = pos[None, :] <= pos[past:, None]
    for h in range(H):
        g = h // (H // KVH)
        s = (q[past:, h] @ k[:, g].t()) / math.sqrt(hd)
        p = torch.softmax(s.masked_fill(~seen, -math.inf), -1)
        out[:, h] = torch.where(seen[:, :, None], p[:, :, None] * v[None, :, g], 0.0).sum(1) \
            if n <= 256 else p @ v[:, g]
    return out.view(n - past, H * hd)


def _run(x, H, KVH, hd, past, room=0):
    kv = KvCache(KVH, hd, x.shape[0] + room)
    if past:
        kv.attention(x[:past].contiguous(), H)
    return kv.attention(x[past:].contiguous(), H)


# one query tile to many blocks; odd and even block counts; a past that leaves tiles and
# steps unaligned, fits one step, or is longer than the prompt; a full and a roomy cache
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("m,past,H,KVH", [(17, 0, 4, 4), (33, 31, 4, 1), (64, 0, 16, 8),
                                          (65, 1000, 8, 2), (128, 63, 8, 8), (129, 64, 4, 4),
                                          (300, 5, 16, 4), (513, 0, 32, 32), (1100, 77, 8, 8),
                                          (40, 3000, 32, 4)])
def test_prompt_plans(hd, m, past, H, KVH):
    print(f"prompt hd={hd} m={m} past={past} H={H} KVH={KVH}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(m + past)
    x = torch.randn(past + m, (H + 2 * KVH) * hd, device="cuda", generator=g)
    ref = _reference(x, H, KVH, hd, past)
    out = _run(x, H, KVH, hd, past, room=m % 3 * 50)
    assert ((out.double() - ref).norm() / ref.norm()).item() < TOL
    assert torch.equal(_run(x, H, KVH, hd, past), out)


# large and small scores, and running maxima that keep rising (the lazy rescale)
@pytest.mark.parametrize("scale", [0.0, 1e-3, 6.0])
def test_prompt_score_ranges(scale):
    H, KVH, hd, m = 4, 2, 64, 200
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn(m, (H + 2 * KVH) * hd, device="cuda", generator=g)
    x[:, : (H + KVH) * hd] *= scale * torch.linspace(0.5, 1.5, m, device="cuda")[:, None]
    ref = _reference(x, H, KVH, hd, 0)
    out = _run(x, H, KVH, hd, 0)
    # a score of size s rounds to 2^-24 s in f32, and so do its exponentials
    assert ((out.double() - ref).norm() / ref.norm()).item() < TOL * max(1.0, 36 * scale / 6)


# non-finite keys and values reach exactly the outputs that see them, as in f32
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("what", ["v_inf", "v_nan", "k_inf", "q_nan"])
def test_prompt_non_finite(hd, what):
    H, KVH, m, past = 4, 2, 100, 37
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(past + m, (H + 2 * KVH) * hd, device="cuda", generator=g)
    bad = float("nan") if what.endswith("nan") else float("inf")
    col = {"q": 5, "k": H * hd + 5, "v": (H + KVH) * hd + 5}[what[0]]
    x[past + 50, col] = bad
    if what == "v_inf":
        x[3, col + hd] = -bad  # in the past, the other kv head
    ref = _reference(x, H, KVH, hd, past).float()
    out = _run(x, H, KVH, hd, past)
    assert torch.equal(out.isnan(), ref.isnan())
    assert torch.equal(out.isinf(), ref.isinf())
    assert torch.equal(out[out.isinf()], ref[ref.isinf()])
    fin = ref.isfinite()
    assert fin.any()
    assert ((out - ref)[fin].norm() / ref[fin].norm()).item() < TOL


# every query of odd 32-query tiles non-finite: the tiles beside them in their workgroup
# keep the bits they have without (each redone tile stays in its own part of LDS)
@pytest.mark.parametrize("hd,m,H", [(64, 128, 4), (128, 128, 4), (64, 1024, 32), (128, 1024, 32)])
def test_prompt_redone_tiles_leave_the_others(hd, m, H):
    print(f"prompt redone tiles hd={hd} m={m} H={H}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(m + hd)
    x = torch.randn(m, 3 * H * hd, device="cuda", generator=g)
    clean = _run(x, H, H, hd, 0)
    odd = torch.arange(m, device="cuda") // 32 % 2 == 1
    x[odd, :H * hd] = float("nan")
    out = _run(x, H, H, hd, 0)
    assert out[odd].isnan().all()
    assert torch.equal(out[~odd], clean[~odd])


# out over qkv (a caller that reuses the projection's buffer): the same bits as beside it;
# unsplit plans, a split one, a decode step, hd 256; and inside a capture
@pytest.mark.parametrize("hd,m,past,H,KVH", [(128, 300, 0, 32, 32), (64, 1000, 0, 32, 4),
                                             (64, 40, 3000, 32, 4), (128, 1, 100, 8, 8),
                                             (256, 40, 5, 4, 2)])
def test_prompt_out_over_qkv(hd, m, past, H, KVH):
    print(f"prompt out over qkv hd={hd} m={m} past={past} H={H} KVH={KVH}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(m)
    width = (H + 2 * KVH) * hd
    x = torch.randn(past + m, width, device="cuda", generator=g)
    want = _run(x, H, KVH, hd, past)
    kv = KvCache(KVH, hd, past + m)
    if past:
        kv.attention(x[:past].contiguous(), H)
    buf = torch.empty(2 * m * width, device="cuda")
    qkv = buf[:m * width].view(m, width)
    s = torch.cuda.Stream()
    kv.reserve(m, H, stream=s)
    for first in (0, 64, m * width - 64, m * width - m * H * hd):  # floats out lies behind qkv
        out = buf[first:first + m * H * hd].view(m, H * hd)
        qkv.copy_(x[past:])
        assert torch.equal(kv.attention(qkv, H, out=out), want)
        kv.truncate(past)
    out = buf[:m * H * hd].view(m, H * hd)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s, capture_error_mode="thread_local"):
        kv.attention(qkv, H, out=out, stream=s)
    for i in range(3):
        kv.truncate(past)
        qkv.copy_(x[past:])
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            graph.replay()
        s.synchronize()
        # (a capture may split the keys otherwise)
        assert ((out - want).norm() / want.norm()).item() < TOL
    del graph


# scores of -inf from position 128 on: a key split that holds no other key (m 40 behind 3000
# takes eight) weighs nothing, and an unsplit call the same
@pytest.mark.parametrize("hd,m,past,H,KVH", [(64, 40, 3000, 32, 4), (128, 40, 3000, 32, 4),
                                             (128, 300, 0, 32, 32)])
def test_prompt_keys_without_weight(hd, m, past, H, KVH):
    print(f"prompt keys without weight hd={hd} m={m} past={past}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(hd + m)
    x = torch.randn(past + m, (H + 2 * KVH) * hd, device="cuda", generator=g)
    # the slowest rotation pair: its angle stays small, so a query of (1, 1) keeps both signs
    q = x[:, :H * hd].view(-1, H, hd)
    q[:, :, hd // 2 - 1] = q[:, :, hd - 1] = 1.0
    x[128:, H * hd:(H + KVH) * hd].view(-1, KVH, hd)[:, :, hd // 2 - 1] = -math.inf
    ref = _reference(x, H, KVH, hd, past)
    assert ref.isfinite().all()
    out = _run(x, H, KVH, hd, past)
    assert ((out.double() - ref).norm() / ref.norm()).item() < TOL


# a NaN row in the middle of a tile, NaN and infinite values behind each other, and every row
# non-finite, over plans that split and pair: exactly the outputs that see them, and soon: a
# recompute costs a scan of the keys a query at most, dealt over the block's waves (m1500
# all-inf v measured under 4 ms; the bar leaves room for a busy machine)
@pytest.mark.parametrize("hd,m,past,H,KVH", [(64, 250, 0, 8, 4), (128, 250, 10, 8, 8),
                                             (64, 45, 900, 32, 4), (128, 45, 900, 32, 4)])
@pytest.mark.parametrize("what", ["row_nan", "v_nan_then_inf", "all_nan", "v_all_inf"])
def test_prompt_redo(hd, m, past, H, KVH, what):
    print(f"prompt redo hd={hd} m={m} past={past} {what}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(hd + m)
    n = past + m
    x = torch.randn(n, (H + 2 * KVH) * hd, device="cuda", generator=g)
    v = x[:, (H + KVH) * hd:].view(n, KVH, hd)
    if what == "row_nan":
        x[past + 21] = math.nan
    elif what == "v_nan_then_inf":
        v[past + 3, 0, 5] = math.nan
        v[past + 9, 1, 6] = math.inf
        v[past + 30, 1, 6] = -math.inf
        v[past + 40, 0, 7] = -math.inf
    elif what == "all_nan":
        x[past:] = math.nan
    else:
        v[past] = math.inf
    ref = _reference(x, H, KVH, hd, past) if n <= 256 else None
    if ref is None:  # each query's own keys: 0 * inf of a masked key is not part of it
        ref = torch.stack([_reference(x[:past + t + 1], H, KVH, hd, past + t)[0]
                           for t in range(m)])
    ref = ref.float()
    out = _run(x, H, KVH, hd, past)
    assert torch.equal(out.isnan(), ref.isnan())
    assert torch.equal(out[out.isinf()], ref[ref.isinf()])
    fin = ref.isfinite()
    if fin.any():
        assert ((out - ref)[fin].norm() / ref[fin].norm()).item() < TOL


def test_prompt_redo_cost():
    H, hd, m = 32, 128, 1500
    x = torch.randn(m, 3 * H * hd, device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    x[0, 2 * H * hd:] = math.inf  # every query of every head
    kv = KvCache(H, hd, m)
    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    kv.attention(x, H)
    kv.clear()
    a.record()
    kv.attention(x, H)
    b.record()
    torch.cuda.synchronize()
    assert a.elapsed_time(b) < 40.0


# a captured call serves every length: right at each, and behind a long past its keys are still
# divided among workgroups (1.4 times the eager call's time measured; kept whole, 4 times)
@pytest.mark.parametrize("hd,m,H,KVH", [(128, 32, 32, 8), (64, 40, 32, 4), (128, 128, 32, 32)])
def test_prompt_captured_at_every_length(hd, m, H, KVH):
    print(f"prompt captured hd={hd} m={m}", flush=True)
    L = 4096
    g = torch.Generator(device="cuda").manual_seed(m)
    x = torch.randn(L, (H + 2 * KVH) * hd, device="cuda", generator=g)
    kv, s = KvCache(KVH, hd, L), torch.cuda.Stream()
    qkv, out = x[:m].clone(), torch.empty(m, H * hd, device="cuda")
    kv.reserve(m, H, stream=s)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s, capture_error_mode="thread_local"):
        kv.attention(qkv, H, out=out, stream=s)

    def timed(f):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            a.record()
            f()
            b.record()
        torch.cuda.synchronize()
        return a.elapsed_time(b)

    for past in (0, 100, L - m):
        kv.clear()
        if past:
            kv.attention(x[:past].contiguous(), H)
        qkv.copy_(x[past:past + m])
        best, eager = 1e9, 1e9
        for _ in range(4):
            kv.truncate(past)
            best = min(best, timed(graph.replay))
            got = out.clone()
            kv.truncate(past)
            eager = min(eager, timed(lambda: kv.attention(qkv, H, out=out, stream=s)))
        assert ((got - out).norm() / out.norm()).item() < TOL
    assert best < 2.5 * eager
    del graph
