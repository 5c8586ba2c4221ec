"""Two host threads on one stream: calls of several launches keep their own data.

Such a call hands its rows from launch to launch through the stream's workspaces; another
thread's launches must not come between.  Each thread's outputs are compared, bit for bit,
with the same call made alone (the paths here add their sums in a fixed order).
"""
import threading

import numpy as np
import pytest
import torch

from unillm_amd import KvCache, Q8_0, QuantLinear

pytestmark = pytest.mark.gpu

ROUNDS = 40


def _dense(g, n, k):
    return QuantLinear.from_dense((torch.randn(n, k, device="cuda", generator=g) * 0.05).bfloat16())


def _quant(n, k):
    rng = np.random.default_rng(n)
    b = rng.integers(0, 256, (n * k // 32, 34), dtype=np.uint8)
    d = rng.uniform(0.5e-3, 2e-3, b.shape[0]).astype(np.float16)
    b[:, :2] = d.view(np.uint8).reshape(-1, 2)
    return QuantLinear.from_blocks(Q8_0, n, k, b.tobytes())


@pytest.mark.parametrize("what", ["dense_norm", "dense_swiglu", "prefill_swiglu", "attention"])
def test_threads_share_a_stream(what):
    print(f"threads share a stream: {what}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(11)
    m, n, k, H, hd = (100, 1024, 512, 8, 64)
    ql = _quant(n, k) if what == "prefill_swiglu" else _dense(g, n, k)
    gamma = torch.rand(k, device="cuda", generator=g)
    s = torch.cuda.Stream()

    def maker(seed):
        g = torch.Generator(device="cuda").manual_seed(seed)
        if what == "attention":
            x = torch.randn(m, 3 * H * hd, device="cuda", generator=g)
            caches = [KvCache(H, hd, m) for _ in range(ROUNDS + 1)]
            return lambda i, out: caches[i].attention(x, H, out=out, stream=s), H * hd
        x = torch.randn(m, k, device="cuda", generator=g) * 0.1
        if what == "dense_norm":
            return lambda i, out: ql.forward_norm(x, gamma, out=out, stream=s), n
        return lambda i, out: ql.forward_swiglu(x, out=out, stream=s), n // 2

    calls = [maker(seed) for seed in (1, 2)]
    outs = [torch.zeros(ROUNDS + 1, m, width, device="cuda") for _, width in calls]
    torch.cuda.synchronize()
    for (call, _), out in zip(calls, outs):
        call(ROUNDS, out[ROUNDS])
    torch.cuda.synchronize()
    start = threading.Barrier(2)
    failed = []

    def work(t):
        try:
            start.wait()
            for i in range(ROUNDS):
                calls[t][0](i, outs[t][i])
        except Exception as e:  # noqa: BLE001  (reported by the main thread)
            failed.append(e)

    threads = [threading.Thread(target=work, args=(t,)) for t in (0, 1)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not failed, failed
    for out in outs:
        assert torch.equal(out[:ROUNDS], out[ROUNDS].expand_as(out[:ROUNDS]))
