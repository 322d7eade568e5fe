"""The small layer ops' shared scratch on the null stream (qh_ops.hip): calls of two threads on it and
of a third on a stream of its own, interleaved, give what each gives alone, bit for bit."""
import threading

import numpy as np
import pytest

from conftest import assert_bitwise

pytestmark = pytest.mark.gpu


def test_threads_share_the_null_streams_scratch(q, torch_cuda):
    torch = torch_cuda
    g = torch.Generator(device="cuda").manual_seed(8)
    i8 = lambda o, k: torch.randint(-127, 128, (o, k), generator=g, device="cuda", dtype=torch.int8)
    sc = lambda o: torch.rand(o, generator=g, device="cuda") * 0.01

    def weight(o, k):
        w, s = i8(o, k), sc(o)
        return w, s, q.Tensor.i8(w, s)

    gate, up, down = weight(3584, 1024), weight(3584, 1024), weight(1024, 3584)
    n = 60
    xs = torch.randn(3, n, 1024, generator=g, device="cuda")
    want = torch.empty_like(xs)
    for t in range(3):
        for i in range(n):
            q.mlp_layer(want[t, i], xs[t, i], gate[2], up[2], down[2], w8a8=bool(i & 1))
            torch.cuda.synchronize()
    got = torch.zeros_like(xs)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    start = threading.Barrier(3)

    def work(t):
        torch.cuda.set_device(0)
        start.wait()
        for i in range(n):
            q.mlp_layer(got[t, i], xs[t, i], gate[2], up[2], down[2], w8a8=bool(i & 1), stream=side if t == 2 else None)

    ts = [threading.Thread(target=work, args=(t,)) for t in range(3)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    torch.cuda.synchronize()
    assert_bitwise(got.cpu().numpy(), want.cpu().numpy(), "mlp outputs of concurrent calls")
