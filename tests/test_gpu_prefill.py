"""Prompts run in groups (qh_prefill.hip) leave what feeding them token by token leaves, bit for
bit: the recurrent, conv and KV state, the next token and its logits.  Lengths at the edges of the
MFMA tiles (16 and 32 tokens) and of the scan's blocks (8), of one group (512, then two halves), of
the positions the grouped attention covers (2048), and prompts that start inside a tile.  The prompt's last token always runs on the executor, so n
tokens take the grouped path for n - 1 of them."""
import threading

import numpy as np
import pytest

from conftest import assert_bitwise, rng
from test_gpu_engine import d2h

pytestmark = pytest.mark.gpu


def _state(e, n, ctx):
    return [d2h(e.device_ptr(1), (18, 16, 128, 128)), d2h(e.device_ptr(2), (18, 6144, 4)),
            d2h(e.device_ptr(3), (6, ctx, 512))[:, :n], d2h(e.device_ptr(4), (6, ctx, 512))[:, :n]]


def _check(q, e, parts, ctx):
    """The prompts `parts` one after another, fed whole and token by token."""
    n = sum(len(p) for p in parts)
    e.reset()
    for p in parts:
        for t in p:
            am, _ = e.decode_token(t)
    want, lw = _state(e, n, ctx), e.decode_token(7, want_logits=True)[1]
    e.reset()
    for p in parts:
        assert e.generate(p, 0) == []
    assert e.pos == n and e.last_argmax == am
    got, lg = _state(e, n, ctx), e.decode_token(7, want_logits=True)[1]
    for a, b, what in zip(got, want, ("recurrent state", "conv state", "k cache", "v cache")):
        assert_bitwise(a, b, f"{what}, prompts {[len(p) for p in parts]}")
    assert_bitwise(lg, lw, "next logits")


@pytest.mark.parametrize("mode", [0, 1], ids=["w8a16", "w8a8"])
@pytest.mark.parametrize("exec_kind", ["graph", "persistent"])
def test_prompt_in_groups_equals_token_by_token(q, blob, torch_cuda, mode, exec_kind):
    ctx = 600
    e = q.Engine(blob, max_ctx=ctx, mode=mode)
    try:
        e.set_exec(q.EXEC_GRAPH if exec_kind == "graph" else q.EXEC_PERSISTENT)
        r = rng(77 + mode)
        ids = lambda n: r.integers(0, q.VOCAB, size=n).astype(np.int32).tolist()
        lens = [[9], [14], [16], [17], [18], [33], [34], [66], [3, 20], [21, 40, 2, 15]]
        if exec_kind == "persistent":
            lens += [[129], [513], [514], [30, 530]]
        for ls in lens:
            _check(q, e, [ids(n) for n in ls], ctx)
    finally:
        e.close()


@pytest.mark.parametrize("mode", [0, 1], ids=["w8a16", "w8a8"])
def test_prompt_past_the_short_contexts(q, blob, torch_cuda, mode):
    """A prompt that ends past 2048 positions: the groups stop there."""
    ctx = 2080
    e = q.Engine(blob, max_ctx=ctx, mode=mode)
    try:
        e.set_exec(q.EXEC_PERSISTENT)
        ids = rng(9).integers(0, q.VOCAB, size=2061).astype(np.int32).tolist()
        _check(q, e, [ids], ctx)
    finally:
        e.close()


# the shortest groups that the rule takes (prefill_min) at the start of a context and late in one
@pytest.mark.parametrize("mode,exec_kind,first,late", [(0, "graph", 4, 5), (1, "graph", 3, 4), (0, "persistent", 7, 7),
                                                       (1, "persistent", 5, 6)])
def test_shortest_groups(q, blob, torch_cuda, mode, exec_kind, first, late):
    """Both sides of the rule's line, from an empty state and after other prompts (a group shorter than
    the four conv taps keeps an old column, and the scan's only block is partial)."""
    ctx = 1900
    e = q.Engine(blob, max_ctx=ctx, mode=mode)
    try:
        e.set_exec(q.EXEC_GRAPH if exec_kind == "graph" else q.EXEC_PERSISTENT)
        r = rng(55 + mode)
        ids = lambda n: r.integers(0, q.VOCAB, size=n).astype(np.int32).tolist()
        for ls in ([first + 1], [first], [2, first + 1, first + 2], [first + 1, 1, first, first + 1],
                   [1842, late + 1, late, first + 1]):
            _check(q, e, [ids(n) for n in ls], ctx)
    finally:
        e.close()


def test_generation_after_a_grouped_prompt(q, blob, torch_cuda):
    """Greedy ids, eos and the position after a grouped prompt equal those of a host loop."""
    ctx = 128
    e = q.Engine(blob, max_ctx=ctx, mode=q.MODE_W8A8)
    try:
        ids = rng(3).integers(0, q.VOCAB, size=70).astype(np.int32).tolist()
        cur = None
        for t in ids:
            cur, _ = e.decode_token(t)
        want = []
        for _ in range(12):
            want.append(cur)
            cur, _ = e.decode_token(cur)
        for ex in (q.EXEC_GRAPH, q.EXEC_PERSISTENT):
            e.set_exec(ex)
            e.reset()
            assert e.generate(ids, 12) == want and e.pos == 82
            e.reset()
            first = want.index(want[5])
            assert e.generate(ids, 12, eos=want[5]) == want[:first] and e.pos == 70 + first
    finally:
        e.close()


@pytest.mark.parametrize("exec_kind", ["graph", "persistent"])
@pytest.mark.parametrize("step", ["prepare", "launch"])
def test_setup_failure_around_the_groups(q, blob, torch_cuda, monkeypatch, exec_kind, step):
    """An executor whose set-up fails (forced from the host: QH_FAIL_SETUP) while a prompt runs in
    groups.  The program or graph is made first, so that its failure leaves position and state as they
    were and the same call then succeeds; a failure after the groups leaves an engine that refuses to
    decode until its reset.  Both end with what an engine without the failure gives."""
    monkeypatch.setenv("QH_FAIL_SETUP", step)
    e = q.Engine(blob, max_ctx=64)
    monkeypatch.delenv("QH_FAIL_SETUP")
    f = q.Engine(blob, max_ctx=64)
    try:
        for eng in (e, f):
            eng.set_exec(q.EXEC_GRAPH if exec_kind == "graph" else q.EXEC_PERSISTENT)
        ids = rng(21).integers(0, q.VOCAB, size=20).astype(np.int32).tolist()
        want, lw = f.generate(ids, 4), f.decode_token(7, want_logits=True)[1]
        with pytest.raises(q.QHError) as ex:
            e.generate(ids, 4)
        assert ex.value.status == q.QH_ENOMEM
        if step == "prepare":
            assert e.pos == 0
            assert all(not a.any() for a in _state(e, 64, 64)), "state touched by the failed call"
        else:
            for call in (lambda: e.decode_token(7), lambda: e.generate(ids, 4)):
                with pytest.raises(q.QHError) as ex:
                    call()
                assert ex.value.status == q.QH_ESTATE
            e.reset()
        assert e.generate(ids, 4) == want and e.pos == 24
        assert_bitwise(e.decode_token(7, want_logits=True)[1], lw, "next logits")
    finally:
        e.close()
        f.close()


def test_two_engines_prompt_in_two_threads(q, blob, torch_cuda):
    """A short and a long prompt, whose attention launches need 4 and 68 KiB of LDS, in two threads at
    once: each engine's state is what it is alone (the kernel's LDS limit belongs to the process)."""
    r = rng(31)
    prompts = [r.integers(0, q.VOCAB, size=n).astype(np.int32).tolist() for n in (40, 950)]
    es = [q.Engine(blob, max_ctx=len(p) + 4, mode=q.MODE_W8A8) for p in prompts]
    try:
        want = []
        for e, p in zip(es, prompts):
            e.set_exec(q.EXEC_GRAPH)
            gen = e.generate(p, 2)
            want.append((gen, _state(e, len(p), len(p) + 4)))
        got = [[], []]
        start = threading.Barrier(2)

        def work(i, passes):
            start.wait()
            for _ in range(passes):
                es[i].reset()
                got[i].append(es[i].generate(prompts[i], 2))

        ts = [threading.Thread(target=work, args=a) for a in ((0, 12), (1, 4))]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        for i, (e, p) in enumerate(zip(es, prompts)):
            assert got[i] and all(g == want[i][0] for g in got[i])
            for a, b, what in zip(_state(e, len(p), len(p) + 4), want[i][1], ("recurrent state", "conv state", "k cache", "v cache")):
                assert_bitwise(a, b, f"{what}, prompt of {len(p)}")
    finally:
        for e in es:
            e.close()
