"""The routes that the single-layer ops choose by size, alignment and overlap, at the edges of each rule:
projection rows per wave (gemv_rows), the activation quantiser's registers, the weight quantiser's row
width, the DeltaNet step's float-aligned taps and its overlapping output.  Against the device twin, bit
for bit."""
import numpy as np
import pytest

from conftest import assert_bitwise, rng

pytestmark = pytest.mark.gpu


def p(a):
    return a.ctypes.data


def f32(a):
    return np.ascontiguousarray(a, dtype=np.float32)


# the rule's lines (2048, 4096 and 8192 rows; K 2048) from both sides, with row counts that leave a
# partial batch of 1, 4 or 8 rows, the smallest shape, and a ragged K below one pass of the wave
@pytest.mark.parametrize("out,inn", [(1, 16), (2048, 48), (2049, 2048), (2051, 2064), (4096, 4096), (4097, 2064),
                                     (8192, 1024), (8195, 1040)])
def test_projection_rows_per_wave(q, orc, torch_cuda, out, inn):
    torch = torch_cuda
    up = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    r = rng(out + 5 * inn)
    w = r.integers(-127, 128, size=(out, inn)).astype(np.int8)
    s, x = f32(r.uniform(1e-3, 1e-2, out)), f32(r.standard_normal(inn))
    guard = 8
    y, acc = torch.full((out + guard,), 7.0, device="cuda"), torch.full((out + guard,), 7, dtype=torch.int32, device="cuda")
    wd, sd = up(w), up(s)
    q.gemv_i8(y, wd, sd, up(x), out, inn)
    want = np.empty(out, np.float32)
    orc.lib().or_dev_gemv_i8(p(want), p(w), p(s), p(x), out, inn)
    got = y.cpu().numpy()
    assert_bitwise(got[:out], want, "W8A16")
    xq, sx = r.integers(-127, 128, size=inn).astype(np.int8), f32([0.01])
    q.gemv_i8_w8a8(y, acc, wd, sd, up(xq), up(sx), out, inn)
    wa = np.empty(out, np.int32)
    orc.lib().or_gemv_w8a8(p(want), p(wa), p(w), p(s), p(xq), float(sx[0]), out, inn)
    np.testing.assert_array_equal(acc.cpu().numpy()[:out], wa)
    assert_bitwise(y.cpu().numpy()[:out], want, "W8A8")
    assert (y[out:] == 7.0).all() and (acc[out:] == 7).all()


# 1024 threads with four registers each: one element, a wave's end, 4096 and one past it (read twice)
@pytest.mark.parametrize("n", [1, 65, 1025, 4095, 4096, 4097, 9000])
def test_quant_act_register_edges(q, orc, torch_cuda, n):
    torch = torch_cuda
    x = f32(rng(n).standard_normal(n))
    x[n - 1] = 9.0   # the maximum at the last element
    xq, sx = torch.full((n + 8,), 99, dtype=torch.int8, device="cuda"), torch.empty(1, device="cuda")
    q.quant_act(xq, sx, torch.from_numpy(x).cuda(), n)
    want, ws = np.empty(n, np.int8), np.empty(1, np.float32)
    orc.lib().or_quant_act(p(want), p(ws), p(x), n)
    np.testing.assert_array_equal(xq.cpu().numpy()[:n], want)
    assert sx.item() == ws[0] and (xq[n:] == 99).all()


# four registers a lane up to 1024 columns, sixteen up to 4096
@pytest.mark.parametrize("cols", [4, 252, 1020, 1024, 1028, 4096, 4100])
@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
def test_quant_rows_register_edges(q, orc, torch_cuda, cols, bf16):
    torch = torch_cuda
    rows = 5
    bits = (f32(rng(cols).standard_normal((rows, cols))).view(np.uint32) >> 16).astype(np.uint16)
    w = (bits.astype(np.uint32) << 16).view(np.float32)
    wd = torch.from_numpy(bits.view(np.int16)).cuda() if bf16 else torch.from_numpy(w).cuda()
    qd, sd = torch.full((rows * cols + 8,), 99, dtype=torch.int8, device="cuda"), torch.empty(rows, device="cuda")
    q.quant_rows(qd, sd, wd, rows, cols)
    want, ws = orc.quant_rows(w)
    np.testing.assert_array_equal(qd.cpu().numpy()[:rows * cols].reshape(rows, cols), want)
    np.testing.assert_array_equal(sd.cpu().numpy(), ws)
    assert (qd[rows * cols:] == 99).all()


@pytest.mark.parametrize("form", ["offset4", "out_in_qkv", "out_over_gates"])
def test_deltanet_step_forms(q, orc, torch_cuda, form):
    """Conv state and taps one float off a 16-byte boundary; an output that overlaps other heads' inputs."""
    torch = torch_cuda
    r = rng(len(form))
    h = {"qkv": f32(r.standard_normal(6144)), "z": f32(r.standard_normal(2048)), "b": f32(r.standard_normal(16)),
         "a": f32(r.standard_normal(16)), "cw": f32(r.standard_normal((6144, 4)) * 0.5),
         "al": f32(np.log(r.uniform(1, 16, 16))), "dt": f32(r.standard_normal(16)), "nw": f32(r.uniform(0.8, 1.2, 128)),
         "rec": f32(r.standard_normal((16, 128, 128)) * 0.05), "conv": f32(r.standard_normal((6144, 4)))}
    off = 1 if form == "offset4" else 0

    def up(a):
        buf = torch.empty(a.size + off, device="cuda")
        buf[off:].copy_(torch.from_numpy(a.reshape(-1)))
        return buf[off:]

    d = {k: up(v) for k, v in h.items()}
    out = torch.empty(2048, device="cuda")
    if form == "out_in_qkv":
        out = d["qkv"][100:100 + 2048]
    elif form == "out_over_gates":   # b, then a, inside the output
        out[500:516], out[900:916] = d["b"], d["a"]
        d["b"], d["a"] = out[500:516], out[900:916]
    ws = torch.empty(q.deltanet_step_workspace(), dtype=torch.uint8, device="cuda")
    q.deltanet_step(out, d["qkv"], d["z"], d["b"], d["a"], d["cw"], d["al"], d["dt"], d["nw"], d["rec"], d["conv"], ws)
    got = out.cpu().numpy()
    want = np.empty(2048, np.float32)
    orc.lib().or_deltanet_step(p(want), *[p(h[k]) for k in ("qkv", "z", "b", "a", "cw", "al", "dt", "nw", "rec", "conv")],
                               orc.ORDER_DEV)
    assert_bitwise(got, want, "out")
    assert_bitwise(d["rec"].cpu().numpy(), h["rec"].reshape(-1), "rec")
    assert_bitwise(d["conv"].cpu().numpy(), h["conv"].reshape(-1), "conv")
