"""bf16 and e4m3 weights streamed at 5..64 rows (whole units of k): the edges of the row
tiles, of the 32 weight rows a wave, of a last step that holds fewer units than slices, and
split k, with every operand form and epilogue, within product_bound of the oracle."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from tests.helpers import from_dev, linear_bound, rng, to_dev
from tests.test_gpu_pipe import operands

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

FORMS = [("f32", "bf16"), ("bf16", "bf16"), ("f32", "e4m3"), ("bf16", "e4m3")]


@pytest.mark.parametrize("x,w", FORMS)
@pytest.mark.parametrize("m,n,k", [(5, 33, 128), (16, 130, 384), (17, 31, 640), (33, 200, 1152), (48, 1000, 256),
                                   (64, 65, 4096), (9, 2500, 1024)])
def test_stream_edges(m, n, k, x, w):
    from tessera_amd import rules as R
    print(f"stream {x} {w} m={m} n={n} k={k}", flush=True)
    r = rng(m + n + k)
    xd, wd, sd, xf, wf, want = operands(r, m, n, k, x, w)
    bound = linear_bound(xf, wf)
    res = r.standard_normal((m, n)).astype(np.float32)
    got = from_dev(R.linear(xd, wd, w_scale=sd, a0=to_dev(res, torch)))
    assert np.all(np.abs(got.astype(np.float64) - (want + res)) <= bound + 1e-6)
    got32 = from_dev(R.linear(xd, wd, w_scale=sd))
    got16 = from_dev(R.linear(xd, wd, w_scale=sd, out_dtype=torch.bfloat16))
    assert np.array_equal(got16, O.bf16_widen(O.bf16_narrow(got32)))


@pytest.mark.parametrize("x,w", FORMS)
@pytest.mark.parametrize("m,n,k", [(6, 50, 192), (20, 70, 1024), (64, 130, 2176)])
def test_stream_gate_up(m, n, k, x, w):
    from tessera_amd import rules as R
    if w == "e4m3":
        k = k // 128 * 128
    r = rng(m + n)
    xd, wd, sd, xf, wf, gu = operands(r, m, 2 * n, k, x, w)
    g, u = gu[:, :n], gu[:, n:]
    want = O.act("silu", g) * u
    b = linear_bound(xf, wf)
    got = from_dev(R.linear(xd, wd, w_scale=sd, silu_mul=True))
    assert np.all(np.abs(got.astype(np.float64) - want) <= 1.1 * b[:, :n] * np.abs(u) + np.abs(g) * b[:, n:] + 1e-5)


@pytest.mark.parametrize("w", ["bf16", "e4m3"])
@pytest.mark.parametrize("m,n,k", [(5, 40, 128), (7, 33, 384), (16, 100, 4096), (11, 20000, 1024)])
def test_stream_norm(m, n, k, w):
    """RmsNorm before the product, one group and several along k and the columns (the first
    two have a last step of fewer units)."""
    from tessera_amd import rules as R
    r = rng(m * n)
    xd, wd, sd, xf, wf, _ = operands(r, m, n, k, "f32", w)
    g = (1 + 0.1 * r.standard_normal(k)).astype(np.float32)
    xn = O.rms_norm(xf * 3, g, 1e-6)
    want = xn.astype(np.float64) @ wf.T.astype(np.float64)
    got = from_dev(R.linear(xd * 3, wd, w_scale=sd, gain=to_dev(g, torch), eps=1e-6))
    assert np.all(np.abs(got - want) <= 2 * linear_bound(xn, wf))


def test_stream_without_workspace():
    """No workspace: the same product with k unsplit, the norm's sums included."""
    from tessera_amd import abi, rules as R
    r = rng(8)
    m, n, k = 12, 256, 4096
    xd, wd, _, xf, wf, _ = operands(r, m, n, k, "f32", "bf16")
    g = np.ones(k, np.float32)
    gd, out = to_dev(g, torch), torch.empty((m, n), device="cuda")
    a = R.linear_args(xd, wd, out, gain=gd, stages=abi.TS_BEFORE_RMS_NORM)
    assert abi.load().tessera_hip_linear_workspace(C.byref(a)) > 0  # k is split where it may be
    abi.call("tessera_hip_linear", C.byref(a), C.c_void_p(torch.cuda.current_stream().cuda_stream))
    xn = O.rms_norm(xf, g, 1e-6)
    assert np.all(np.abs(from_dev(out) - xn.astype(np.float64) @ wf.T) <= 2 * linear_bound(xn, wf))


@pytest.mark.parametrize("m,n,k,norm,silu", [(12, 256, 4096, True, False), (12, 130, 4096, True, True),
                                             (40, 1000, 8192, False, False)])
def test_stream_smaller_workspace(m, n, k, norm, silu):
    """A workspace of fewer splits than the query names holds that many: the same product, and
    nothing behind it is written."""
    from tessera_amd import abi, rules as R
    r = rng(m + n)
    xd, wd, _, xf, wf, _ = operands(r, m, 2 * n if silu else n, k, "f32", "bf16")
    gd = torch.ones(k, device="cuda") if norm else None
    xn = O.rms_norm(xf, np.ones(k, np.float32), 1e-6) if norm else xf
    want, bound = xn.astype(np.float64) @ wf.T.astype(np.float64), 2 * linear_bound(xn, wf)
    if silu:
        g, u, bg, bu = want[:, :n], want[:, n:], bound[:, :n], bound[:, n:]
        want, bound = g / (1 + np.exp(-g)) * u, 1.1 * bg * np.abs(u) + np.abs(g) * bu + 1e-5
    out = torch.empty((m, n), device="cuda")
    stages = (abi.TS_BEFORE_RMS_NORM if norm else 0) | (abi.TS_AFTER_SILU_MUL if silu else 0)
    a = R.linear_args(xd, wd, out, gain=gd, stages=stages)
    need = abi.load().tessera_hip_linear_workspace(C.byref(a))
    one = (m * n * (2 if silu else 1) + (m if norm else 0)) * 4
    splits = need // one
    assert splits >= 3 and need == splits * one
    for size in (need, need - 1, 2 * one, 2 * one - 1, one, 1):
        buf = torch.full((need + 64,), 0xA5, dtype=torch.uint8, device="cuda")
        out.zero_()
        a.workspace, a.workspace_bytes = buf.data_ptr(), size
        abi.call("tessera_hip_linear", C.byref(a), R._stream())
        assert np.all(np.abs(from_dev(out) - want) <= bound), f"{size} of {need} bytes"
        assert bool((buf[size:] == 0xA5).all())


@pytest.mark.parametrize("x,w", FORMS)
@pytest.mark.parametrize("m,n,k,silu", [(16, 70, 4072, False), (40, 130, 2056, True), (64, 200, 1032, False)])
def test_lanes_smaller_workspace(m, n, k, silu, x, w):
    """The kernel for any k (here in no whole units), split as often as its workspace holds: the
    same product, and nothing behind the workspace is written."""
    from tessera_amd import abi, rules as R
    r = rng(m + n)
    xd, wd, sd, xf, wf, want = operands(r, m, 2 * n if silu else n, k, x, w)
    bound = linear_bound(xf, wf)
    if silu:
        g, u, bg, bu = want[:, :n], want[:, n:], bound[:, :n], bound[:, n:]
        want, bound = O.act("silu", g) * u, 1.1 * bg * np.abs(u) + np.abs(g) * bu + 1e-5
    out = torch.empty((m, n), device="cuda")
    a = R.linear_args(xd, wd, out, w_scale=sd, stages=abi.TS_AFTER_SILU_MUL if silu else 0)
    need, one = abi.load().tessera_hip_linear_workspace(C.byref(a)), m * n * (2 if silu else 1) * 4
    assert need >= 3 * one and need % one == 0
    for size in (need, need - 1, 2 * one, 2 * one - 1, 0):
        buf = torch.full((need + 64,), 0xA5, dtype=torch.uint8, device="cuda")
        out.zero_()
        a.workspace, a.workspace_bytes = buf.data_ptr() if size else None, size
        abi.call("tessera_hip_linear", C.byref(a), R._stream())
        assert np.all(np.abs(from_dev(out) - want) <= bound), f"{size} of {need} bytes"
        assert bool((buf[size:] == 0xA5).all())
