"""The pipelined tiles over every operand form (f32 or bf16 rows, bf16 or e4m3 weights)
at the edges of their tiles, against the oracle's product within product_bound."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import bf16_bits_normal, from_dev, linear_bound, max_rel, rng, to_dev

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

FORMS = [("f32", "bf16"), ("f32", "e4m3"), ("bf16", "e4m3")]


def operands(r, m, rows, k, x, w):
    """(device operands and scale, the f32 values of x and w, the oracle's product)."""
    if x == "f32":
        xd = xf = r.standard_normal((m, k)).astype(np.float32)
    else:
        xd, xf = bf16_bits_normal(r, (m, k))
    if w == "bf16":
        wd, wf = bf16_bits_normal(r, (rows, k), 0.05)
        return to_dev(xd, torch), to_dev(wd, torch), None, xf, wf, O.product_bf16w(xf, wd)
    v = (r.standard_normal((rows, k)) * 0.05).astype(np.float32)
    s = O.bf16_narrow((np.abs(v).max(1) / 448.0).astype(np.float32))
    codes = O.e4m3_narrow(v / O.bf16_widen(s)[:, None])
    wf = O.e4m3_widen(codes) * O.bf16_widen(s)[:, None]
    return (to_dev(xd, torch), to_dev(codes, torch), to_dev(s, torch), xf, wf, O.product_e4m3w(xf, codes, s))


@pytest.mark.parametrize("x,w", FORMS)
@pytest.mark.parametrize("m,n,k", [(65, 64, 64), (129, 190, 128), (200, 33, 1024), (1000, 4100, 192),
                                   (1025, 4096, 64)])
def test_pipe_edges(m, n, k, x, w):
    """One k step and several, ragged rows and columns, 64 x 64 tiles (the first three) and
    128 x 128 ones; with a residual, to f32 and to bf16."""
    from tessera_amd import rules as R
    print(f"pipe {x} {w} m={m} n={n} k={k}", flush=True)
    r = rng(m + n + k)
    O.set_threads(O.lib().or_threads_available())
    xd, wd, sd, xf, wf, want = operands(r, m, n, k, x, w)
    O.set_threads(1)
    res = r.standard_normal((m, n)).astype(np.float32)
    got = from_dev(R.linear(xd, wd, w_scale=sd, a0=to_dev(res, torch)))
    bound = linear_bound(xf, wf)
    assert np.all(np.abs(got.astype(np.float64) - (want + res)) <= bound + 1e-6)
    got32 = from_dev(R.linear(xd, wd, w_scale=sd))
    assert np.all(np.abs(got32.astype(np.float64) - want) <= bound)
    # The bf16 output (through LDS) is the f32 one rounded once, element for element.
    got16 = from_dev(R.linear(xd, wd, w_scale=sd, out_dtype=torch.bfloat16))
    assert np.array_equal(got16, O.bf16_widen(O.bf16_narrow(got32)))


@pytest.mark.parametrize("x,w", FORMS + [("bf16", "bf16")])
@pytest.mark.parametrize("m,n,most", [(66, 30, 12), (1030, 4100, 6)])
def test_pipe_step_counts(m, n, most, x, w):
    """Every count of k steps around the ring: none that refills a stage, some, whole turns of
    the ring and what is left behind them, on 64 x 64 and 128-wide tiles."""
    from tessera_amd import rules as R
    r = rng(m + most)
    O.set_threads(O.lib().or_threads_available())
    for steps in range(1, most + 1):
        xd, wd, sd, xf, wf, want = operands(r, m, n, 64 * steps, x, w)
        got = from_dev(R.tiled(xd, wd, w_scale=sd))
        assert np.all(np.abs(got.astype(np.float64) - want) <= linear_bound(xf, wf)), f"{steps} steps"
    O.set_threads(1)


@pytest.mark.parametrize("x,w", FORMS)
@pytest.mark.parametrize("m,n,k", [(70, 40, 128), (1030, 2050, 64)])
def test_pipe_gate_up(m, n, k, x, w):
    """Gate/up pairs on 64 x 64 and on 128 x 128 tiles: silu(g) u, first-order error of the
    pair's bounds."""
    from tessera_amd import rules as R
    r = rng(m + n + k + 1)
    O.set_threads(O.lib().or_threads_available())
    xd, wd, sd, xf, wf, gu = operands(r, m, 2 * n, k, x, w)
    O.set_threads(1)
    g, u = gu[:, :n], gu[:, n:]
    want = O.act("silu", g) * u
    got = from_dev(R.linear(xd, wd, w_scale=sd, silu_mul=True))
    b = linear_bound(xf, wf)
    assert np.all(np.abs(got.astype(np.float64) - want) <= 1.1 * b[:, :n] * np.abs(u) + np.abs(g) * b[:, n:] + 1e-5)


@pytest.mark.parametrize("x,w", FORMS + [("bf16", "bf16")])
@pytest.mark.parametrize("silu,counts", [
    (False, ((0, 1), (1, 128), (2, 129), (4, 300), (5, 17), (9, 6))),
    (True, ((0, 1), (1, 128), (2, 129), (4, 300), (5, 17), (9, 6))),
    (False, ((0, 1), (1, 31), (3, 32), (4, 20), (9, 2))),
    (True, ((0, 33), (2, 16), (5, 17), (8, 1)))])
def test_pipe_picked(x, w, silu, counts):
    """Expert products on the same tiles: matrices of 0, 1, 128, 129 and more rows, and on 32-row
    tiles (16 rows a matrix on average) of 0 to 33; ids outside the set."""
    from tessera_amd import rules as R
    r = rng(17 + silu)
    count, n, k, offset = 6, 72, 128, 3
    used = 2 * n if silu else n
    stride = used + 5
    ids = np.concatenate([np.full(c, e) for e, c in counts])
    ids = r.permutation(ids).astype(np.uint32)
    rows = len(ids)
    xd, wd, sd, xf, wf, _ = operands(r, rows, count * stride, k, x, w)
    shape = (count, stride, k)
    got = from_dev(R.picked(xd, wd.view(shape), to_dev(ids.astype(np.int32), torch), n=n, offset=offset, silu_mul=silu,
                            w_scale=None if sd is None else sd.view(count, stride)))
    table = wf.reshape(shape)
    for e in range(10):
        sel = ids == e
        if e >= count:
            assert np.all(got[sel] == 0.0)
            continue
        if not sel.any():
            continue
        we = table[e, offset:offset + used]
        full, b = xf[sel].astype(np.float64) @ we.T.astype(np.float64), linear_bound(xf[sel], we)
        if not silu:
            assert np.all(np.abs(got[sel] - full) <= b), f"matrix {e}"
            continue
        g, u = full[:, :n], full[:, n:]
        want = g / (1 + np.exp(-g)) * u
        assert np.all(np.abs(got[sel] - want) <= 1.1 * b[:, :n] * np.abs(u) + np.abs(g) * b[:, n:] + 1e-5), f"matrix {e}"


@pytest.mark.parametrize("x,w", FORMS + [("bf16", "bf16")])
@pytest.mark.parametrize("silu,n,k", [(False, 136, 192), (True, 136, 192), (False, 8070, 128), (True, 4100, 128)])
def test_pipe_picked_skewed(x, w, silu, n, k):
    """Few rows a matrix on average, and some matrices with many: 32-row tiles, with many columns
    128-row ones for the matrices of more than 64 rows."""
    from tessera_amd import rules as R
    r = rng(23 + silu)
    count = 40
    rows_of = {0: 161, 3: 128, 5: 65, 9: 64, 10: 33, 11: 32, 39: 1, 45: 50}
    used = 2 * n if silu else n
    ids = r.permutation(np.repeat(list(rows_of), list(rows_of.values()))).astype(np.uint32)
    xd, wd, sd, xf, wf, _ = operands(r, len(ids), count * used, k, x, w)
    got = from_dev(R.picked(xd, wd.view(count, used, k), to_dev(ids.astype(np.int32), torch), n=n, silu_mul=silu,
                            w_scale=None if sd is None else sd.view(count, used)))
    table = wf.reshape(count, used, k)
    assert np.all(got[ids >= count] == 0.0)
    for e in (e for e in rows_of if e < count):
        sel = ids == e
        full, b = xf[sel].astype(np.float64) @ table[e].T.astype(np.float64), linear_bound(xf[sel], table[e])
        if not silu:
            assert np.all(np.abs(got[sel] - full) <= b), f"matrix {e}"
            continue
        g, u = full[:, :n], full[:, n:]
        assert np.all(np.abs(got[sel] - g / (1 + np.exp(-g)) * u) <=
                      1.1 * b[:, :n] * np.abs(u) + np.abs(g) * b[:, n:] + 1e-5), f"matrix {e}"


@pytest.mark.parametrize("x,w", FORMS + [("bf16", "bf16")])
@pytest.mark.parametrize("m,n,k,pair", [(65, 64, 4096, False), (100, 130, 4160, False), (129, 33, 2048, True),
                                        (700, 700, 6144, False)])
def test_pipe_split_k(m, n, k, pair, x, w):
    """Few tiles and a deep k: split across groups (64 x 64 and 128 x 128 tiles, ragged columns,
    a step count the splits do not divide), the sums finished by the second kernel; the same
    product without the workspace runs unsplit."""
    import ctypes as C

    from tessera_amd import abi, rules as R
    if w == "e4m3":
        k = k // 128 * 128
    r = rng(m + n)
    O.set_threads(O.lib().or_threads_available())
    xd, wd, sd, xf, wf, full = operands(r, m, 2 * n if pair else n, k, x, w)
    O.set_threads(1)
    bound = linear_bound(xf, wf)
    if pair:
        g, u, bg, bu = full[:, :n], full[:, n:], bound[:, :n], bound[:, n:]
        want = O.act("silu", g) * u
        bound = 1.1 * bg * np.abs(u) + np.abs(g) * bu + 1e-5
    else:
        want = full
    out = torch.empty((m, n), device="cuda")
    a = R.linear_args(xd, wd, out, w_scale=sd, stages=abi.TS_AFTER_SILU_MUL if pair else 0)
    assert abi.load().tessera_hip_linear_workspace(C.byref(a)) > 0
    got = from_dev(R.linear(xd, wd, w_scale=sd, silu_mul=pair))
    assert np.all(np.abs(got.astype(np.float64) - want) <= bound)
    res = r.standard_normal((m, n)).astype(np.float32)
    added = from_dev(R.linear(xd, wd, w_scale=sd, silu_mul=pair, a0=to_dev(res, torch)))
    assert np.array_equal(added, got + res)
    got16 = from_dev(R.linear(xd, wd, w_scale=sd, silu_mul=pair, out_dtype=torch.bfloat16))
    assert np.array_equal(got16, O.bf16_widen(O.bf16_narrow(got)))
    abi.call("tessera_hip_linear", C.byref(a), C.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert np.all(np.abs(from_dev(out).astype(np.float64) - want) <= bound)
