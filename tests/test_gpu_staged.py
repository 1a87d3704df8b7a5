"""The register-staged tiles, which serve more than 64 rows at depths that are no multiple of
64 (and picked products at those depths or with a chain): every operand form, pairs, chains and
ragged last steps of k, on 64 x 64 and on 128 x 128 tiles, within the product bound."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import from_dev, linear_bound, product_bound, rng, to_dev
from tests.test_gpu_map import FUSED, _check_fused
from tests.test_gpu_pipe import operands

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

FORMS = [("f32", "bf16"), ("bf16", "bf16"), ("f32", "e4m3"), ("bf16", "e4m3")]
# The last two have 512 tiles of 128 x 128, from where on those are taken.
SIZES = [(100, 70, 72), (300, 130, 200), (65, 33, 8), (2050, 4000, 72), (1030, 7300, 136)]


def _operands(r, m, rows, k, x, w):
    O.set_threads(O.lib().or_threads_available())
    got = operands(r, m, rows, k, x, w)
    O.set_threads(1)
    return got


@pytest.mark.parametrize("x,w", FORMS)
@pytest.mark.parametrize("m,n,k", SIZES)
def test_staged_product(m, n, k, x, w):
    from tessera_amd import rules as R
    print(f"staged {x} {w} m={m} n={n} k={k}", flush=True)
    r = rng(m + n + k)
    xd, wd, sd, xf, wf, want = _operands(r, m, n, k, x, w)
    bound = linear_bound(xf, wf)
    got = from_dev(R.linear(xd, wd, w_scale=sd))
    assert np.all(np.abs(got.astype(np.float64) - want) <= bound)
    got16 = from_dev(R.linear(xd, wd, w_scale=sd, out_dtype=torch.bfloat16))
    assert np.array_equal(got16, O.bf16_widen(O.bf16_narrow(got)))
    res = r.standard_normal((m, n)).astype(np.float32)
    added = from_dev(R.linear(xd, wd, w_scale=sd, a0=to_dev(res, torch)))
    assert np.array_equal(added, got + res)


@pytest.mark.parametrize("x,w", FORMS)
@pytest.mark.parametrize("m,n,k", [(100, 70, 72), (300, 33, 200), (2050, 2050, 72)])
def test_staged_gate_up(m, n, k, x, w):
    from tessera_amd import rules as R
    r = rng(m + n + k + 1)
    xd, wd, sd, xf, wf, gu = _operands(r, m, 2 * n, k, x, w)
    g, u, b = gu[:, :n], gu[:, n:], linear_bound(xf, wf)
    got = from_dev(R.linear(xd, wd, w_scale=sd, silu_mul=True))
    assert np.all(np.abs(got.astype(np.float64) - O.act("silu", g) * u) <=
                  1.1 * b[:, :n] * np.abs(u) + np.abs(g) * b[:, n:] + 1e-5)


@pytest.mark.parametrize("xdt", ["f32", "bf16"])
@pytest.mark.parametrize("m,n,k", [(100, 70, 72), (300, 33, 200)])
def test_staged_f32_weights(m, n, k, xdt):
    from tessera_amd import rules as R
    r = rng(m + n)
    w = (r.standard_normal((n, k)) * 0.05).astype(np.float32)
    x = r.standard_normal((m, k)).astype(np.float32)
    if xdt == "bf16":
        x = O.bf16_round(x)
    xd = to_dev(x if xdt == "f32" else O.bf16_narrow(x), torch)
    got = from_dev(R.linear(xd, R.pack_f32(to_dev(w, torch)), w_form="f32_parts"))
    bound = product_bound(x, w, x_bits=16 if xdt == "f32" else None, parts=4, w_bits=16, lane=9)
    assert np.all(np.abs(got.astype(np.float64) - O.product(x, w)) <= bound)


@pytest.mark.parametrize("x,w", FORMS)
@pytest.mark.parametrize("m,n,k", [(100, 70, 72), (2050, 4000, 72)])
@pytest.mark.parametrize("chain_i", range(len(FUSED)))
def test_staged_chain(m, n, k, x, w, chain_i):
    from tessera_amd import rules as R
    stages, nops, sum_at = FUSED[chain_i]
    r = rng(m + n + chain_i)
    xd, wd, sd, xf, wf, sums = _operands(r, m, n, k, x, w)
    ops = [r.standard_normal((m, n)).astype(np.float32) for _ in range(nops)]
    got = from_dev(R.linear(xd, wd, w_scale=sd, after=R.chain(stages, [to_dev(o, torch) for o in ops], sum_at=sum_at)))
    _check_fused(got, sums, linear_bound(xf, wf), stages, ops, sum_at)


@pytest.mark.parametrize("x,w", FORMS)
@pytest.mark.parametrize("silu", [False, True])
def test_staged_picked(x, w, silu):
    """Expert products at such a depth: matrices of 0 to 300 rows, ids outside the set."""
    from tessera_amd import rules as R
    r = rng(3 + silu)
    count, n, k = 5, 70, 72
    used = 2 * n if silu else n
    ids = r.permutation(np.repeat([0, 1, 2, 4, 7], [1, 128, 129, 300, 6])).astype(np.uint32)
    xd, wd, sd, xf, wf, _ = operands(r, len(ids), count * used, k, x, w)
    got = from_dev(R.picked(xd, wd.view(count, used, k), to_dev(ids.astype(np.int32), torch), n=n, silu_mul=silu,
                            w_scale=None if sd is None else sd.view(count, used)))
    table = wf.reshape(count, used, k)
    assert np.all(got[ids >= count] == 0.0)
    for e in (0, 1, 2, 4):
        sel = ids == e
        full, b = xf[sel].astype(np.float64) @ table[e].T.astype(np.float64), linear_bound(xf[sel], table[e])
        if not silu:
            assert np.all(np.abs(got[sel] - full) <= b), f"matrix {e}"
            continue
        g, u = full[:, :n], full[:, n:]
        assert np.all(np.abs(got[sel] - g / (1 + np.exp(-g)) * u) <=
                      1.1 * b[:, :n] * np.abs(u) + np.abs(g) * b[:, n:] + 1e-5), f"matrix {e}"
