"""Block-form weights at 5..64 rows: every form over the edges of the kernel's tiles (row
tiles of 16, 32 weight rows a wave, units of 128 codes, an odd last unit, split k), against
the CPU product over the decoded weights within the block path's bound (two f32 roundings a
block, as tests/test_gpu_blocks.py derives it)."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from tests.helpers import from_dev, product_bound, rng, to_dev

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

FORMS = list(O.BLOCK_FORMS)


def _packed(r, form, n, k):
    wb = O.block_pack(form, (r.standard_normal((n, k)) * 0.05).astype(np.float32))
    return torch.from_numpy(wb).cuda(), O.block_unpack(form, wb, n * k).reshape(n, k)


def _rows(r, m, k, bf16):
    x = r.standard_normal((m, k)).astype(np.float32)
    if bf16:
        b = O.bf16_narrow(x)
        return to_dev(b, torch), O.bf16_widen(b)
    return to_dev(x, torch), x


def _bound(form, x, w, bf16, lane=0):
    lane += 2 * w.shape[1] / O.block_size(form) + 8
    return product_bound(x, w, lane=lane) if bf16 else product_bound(x, w, x_bits=16, parts=2, lane=lane)


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("m,n,k,bf16", [(5, 37, 512, False), (16, 130, 1536, True), (17, 33, 1024, False),
                                        (33, 100, 2560, True), (48, 260, 512, False), (64, 40, 4096, False),
                                        (64, 65, 8192, True)])
def test_block_lanes(form, m, n, k, bf16):
    from tessera_amd import rules as R
    print(f"block lanes {form} m={m} n={n} k={k} bf16={bf16}", flush=True)
    r = rng(m + n + k)
    wd, w = _packed(r, form, n, k)
    xd, x = _rows(r, m, k, bf16)
    want = O.product(x, w)
    res = r.standard_normal((m, n)).astype(np.float32)
    got = from_dev(R.linear(xd, wd, w_form=form, rows=n, a0=to_dev(res, torch)))
    assert np.all(np.abs(got.astype(np.float64) - (want + res)) <= _bound(form, x, w, bf16, 1) + 1e-6)
    got32 = from_dev(R.linear(xd, wd, w_form=form, rows=n))
    got16 = from_dev(R.linear(xd, wd, w_form=form, rows=n, out_dtype=torch.bfloat16))
    assert np.array_equal(got16, O.bf16_widen(O.bf16_narrow(got32)))  # one rounding of the same sums


@pytest.mark.parametrize("form", ["int4_g32", "q4_0", "mxfp8", "nvfp4", "int4_g128"])
@pytest.mark.parametrize("k", [128, 384, 640])
def test_block_lanes_odd_units(form, k):
    """One unit of 128 codes, and an odd count: the last step holds one unit of two."""
    from tessera_amd import rules as R
    if k % (4 * O.block_size(form)):
        k = 512
    r = rng(k)
    wd, w = _packed(r, form, 50, k)
    xd, x = _rows(r, 9, k, False)
    got = from_dev(R.linear(xd, wd, w_form=form, rows=50))
    assert np.all(np.abs(got - O.product(x, w)) <= _bound(form, x, w, False))


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("m,n,k", [(6, 70, 1024), (40, 130, 4096)])
def test_block_lanes_gate_up(form, m, n, k):
    from tessera_amd import rules as R
    r = rng(m + n)
    wd, w = _packed(r, form, 2 * n, k)
    xd, x = _rows(r, m, k, False)
    gu = O.product(x, w)
    g, u = gu[:, :n], gu[:, n:]
    want = O.act("silu", g) * u
    b = _bound(form, x, w, False)
    got = from_dev(R.linear(xd, wd, w_form=form, rows=2 * n, silu_mul=True))
    assert np.all(np.abs(got.astype(np.float64) - want) <= 1.1 * b[:, :n] * np.abs(u) + np.abs(g) * b[:, n:] + 1e-5)


def test_block_lanes_without_workspace():
    """A caller that passes no workspace gets the same product, its k unsplit."""
    from tessera_amd import abi, rules as R
    r = rng(3)
    m, n, k, form = 16, 64, 8192, "int4_g32"
    wd, w = _packed(r, form, n, k)
    xd, x = _rows(r, m, k, False)
    out = torch.empty((m, n), device="cuda")
    a = R.linear_args(xd, wd, out, w_form=form)
    assert abi.load().tessera_hip_linear_workspace(C.byref(a)) > 0  # k is split where it may be
    abi.call("tessera_hip_linear", C.byref(a), C.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert np.all(np.abs(from_dev(out) - O.product(x, w)) <= _bound(form, x, w, False))
    split = from_dev(R.linear(xd, wd, w_form=form, rows=n))
    assert np.all(np.abs(split - O.product(x, w)) <= _bound(form, x, w, False))
