"""Stage chains on products whose k is split across groups: the second kernel, which adds the
splits' sums, runs the chain (and the residual chain operands at every index) within the
carried product bound of tests/test_gpu_map.py."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from tests.helpers import from_dev, linear_bound, product_bound, rng, to_dev
from tests.test_gpu_map import FUSED, _check_fused
from tests.test_gpu_pipe import operands

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _split(R, xd, wd, m, n, **kw):
    """The product's k is split when its workspace is there."""
    from tessera_amd import abi
    a = R.linear_args(xd, wd, torch.empty((m, n), device="cuda"), **kw)
    return abi.load().tessera_hip_linear_workspace(C.byref(a)) > 0


# n % 4 == 0 takes four outputs a thread in the second kernel, other n one.
@pytest.mark.parametrize("m,n,k,x,w", [(16, 1024, 3072, "f32", "bf16"), (9, 1030, 4096, "bf16", "bf16"),
                                       (40, 1001, 8192, "f32", "e4m3"), (100, 130, 4096, "f32", "bf16"),
                                       (100, 128, 4096, "bf16", "bf16"), (129, 33, 4096, "bf16", "e4m3")])
@pytest.mark.parametrize("chain_i", range(len(FUSED)))
def test_chain_after_split_sums(m, n, k, x, w, chain_i):
    from tessera_amd import rules as R
    stages, nops, sum_at = FUSED[chain_i]
    r = rng(m + n + chain_i)
    xd, wd, sd, xf, wf, sums = operands(r, m, n, k, x, w)
    assert _split(R, xd, wd, m, n, w_scale=sd)
    ops = [r.standard_normal((m, n)).astype(np.float32) for _ in range(nops)]
    got = from_dev(R.linear(xd, wd, w_scale=sd, after=R.chain(stages, [to_dev(o, torch) for o in ops], sum_at=sum_at)))
    _check_fused(got, sums, linear_bound(xf, wf), stages, ops, sum_at)


@pytest.mark.parametrize("m,n,k,x,w", [(16, 200, 4096, "f32", "e4m3"), (24, 65, 4096, "bf16", "bf16"),
                                       (129, 33, 2048, "f32", "bf16"), (100, 64, 4096, "bf16", "e4m3")])
def test_chain_after_split_pair(m, n, k, x, w):
    """silu(gate) up of the splits' sums, then the chain."""
    from tessera_amd import abi, rules as R
    r = rng(m + n)
    xd, wd, sd, xf, wf, gu = operands(r, m, 2 * n, k, x, w)
    assert _split(R, xd, wd, m, n, w_scale=sd, stages=abi.TS_AFTER_SILU_MUL)
    op = r.standard_normal((m, n)).astype(np.float32)
    stages = ["mul", ("scale", 2.0), "tanh"]
    got = from_dev(R.linear(xd, wd, w_scale=sd, silu_mul=True, after=R.chain(stages, [to_dev(op, torch)])))
    g, u, b = gu[:, :n], gu[:, n:], linear_bound(xf, wf)
    inner = O.act("silu", g) * u
    _check_fused(got, inner, 1.1 * b[:, :n] * np.abs(u) + np.abs(g) * b[:, n:] + 1e-6, stages, [op], 0)


@pytest.mark.parametrize("m,n,k", [(16, 64, 4096), (100, 33, 4096)])
def test_chain_after_split_f32_weights(m, n, k):
    """f32 weights as two parts: the pair's sum, then the chain."""
    from tessera_amd import rules as R
    r = rng(m)
    w = (r.standard_normal((n, k)) * 0.05).astype(np.float32)
    x = r.standard_normal((m, k)).astype(np.float32)
    xd, packed = to_dev(x, torch), R.pack_f32(to_dev(w, torch))
    assert _split(R, xd, packed, m, n, w_form="f32_parts")
    op = r.standard_normal((m, n)).astype(np.float32)
    got = from_dev(R.linear(xd, packed, w_form="f32_parts", after=R.chain(["add", "silu"], [to_dev(op, torch)], sum_at=1)))
    _check_fused(got, O.product(x, w), product_bound(x, w, x_bits=16, parts=4, w_bits=16, lane=9), ["add", "silu"], [op], 1)


@pytest.mark.parametrize("form,n", [("int4_g32", 64), ("nvfp4", 65), ("q8_0", 130)])
def test_chain_after_split_block_forms(form, n):
    from tessera_amd import rules as R
    r = rng(n)
    m, k = 12, 8192
    packed = O.block_pack(form, (r.standard_normal((n, k)) * 0.05).astype(np.float32))
    w = O.block_unpack(form, packed, n * k).reshape(n, k)
    x = r.standard_normal((m, k)).astype(np.float32)
    xd, wd = to_dev(x, torch), torch.from_numpy(packed).cuda()
    assert _split(R, xd, wd, m, n, w_form=form)
    ops = [r.standard_normal((m, n)).astype(np.float32) for _ in range(2)]
    stages = ["add", "mul", "tanh"]
    got = from_dev(R.linear(xd, wd, w_form=form, rows=n, after=R.chain(stages, [to_dev(o, torch) for o in ops], sum_at=1)))
    bound = product_bound(x, w, x_bits=16, parts=2, lane=2 * k / O.block_size(form) + 8)
    _check_fused(got, O.product(x, w), bound, stages, ops, 1)
