"""RmsNorm with a row in registers and the group-per-row q/k norm + RoPE + append, at the
edges of their ranges, against the oracle."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import bf16_bits_normal, from_dev, rng, to_dev

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width", [1, 64, 65, 512, 513, 1024, 1030, 2049, 4096, 4097])
def test_rms_norm_rows(width):
    """The edges of each count of values a lane holds, and the looped form past them; a row
    start that is not 16-byte aligned, and in place."""
    from tessera_amd import rules as R
    r = rng(width)
    x = r.standard_normal((5, width)).astype(np.float32)
    g = (1 + 0.1 * r.standard_normal(width)).astype(np.float32)
    want = O.rms_norm(x, g, 1e-6)
    xd, gd = to_dev(x, torch), to_dev(g, torch)
    np.testing.assert_allclose(from_dev(R.rms_norm(xd, gd, 1e-6)), want, rtol=1e-5, atol=1e-6)
    buf = torch.empty(5 * width + 1, device="cuda")
    odd = buf[1:].view(5, width)
    odd.copy_(xd)
    np.testing.assert_allclose(from_dev(R.rms_norm(odd, gd, 1e-6)), want, rtol=1e-5, atol=1e-6)
    R.rms_norm(xd, gd, 1e-6, out=xd)
    np.testing.assert_allclose(from_dev(xd), want, rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("heads,kvh", [(1, 1), (16, 8), (7, 7)])
def test_qk_norm_rope_append_many_rows(heads, kvh):
    """From 256 rows on a group takes a row; the same bits as the wave-per-head form gives for
    the same rows in two halves, positions past the slot append nothing."""
    from tessera_amd import rules as R
    r = rng(heads)
    rows, keys = 300, 290
    qkv = to_dev(r.standard_normal((rows, (heads + 2 * kvh) * 128)).astype(np.float32), torch)
    qg, kg = (to_dev((1 + 0.02 * r.standard_normal(128)).astype(np.float32), torch) for _ in range(2))
    pos = to_dev(r.permutation(rows).astype(np.uint32), torch, torch.int32)
    slots = torch.zeros(rows, dtype=torch.int32, device="cuda")

    def call(parts):
        q = torch.full((rows, heads, 128), 7.0, device="cuda")
        k = torch.zeros((keys, kvh, 128), dtype=torch.bfloat16, device="cuda")
        v = torch.zeros_like(k)
        for lo, hi in parts:
            R.qk_norm_rope_append(qkv[lo:hi], qg, kg, q[lo:hi], k, v, slots[lo:hi], pos[lo:hi], heads=heads,
                                  kv_heads=kvh, keys=keys, eps=1e-6, theta=1e6)
        return q, k, v

    for a, b in zip(call([(0, rows)]), call([(0, 150), (150, rows)])):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


@pytest.mark.parametrize("heads,kvh,rows", [(12, 2, 512), (7, 7, 391), (10, 2, 600), (8, 4, 1200)])
def test_qk_norm_rope_append_group_a_row(heads, kvh, rows):
    """Around the rule of the two forms (16 heads a row, 8192 heads in all): every row's bits are
    those it has among few rows, which take a wave a head."""
    from tessera_amd import rules as R
    r = rng(rows)
    qkv = to_dev(r.standard_normal((rows, (heads + 2 * kvh) * 128)).astype(np.float32), torch)
    qg, kg = (to_dev((1 + 0.02 * r.standard_normal(128)).astype(np.float32), torch) for _ in range(2))
    pos = to_dev(r.permutation(rows).astype(np.uint32), torch, torch.int32)
    slots = torch.zeros(rows, dtype=torch.int32, device="cuda")

    def call(step):
        q = torch.full((rows, heads, 128), 7.0, device="cuda")
        k = torch.zeros((rows, kvh, 128), dtype=torch.bfloat16, device="cuda")
        v = torch.zeros_like(k)
        for lo in range(0, rows, step):
            s = slice(lo, min(lo + step, rows))
            R.qk_norm_rope_append(qkv[s], qg, kg, q[s], k, v, slots[s], pos[s], heads=heads, kv_heads=kvh, keys=rows,
                                  eps=1e-6, theta=1e6)
        return q, k, v

    for a, b in zip(call(rows), call(100)):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
