"""flash_rows with a head a group (few row groups) against two heads a group (many): the same
prompt alone and among others gives the same bits."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q_dtype", [torch.float32, torch.bfloat16])  # bf16: two heads a group always
@pytest.mark.parametrize("heads,kvh", [(16, 8), (16, 2)])
def test_flash_head_groups_agree(heads, kvh, q_dtype):
    from tessera_amd import rules as R
    n, seqs = 256, 9  # 2 row groups alone (16 pairs of heads), 18 together (144: past 128)
    g = torch.Generator(device="cuda").manual_seed(heads + kvh)
    k, v = (torch.randn((n, kvh, 128), device="cuda", generator=g).to(torch.bfloat16) for _ in range(2))
    q = torch.randn((n, heads, 128), device="cuda", generator=g).to(q_dtype)
    pos = torch.arange(n, dtype=torch.int32, device="cuda")
    slots = torch.zeros(n, dtype=torch.int32, device="cuda")
    kw = dict(keys=n, scale=128 ** -0.5, max_position=n - 1)
    alone = R.flash_rows(q, k, v, slots, pos, **kw)
    many = R.flash_rows(q.repeat(seqs, 1, 1), k, v, slots.repeat(seqs), pos.repeat(seqs), **kw).view(seqs, n, heads, 128)
    for s in range(seqs):
        assert torch.equal(many[s], alone)
