"""The persistent decode step at contexts of several attention passes a wave: passes that end
before the position and the edge passes that meet it, at the counts where they change."""
import numpy as np
import pytest

from tests.helpers import cosine, max_rel

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prompt", [156, 160, 163, 319, 355, 700])
def test_persistent_step_matches_graph_at_long_contexts(prompt):
    """Six steps across a pass boundary (160 keys a pass: 8 waves of 5 blocks of 4 keys), one
    launch, against the graph of the lowered kernels over the same weights and kept rows."""
    from tessera_amd.qwen3 import Qwen3, default_config
    cfg = default_config(vocab=2000, hidden=512, layers=3, heads=8, kv_heads=4, ffn=1024, max_context=prompt + 8,
                         max_prompt=prompt)
    tokens = np.random.default_rng(prompt).integers(0, cfg.vocab, prompt).astype(np.uint32)
    got = {}
    for step in (True, False):
        m = Qwen3(cfg, seed=4)
        m.set_step(step)
        m.prefill(tokens)
        picks = m.decode(6)
        got[step] = (picks, m.logits())
        m.close()
    assert np.array_equal(got[True][0], got[False][0])
    assert cosine(got[True][1], got[False][1]) >= 0.99999
    assert max_rel(got[True][1], got[False][1]) <= 1e-3
