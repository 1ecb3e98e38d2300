"""The last product of a replayed step is made behind its graph, or inside it where it takes the residual's pass with it."""
import pytest
import torch

from k8s_llm_rca_amd.engine.engine import EngineConfig, LLMEngine
from k8s_llm_rca_amd.models.registry import get_any_config
from k8s_llm_rca_amd.ops import row_step as R


@pytest.mark.gpu
@pytest.mark.parametrize("model", ["fikerax-1b", "lizesun-1b"])
@pytest.mark.parametrize("into", [True, False])
def test_replays_equal_eager_steps(model, into, monkeypatch):
    if not into:                                     # (one row: the next product makes the pass)
        monkeypatch.setattr(R, "into_ok", lambda *a, **k: False)
    fewer = {"layers": get_any_config(model).layers[:2]} if model == "lizesun-1b" else {}
    said = []
    for graphs in (True, False):
        eng = LLMEngine(EngineConfig(model=model, model_overrides=fewer, device="cuda", dtype=torch.bfloat16, seed=5,
                                     num_blocks=32, block_size=64, max_context=512, state_slots=2, use_graphs=graphs))
        sids = [eng.new_sequence(), eng.new_sequence()]
        out = [eng.feed([(s, [7, 8, 9], [2]) for s in sids])]
        out += [eng.feed([(sids[0], [11 + i], [0])]) for i in range(10)]
        out += [eng.feed([(s, [31 + i], [0]) for s in sids]) for i in range(10)]
        said.append(out)
        if graphs:
            whole = {key[0]: got[3] for key, got in eng._seg.graphs.items()}
            assert whole == {1: not into, 2: False} and eng.stats["graph_steps"] >= 10
    assert all(torch.equal(a, b) for a, b in zip(*said))     # (all kept until here)
