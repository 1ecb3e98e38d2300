"""Token ids that the embedding does not have are refused on the host, in front of everything else."""
import pytest

from k8s_llm_rca_amd.engine.engine import EngineConfig, LLMEngine


@pytest.mark.parametrize("dev", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("bad", [-1, "rows", 1 << 40])
def test_refused(dev, bad):
    eng = LLMEngine(EngineConfig(model="tiny-llama", device=dev, seed=1, num_blocks=16, block_size=64, max_context=256))
    rows = eng.model.embed.shape[0]
    a, b = eng.new_sequence(), eng.new_sequence()
    ids = [3, rows if bad == "rows" else bad, 4]
    with pytest.raises(IndexError):
        eng.feed([(a, [1, 2], [1]), (b, ids, [2])])
    assert not eng.seqs[a].tokens and not eng.seqs[b].tokens            # nothing was taken of either
    with pytest.raises(IndexError):
        eng.submit(a, ids)
    assert not eng._incoming
    out = eng.feed([(a, [0, rows - 1], [0, 1])])                        # both ends of the table
    assert bool(out.isfinite().all()) and len(out) == 2
