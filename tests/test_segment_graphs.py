"""Steps of single tokens of the segment-layout models as graph replays: every replay against the eager step, with prompts,
other batches and eager work between, over block-table widths, slots and pages that change hands, and bounded in number."""
import pytest
import torch

from k8s_llm_rca_amd.engine import graph_runner as G
from k8s_llm_rca_amd.engine.engine import EngineConfig, LLMEngine

pytestmark = pytest.mark.gpu


def engine(model, dtype, graphs):
    return LLMEngine(EngineConfig(model=model, device="cuda", dtype=dtype, num_blocks=96, block_size=64, max_context=2048,
                                  state_slots=6, use_graphs=graphs, prefix_sharing=False, max_decode_seqs=64,
                                  temperature=0.0, seed=3))


def schedule(eng):
    """Logits of a schedule of prompts and single tokens: batches of 3, 2 and 1 that come back after one another, a sequence
    that grows over block-table widths of 1, 2 and 4 pages, releases in between, wanted rows left out and reordered."""
    g = torch.Generator().manual_seed(1)

    def toks(n):
        return torch.randint(0, eng.mc.vocab_size, (n,), generator=g).tolist()
    out, a, b, c = [], eng.new_sequence(), eng.new_sequence(), eng.new_sequence()
    out.append(eng.feed([(a, toks(50), [49]), (b, toks(3), [0, 2]), (c, toks(100), [])]))
    for i in range(12):
        out.append(eng.feed([(a, toks(1), [0]), (b, toks(1), [0]), (c, toks(1), [0])]))
        if i % 3 == 2:
            torch.randn(512, 512, device="cuda").mm(torch.randn(512, 512, device="cuda")).sum().item()
    for _ in range(6):
        out.append(eng.feed([(c, toks(1), [0]), (a, toks(1), [])]))
    eng.release_sequence(b)
    d = eng.new_sequence()
    out.append(eng.feed([(d, toks(30), [29]), (a, toks(1), [0])]))
    for _ in range(8):
        out.append(eng.feed([(d, toks(1), [0]), (c, toks(1), [0]), (a, toks(1), [0])]))
    for _ in range(70):
        out.append(eng.feed([(a, toks(1), [0])]))
    out.append(eng.feed([(a, toks(90), [89])]))
    for _ in range(6):
        out.append(eng.feed([(a, toks(1), [0])]))
    return out


@pytest.mark.parametrize("model", ["tiny-fikerax", "tiny-lizesun"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_replays_equal_eager_steps(model, dtype, monkeypatch):
    want = schedule(engine(model, dtype, False))
    eng = engine(model, dtype, True)
    got = schedule(eng)
    torch.cuda.synchronize()
    assert eng.stats["graph_steps"] > 60 and eng.stats["captures"] >= 4
    for w, x in zip(want, got):       # (all kept until here: what a step returned is not the next one's buffer)
        assert w.shape == x.shape and torch.equal(w, x)
    # the same schedule again on graphs and slots that exist, then with room for two graphs only
    before = eng.stats["captures"]
    for sid in list(eng.seqs):
        eng.release_sequence(sid)
    assert all(torch.equal(w, x) for w, x in zip(want, schedule(eng)))
    assert eng.stats["captures"] == before
    monkeypatch.setattr(G, "SEG_GRAPHS", 2)
    for sid in list(eng.seqs):
        eng.release_sequence(sid)
    assert all(torch.equal(w, x) for w, x in zip(want, schedule(eng)))


@pytest.mark.parametrize("model", ["tiny-fikerax", "tiny-lizesun"])
def test_generation_with_and_without_graphs(model):
    texts = []
    for graphs in (False, True):
        eng = engine(model, torch.float32, graphs)
        done = {}
        for i, n in enumerate((5, 70, 12)):
            prompt = torch.randint(0, eng.mc.vocab_size, (n,), generator=torch.Generator().manual_seed(n)).tolist()
            eng.submit(eng.new_sequence(), prompt, max_new=20 + i, on_done=lambda gen, st, i=i: done.__setitem__(i, list(gen)))
        eng.run_until_idle()
        texts.append(done)
        assert (eng.stats["graph_steps"] > 0) == graphs
    assert texts[0] == texts[1] and len(texts[0]) == 3


@pytest.mark.parametrize("model", ["tiny-fikerax", "tiny-lizesun"])
def test_weights_loaded_after_capture_are_used(model):
    """A graph reads the weights it was captured with: new ones are captured anew; rows without wanted logits replay too."""
    engines = [engine(model, torch.bfloat16, graphs) for graphs in (True, False)]
    sids = [eng.new_sequence() for eng in engines]
    for n in (9, *[1] * 8):
        a, b = (eng.feed([(s, list(range(n)), [n - 1])]) for eng, s in zip(engines, sids))
        assert torch.equal(a, b)
    assert engines[0].stats["captures"] == 1
    for eng in engines:
        eng.model._random_init(11)
    for _ in range(8):
        a, b = (eng.feed([(s, [5], [0])]) for eng, s in zip(engines, sids))
        assert torch.equal(a, b)
    assert engines[0].stats["captures"] == 2
    a, b = (eng.feed([(s, [5], [])]) for eng, s in zip(engines, sids))
    assert a.shape == b.shape and a.shape[0] == 0


def test_a_check_behind_every_launch_runs_steps_eagerly(monkeypatch):
    monkeypatch.setattr(G.KNOBS, "sync_debug", True)
    eng = engine("tiny-fikerax", torch.bfloat16, True)
    sid = eng.new_sequence()
    for _ in range(6):
        eng.feed([(sid, [3], [0])])
    assert eng.stats["captures"] == 0


@pytest.mark.parametrize("model", ["tiny-fikerax", "tiny-lizesun"])
def test_a_capture_that_fails_leaves_the_step_to_the_eager_path(model, monkeypatch):
    """An error that only a capture meets (memory, say): the same logits, no further try at once, and captures of other
    shapes as before."""
    engines = [engine(model, torch.bfloat16, graphs) for graphs in (True, False)]
    eng, forward = engines[0], engines[0].model.forward

    def fails(inp, *a, **k):
        out = forward(inp, *a, **k)
        if torch.cuda.is_current_stream_capturing():
            raise torch.OutOfMemoryError("no memory for a capture")
        return out
    monkeypatch.setattr(eng.model, "forward", fails)
    sids = [[e.new_sequence() for _ in range(2)] for e in engines]

    def step(n, k=1):
        a, b = (e.feed([(s, list(range(n)), [n - 1]) for s in ss[:k]]) for e, ss in zip(engines, sids))
        assert torch.equal(a, b)
    for n in (9, *[1] * 8):
        step(n)
    assert eng.stats["captures"] == 0 == eng.stats["graph_steps"] and not eng._seg.off
    monkeypatch.setattr(eng.model, "forward", forward)
    for _ in range(8):
        step(1)
    assert eng.stats["captures"] == 0                     # (the shape that failed waits)
    for n in (9, *[1] * 8):
        step(n, 2)
    assert eng.stats["captures"] == 1 and eng.stats["graph_steps"] > 0


def test_many_shapes_in_rotation_are_not_captured_again_and_again(monkeypatch):
    monkeypatch.setattr(G, "SEG_GRAPHS", 2)
    engines = [engine("tiny-fikerax", torch.bfloat16, graphs) for graphs in (True, False)]
    sids = [[e.new_sequence() for _ in range(5)] for e in engines]
    for i in range(60):                                   # batches of 5, 4, 3, 2, 1, 5, ..
        k = 5 - i % 5
        a, b = (e.feed([(s, [7 + i], [0]) for s in ss[:k]]) for e, ss in zip(engines, sids))
        assert torch.equal(a, b)
    st = engines[0].stats
    assert st["captures"] * G.SEG_PRICE <= st["graph_steps"] + G.SEG_PRICE * G.SEG_AHEAD and len(engines[0]._seg.graphs) <= 2
