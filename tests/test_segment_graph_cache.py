"""Which shapes of steps an engine captures: paid for by replays, earned again after giving way, not retried after a failure."""
import random

from k8s_llm_rca_amd.engine import graph_runner as G


def drive(cache, shapes):
    """(captures, replays, eager steps) of a run of steps."""
    n = [0, 0, 0]
    for key in shapes:
        if cache.get(key) is not None:
            n[1] += 1
        elif cache.worth(key):
            cache.put(key, (key,))
            n[0] += 1
        else:
            n[2] += 1
        assert len(cache.graphs) <= G.SEG_GRAPHS
    return n


def test_a_steady_shape_is_captured_after_a_few_steps():
    assert drive(G.SegGraphCache(), [(1, 2)] * 100) == [1, 96, 3]


def test_captures_are_paid_for():
    """More shapes than graphs in rotation, batches that shrink by one every few steps, and random ones: against eager steps
    alone an engine loses no more than its first captures and one per many steps of a shape."""
    r = random.Random(3)
    runs = [[(b, 8) for _ in range(200) for b in range(40, 90)],
            [(b, 8) for b in range(256, 0, -1) for _ in range(5)],
            [(b, 16 + 8 * (i // 50)) for i in range(400) for b in (64, 63, 62, 61)],
            [(r.randint(1, 64), r.choice([8, 16, 24])) for _ in range(20000)]]
    for shapes in runs:
        captures, replays, eager = drive(G.SegGraphCache(), shapes)
        assert captures + replays + eager == len(shapes)
        assert captures * G.SEG_PRICE <= replays + G.SEG_PRICE * (G.SEG_AHEAD + eager // G.SEG_LONG)


def test_a_shape_that_gave_way_is_earned_again(monkeypatch):
    monkeypatch.setattr(G, "SEG_GRAPHS", 2)
    c = G.SegGraphCache()
    drive(c, [(1, 1)] * 8 + [(2, 1)] * 8 + [(3, 1)] * 8)
    assert list(c.graphs) == [(2, 1), (3, 1)]
    for _ in range(G.SEG_GRAPH_AFTER):
        assert c.get((1, 1)) is None and not c.worth((1, 1))
    assert c.worth((1, 1))


def test_a_lonely_shape_comes_to_its_graph_without_credit():
    c = G.SegGraphCache()
    c.credit = 0
    assert drive(c, [(5, 1)] * 200) == [1, 199 - G.SEG_LONG, G.SEG_LONG]


def test_a_failed_capture_is_not_tried_again_at_once():
    c = G.SegGraphCache()
    while not c.worth((1, 1)):
        pass
    c.failed((1, 1))
    assert not any(c.worth((1, 1)) for _ in range(G.SEG_BACKOFF))
    assert drive(c, [(2, 1)] * 10)[0] == 1
    c.off = True
    assert not any(c.worth((3, 1)) for _ in range(1000))
