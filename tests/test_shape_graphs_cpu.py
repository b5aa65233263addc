"""Which batch shapes of a service get a graph: captures are slower than eager calls and must not be made again and again."""
import random

import pytest

from shai_amd.engines.encoders import ShapeGraphs


class Made(list):
    def __call__(self, *shape):
        self.append(shape)
        return shape


def test_second_call_captures():
    made = Made()
    g = ShapeGraphs(made)
    assert g.get((1, 32), 16) is None and g.get((2, 32), 16) is None
    assert g.get((1, 32), 16) == (1, 32) and g.get((1, 32), 16) == (1, 32)
    assert made == [(1, 32)] and len(g) == 1


def test_shapes_that_take_turns():
    """32 batch sizes at two lengths, more than there is room for: one capture each for as many as there is room."""
    made = Made()
    g = ShapeGraphs(made)
    for _ in range(50):
        for b in range(1, 33):
            for n in (32, 128):
                g.get((b, n), 16)
    assert len(made) == 16 and len(set(made)) == 16


@pytest.mark.parametrize("shapes", [64, 2000])
def test_random_shapes(shapes):
    """However shapes come, captures stay few beside calls."""
    made, rng = Made(), random.Random(1)
    g = ShapeGraphs(made)
    for _ in range(20000):
        g.get((rng.randrange(shapes), 32), 16)
        assert len(g) <= 16 and len(g.seen) <= 2 * (g.RECENT + 16) + 1
    assert len(made) <= 16 + 16 * 20000 // g.IDLE


def test_idle_graph_gives_way():
    made = Made()
    g = ShapeGraphs(made)
    g.IDLE = 10
    for s in ("a", "a", "b", "b", "c", "c"):
        g.get((s,), 2)
    assert made == [("a",), ("b",)]
    for _ in range(10):
        assert g.get(("b",), 2) == ("b",)
    assert g.get(("c",), 2) == ("c",) and len(g) == 2 and made == [("a",), ("b",), ("c",)]
    assert g.get(("a",), 2) is None


def test_far_apart_stays_eager():
    made = Made()
    g = ShapeGraphs(made)
    for i in range(400):
        g.get((i % 100,), 16)
    assert not made
