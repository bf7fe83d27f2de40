"""Which decode shapes are recorded, kept and given up (``llmctl.serve.decode_graph.GraphTable``), with stand-ins for graphs."""

import copy

import pytest
import torch

from llmctl.serve import decode_graph as dg


class _Graph:
    def __init__(self, shape):
        self.shape, self.released = shape, False

    def release(self):
        self.released = True


def _walk(table, shape, steps, made):
    def record(s):
        g = _Graph(s)
        made.append(g)
        return g

    return [table.step(shape, record) for _ in range(steps)]


def test_a_shape_is_recorded_after_its_eager_steps():
    t, made = dg.GraphTable(), []
    got = _walk(t, (4, 64), dg.WARM_STEPS + 3, made)
    assert got[:dg.WARM_STEPS] == [None] * dg.WARM_STEPS and len(made) == 1 and len(t) == 1
    assert all(g is made[0] for g in got[dg.WARM_STEPS:])


def test_a_full_table_gives_up_the_shape_that_was_not_used_for_longest(monkeypatch):
    monkeypatch.setattr(dg, "MAX_GRAPHS", 3)
    t, made = dg.GraphTable(), []
    for n in (1, 2, 3):
        _walk(t, (n, 64), dg.WARM_STEPS + 1, made)
    _walk(t, (1, 64), 1, made)  # used again: shape 2 is the oldest now
    got = _walk(t, (4, 64), dg.CROWDED_STEPS + 1, made)  # a longer wait once another one has to go
    assert got[:dg.CROWDED_STEPS] == [None] * dg.CROWDED_STEPS and got[-1] is made[3]
    assert [g.released for g in made] == [False, True, False, False] and len(t) == 3
    assert _walk(t, (1, 64), 1, made) == [made[0]] and _walk(t, (3, 64), 1, made) == [made[2]]
    assert _walk(t, (2, 64), 1, made) == [None] and len(made) == 4  # counts its eager steps anew
    t.clear()
    assert len(t) == 0 and all(g.released for g in made)


def test_a_shape_that_does_not_record_stays_eager():
    t, tries = dg.GraphTable(), []
    got = [t.step((2, 32), lambda s: tries.append(s)) for _ in range(dg.WARM_STEPS + 5)]
    assert got == [None] * len(got) and tries == [(2, 32)] and len(t) == 0
    t.clear()  # (weights changed: it may record now)
    assert [t.step((2, 32), _Graph) is None for _ in range(dg.WARM_STEPS + 1)] == [True] * dg.WARM_STEPS + [False]


def _key_changes(change):
    from llmctl.serve.engine import InferenceEngine

    e = InferenceEngine("dumazen-w128-l4-h4-g2", device="cpu", max_batch_size=2, num_kv_blocks=16, block_size=16, max_model_len=64)
    key = e._weights_key()
    assert e._weights_key() == key
    with torch.no_grad():
        change(e.model)
    return e._weights_key() != key


@pytest.mark.parametrize("change", [
    lambda m: m.layers[0].ff.w_up.mul_(2.0),
    lambda m: m.load_state_dict({k: v.clone() for k, v in m.state_dict().items()}, assign=True),
    lambda m: setattr(m.layers[0].ff, "w_up", torch.nn.Parameter(m.layers[0].ff.w_up.clone())),
    lambda m: _change_places(m.layers[0].ff.w_up, m.layers[1].ff.w_up),
    lambda m: setattr(m.layers[0], "ff", m.layers[1].ff),
    lambda m: setattr(m.layers[2], "ff", copy.deepcopy(m.layers[2].ff)),
    lambda m: m.layers[0].ff.register_buffer("extra", torch.zeros(1))])
def test_every_change_of_the_weights_shows(change):
    assert _key_changes(change)


def _change_places(a, b):
    a.data, b.data = b.data, a.data


def test_an_unchanged_model_keeps_its_key():
    assert not _key_changes(lambda m: None)
    with torch.inference_mode():  # weights made in inference mode have no versions
        assert not _key_changes(lambda m: None)
