"""Several steps as one graph, each embedding the next one's token (host/sequence.cpp): the same, bit for bit, as steps one by one, for every kind of embedding, with tokens fed and chosen, across the
end of what was fed and across the forms of a step; replayed with other work between."""
import importlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
synth = importlib.import_module("bitnet-rs_amd.synth")


@pytest.mark.parametrize("design", ["lasapel", "mimolix", "lurepel", "sipelorn"])
@pytest.mark.parametrize("fed,prompt,steps", [(30, 6, 23), (6, 6, 9), (12, 3, 14), (140, 120, 19)])
def test_chained_steps(pkg, tmp_path, design, fed, prompt, steps):
    config = getattr(synth, design + "_config")("1b", 2 if design != "mimolix" else 4)
    config["vocab"] = 640
    getattr(synth, "write_" + design)(str(tmp_path), config)
    m = pkg.open_model(str(tmp_path), max_pos=512)
    tokens = np.random.default_rng(fed).integers(0, 640, fed).astype(np.int32)

    def start():
        m.reset()
        m.feed(tokens)
        m.prefill(prompt, with_logits=True, digits=2)

    start()
    one = []
    for _ in range(steps):
        m.run(1)
        one.append(m.last_logits().copy())
    history = m.history(prompt + steps + 1)
    for again in range(3):
        start()
        at = 0
        for n in (steps,) if again == 0 else (5, steps - 5) if again == 1 else (1, 4, steps - 5):
            m.run(n)
            at += n
            assert np.array_equal(m.last_logits(), one[at - 1])
        assert np.array_equal(m.history(prompt + steps + 1), history)


@pytest.mark.parametrize("design", ["lasapel", "lurepel"])
def test_last_hidden_of_replayed_steps(pkg, tmp_path, design):
    """the row of the last position, not of the prompt, on every sequence of a model: as steps without graphs leave it"""
    config = getattr(synth, design + "_config")("1b", 2)
    config["vocab"] = 640
    getattr(synth, "write_" + design)(str(tmp_path), config)
    m = pkg.open_model(str(tmp_path), max_pos=256)
    tokens = np.random.default_rng(3).integers(0, 640, 20).astype(np.int32)
    for again in range(2):
        for n in (1, 9):
            rows = []
            for use_graph in (False, True):
                m.reset()
                m.feed(tokens)
                m.prefill(6, with_logits=True, digits=2)
                prompt = m.last_hidden()
                m.run(n, use_graph=use_graph)
                rows.append(m.last_hidden())
            assert np.array_equal(*rows) and not np.array_equal(prompt, rows[1])
        m.run(1, with_logits=False)
        with pytest.raises(pkg.BitNetHipError, match="without logits"):
            m.last_hidden()


@pytest.mark.parametrize("design", ["lasapel", "mimolix", "lurepel", "sipelorn"])
def test_steps_are_chained(pkg, tmp_path, design):
    """one graph does make several steps where as many are asked for, and is there behind prepare_graphs"""
    config = getattr(synth, design + "_config")("1b", 2 if design != "mimolix" else 4)
    config["vocab"] = 640
    getattr(synth, "write_" + design)(str(tmp_path), config)
    m = pkg.open_model(str(tmp_path), max_pos=128)
    m.prepare_graphs(True)
    m.feed(np.arange(40, dtype=np.int32))
    m.prefill(10, with_logits=True, digits=2)
    for n in (9, 1, 4):
        m.run(n)
        assert (m.last_graph_steps() > 1) == (n > 1)
    m.run(4, use_graph=False)
    assert m.last_graph_steps() == 0
