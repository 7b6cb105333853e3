"""Steps of single tokens replayed from a recording: the layout written in one call, and what it leaves to the general one."""
import numpy as np
import pytest
import torch

from tests.util import TINY, make_model_dir, random_tokens

pytestmark = pytest.mark.gpu


def test_the_same_layout_and_the_same_refusals(tmp_path):
    from leone_amd.engine.engine import Engine, PackedStep, StepEntry, StepError
    from leone_amd.runtime import load_model
    folder = make_model_dir(str(tmp_path / "m"), TINY["M"], 6, torch.bfloat16)
    engine = Engine(load_model(folder, "bfloat16"), num_pages=32, page_tokens=16, max_requests=4)
    vocab = engine.vocab_size
    for i, n in enumerate((3, 40, 17)):
        engine.step([StepEntry(f"r{i}", random_tokens(i, n, vocab))])
    entries = [StepEntry(f"r{i}", [5 + i], [0]) for i in (2, 0, 1)]
    first = engine.step(entries).logits                                     # recorded
    state = engine._decode_graphs[3]
    for tokens in ([5, 6, 7], [np.int64(8), 9, 10], np.array([[11], [12], [0]])[:, 0]):
        made = [StepEntry(e.request, [t], e.want) for e, t in zip(entries, tokens)]
        taken = state._pack_single(engine, made)
        assert (taken is None) == any(type(t) is not int for t in tokens)
        want = PackedStep(engine.cache, vocab, made, all_rows_wanted=True, tilings=engine.tilings)
        if taken is not None:
            assert taken == want.max_position and torch.equal(state.host, want.host[:state.host.numel()])
        assert engine.step(made).logits.shape == first.shape
    lengths = [engine.length(f"r{i}") for i in range(3)]
    for bad in ([vocab, 1, 1], [-1, 1, 1], [True, 1, 1], [1.0, 1, 1]):
        with pytest.raises(StepError):
            engine.step([StepEntry(e.request, [t], e.want) for e, t in zip(entries, bad)])
    with pytest.raises(StepError):
        state.fill(engine, [StepEntry("r0", [1], [0]), StepEntry("nobody", [1], [0]), StepEntry("r1", [1], [0])])
    with pytest.raises(StepError):
        state.fill(engine, [StepEntry("r0", [1], [0]), StepEntry("r0", [1], [0]), StepEntry("r1", [1], [0])])
    assert [engine.length(f"r{i}") for i in range(3)] == lengths
    some = engine.step([StepEntry("r0", [1], []), StepEntry("r1", [1], [0]), StepEntry("r2", [1], [])])
    assert some.rows == [("r1", 0)] and some.logits.shape == (1, vocab)
