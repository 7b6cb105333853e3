"""The 32-bit engine: what a request gets does not depend on the requests beside it, to the bit."""
import pytest
import torch

from tests import util

pytestmark = pytest.mark.gpu


def test_logits_alone_and_beside_others(tmp_path):
    """A prompt of 70 tokens, a portion behind it and decoded tokens, alone and in steps with prompts and decoded tokens of up to 40
    other requests: widths that are cut into segments, heads on the matrix instructions, every kernel that a row count chooses."""
    from leone_amd.engine.engine import Engine, StepEntry
    from leone_amd.runtime import load_model
    folder = util.make_model_dir(str(tmp_path / "m"), util.TINY_M, 5, torch.float32, sharpen=3.0)
    vocab = util.TINY_M["vocab_size"]
    mine = util.random_tokens(1, 96, vocab)
    cuts = [mine[:70], mine[70:93]] + [[t] for t in mine[93:]]

    def logits(others):
        engine = Engine(load_model(folder, "float32"), max_tokens=4096, page_tokens=16, max_requests=42)
        for i in range(others):
            engine.step([StepEntry(f"o{i}", util.random_tokens(50 + i, 3 + 5 * i % 37, vocab))])
        out = []
        for n, cut in enumerate(cuts):
            beside = [StepEntry(f"o{i}", util.random_tokens(100 * n + i, 1 if i else 60, vocab)) for i in range(others)]
            step = engine.step(beside[:others // 2] + [StepEntry("mine", cut, range(len(cut)))] + beside[others // 2:])
            out.append(step.logits.clone())
        return torch.cat(out)

    alone = logits(0)
    assert alone.shape == (96, vocab) and bool(torch.isfinite(alone).all())
    for others in (1, 7, 40):
        assert torch.equal(logits(others), alone), others
