"""Exponential gates made in the step's launch, their maxima kept by the norm behind it, against gates of their own launch: the same bits."""
import pytest
import torch

from leone_amd import ops
from tests.test_gpu_memory_steps import DEV, SINGLE, SLOTS, state_of, step_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,vdim", [(32, 1), (64, 63), (128, 65), (256, 512), (32, 1040), (96, 64)])      # one to eight waves; wide heads; not taken
@pytest.mark.parametrize("biases", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("write", [True, False])
def test_gates_in_the_step(dim, vdim, biases, write):
    heads, gen = 5, torch.Generator().manual_seed(dim + vdim)
    width = 2 * heads * dim + heads * vdim
    x = (3.0 * torch.randn(3, width + 2 * heads, generator=gen)).to(DEV)
    x[1, width] = float("inf")                                # beyond the cap, and not a number
    x[2, width + heads + 1] = float("nan")
    state = state_of((4, heads, dim * vdim + dim + 1), gen)
    bias = torch.randn(2, heads, generator=gen).to(biases).to(DEV)
    gates = {"i_bias": bias[0].contiguous(), "f_bias": bias[1].contiguous(), "cap": 15.0}
    columns = {"q": 0, "k": heads * dim, "v": 2 * heads * dim, "i": width, "f": width + heads}
    found = []
    for later in (False, True):
        step, kept = step_of(SINGLE), state.to(DEV)
        out, under = ops.outer_scan(x, columns, kept, step, heads, dim, vdim, gates=gates, q_scale=dim ** -0.5, write_state=write, keep_later=later)
        assert len(under) == (3 if later and write and dim != 96 else 2)
        y = ops.head_norm_gate(out, heads, vdim, 1e-5, torch.float32, denominator=under)
        found.append([out, under[0], under[1], y, kept])
    for one, two in zip(*found):
        assert torch.equal(one.nan_to_num(7e7, 8e7, -8e7), two.nan_to_num(7e7, 8e7, -8e7))
    assert not write or not torch.equal(found[0][4][SLOTS[1], :, -1].cpu(), state[SLOTS[1], :, -1])


def test_longer_entries_keep_their_gates_launch():
    heads, dim, vdim, gen = 2, 32, 16, torch.Generator().manual_seed(1)
    width = 2 * heads * dim + heads * vdim
    step = step_of(SINGLE[:1] + [(2, 0)])
    x = torch.randn(step.rows, width + 2 * heads, generator=gen).to(DEV)
    state = state_of((4, heads, dim * vdim + dim + 1), gen).to(DEV)
    bias = torch.zeros(heads, device=DEV)
    _, under = ops.outer_scan(x, {"q": 0, "k": heads * dim, "v": 2 * heads * dim, "i": width, "f": width + heads}, state, step, heads, dim, vdim,
                              gates={"i_bias": bias, "f_bias": bias, "cap": 15.0}, keep_later=True)
    assert len(under) == 2
