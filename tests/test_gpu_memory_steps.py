"""Matrix memories in steps of single rows, which kernels of their own take, against the same rows in a step that also holds a
portion of two rows and is walked by the general kernels (those are tested against the recurrence in double precision)."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
SINGLE = [(1, 0), (1, 7), (1, 40)]                            # rows and place they start at: a first token and later ones
SLOTS = [2, 0, 3, 1]


def step_of(entries):
    from leone_amd.parts.context import EntryInfo, StepContext
    infos, positions, owners = [], [], []
    for i, (slot, (count, start)) in enumerate(zip(SLOTS, entries)):
        infos.append(EntryInfo(f"r{i}", slot, len(positions), count, start))
        positions += range(start, start + count)
        owners += [i] * count
    on = lambda values: torch.tensor(values, dtype=torch.int32, device=DEV)     # noqa: E731
    return StepContext(rows=len(positions), dtype=torch.float32, device=torch.device(DEV), positions=on(positions), row_entry=on(owners),
                       entries=infos, entry_slots=on(SLOTS[:len(entries)]), want_rows=None)


def same(got, want):
    # the same sums in the same order, products perhaps fused into sums on one side only: a few 2^-24 of the result's size
    got, want = got.cpu().double(), want.cpu().double()
    assert float((got - want).norm()) <= 1e-6 * float(want.norm()), float((got - want).norm() / want.norm())


def state_of(size, gen):
    state = torch.randn(*size, generator=gen)
    state[SLOTS[0]] = math.nan                                # a first token starts from zeros, whatever its slot holds
    return state


@pytest.mark.parametrize("dim,vdim,rot", [(32, 1, 0), (64, 63, 64), (64, 64, 0), (128, 65, 64), (256, 512, 0), (256, 130, 256), (96, 64, 0),
                                          (255, 16, 0)])
@pytest.mark.parametrize("gated,silu,write", [(True, False, True), (False, True, True), (False, False, False)])
def test_outer_products_of_single_rows(dim, vdim, rot, gated, silu, write):
    """Columns below, at and off a wave's 64; one to eight waves; sizes that the kernel for single rows does not take."""
    from leone_amd import ops
    heads, gen = 3, torch.Generator().manual_seed(dim + vdim)
    width = 2 * heads * dim + heads * vdim
    x = torch.randn(5, width + 2 * heads, generator=gen).to(DEV)
    state = state_of((4, heads, dim * vdim + (dim + 1 if gated else 0)), gen)
    bias, decay = torch.randn(2, heads, generator=gen).to(DEV), torch.tensor([0.97, 0.0, 1.0], device=DEV)
    cos, sin = ops.rope_table(1e4, rot, 300, DEV) if rot else (None, None)
    columns = {"q": 0, "k": heads * dim, "v": 2 * heads * dim, "i": width, "f": width + heads}
    results = []
    for entries in (SINGLE, SINGLE + [(2, 0)]):
        step, kept = step_of(entries), state.to(DEV)
        out, under = ops.outer_scan(x[:step.rows].contiguous(), columns, kept, step, heads, dim, vdim, q_scale=dim ** -0.5, k_scale=0.7,
                                    cos=cos, sin=sin, activation="silu" if silu else None, write_state=write,
                                    **(dict(gates={"i_bias": bias[0], "f_bias": bias[1], "cap": 15.0}) if gated else dict(decay=decay)))
        results.append([out[:3]] + [u[:3] for u in under or ()] + [kept[SLOTS[:3] if write else SLOTS[1:3]]])
        assert write or torch.equal(kept[SLOTS[1:3]].cpu(), state[SLOTS[1:3]])
    for got, want in zip(*results):
        same(got, want)


@pytest.mark.parametrize("dim,vdim", [(32, 1), (64, 63), (128, 64), (128, 128), (256, 65), (96, 64), (100, 16)])
@pytest.mark.parametrize("per_head,weights,write", [(False, torch.bfloat16, True), (True, torch.float32, True), (False, torch.float32, False)])
def test_delta_rule_of_single_rows(dim, vdim, per_head, weights, write):
    from leone_amd import ops
    heads, kv_heads, gen = 4, 2, torch.Generator().manual_seed(dim + vdim)
    width = 2 * kv_heads * dim + heads * vdim
    x = torch.randn(5, width, generator=gen).to(DEV)
    beta, step_size = torch.randn(5, heads, generator=gen).to(DEV), torch.randn(5, heads * (1 if per_head else dim), generator=gen).to(DEV)
    rate, bias = torch.randn(heads, generator=gen).to(weights).to(DEV), torch.randn(step_size.shape[1], generator=gen).to(weights).to(DEV)
    state = state_of((4, heads, dim, vdim), gen)
    columns = {"q": 0, "k": kv_heads * dim, "v": 2 * kv_heads * dim}
    results = []
    for entries in (SINGLE, SINGLE + [(2, 0)]):
        step, kept = step_of(entries), state.to(DEV)
        n = step.rows
        out = ops.delta_scan(x[:n].contiguous(), columns, beta[:n].contiguous(), step_size[:n].contiguous(), rate, bias, kept, step, heads,
                             kv_heads, dim, vdim, dim ** -0.5, 1e-6, write)
        results.append([out[:3], kept[SLOTS[:3] if write else SLOTS[1:3]]])
    for got, want in zip(*results):
        same(got, want)
