"""The router's choice by ranks, the tiles of many experts, and the experts' products in tiles of 16 and 64 pairs, at their edges."""
import math

import pytest
import torch

from tests.plain import zukinex_plain as plain

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
F = torch.float64


@pytest.mark.parametrize("total,top,count,keep", [(1, 1, 1, 1), (64, 64, 1, 1), (64, 6, 8, 3), (63, 5, 9, 2), (64, 8, 64, 8), (35, 4, 7, 4)])
def test_ranks_of_one_output_a_lane(total, top, count, keep):
    """Scores of few values, so that most of them tie: of equals the lower index wins, in groups and among the open outputs."""
    from leone_amd import ops
    gen = torch.Generator().manual_seed(total + top)
    logits = torch.zeros(90, total)
    correction = torch.randint(-2, 3, (total,), generator=gen).float() * 0.25
    chosen, weight = ops.route_topk(logits.to(DEV), correction.to(DEV), top, count, keep)
    score = torch.full((total,), 1.0 / total) + correction
    groups = score.view(count, -1).max(-1).values
    order = sorted(range(count), key=lambda g: (-float(groups[g]), g))[:keep]
    open_ = [e for e in range(total) if e // (total // count) in order]
    want = sorted(open_, key=lambda e: (-float(score[e]), e))[:top]
    assert chosen.cpu().tolist() == [want] * 90
    assert float((weight.cpu() - 1.0 / top).abs().max()) < 1e-6       # equal scores over their sum: rounded a few times


def test_scores_that_are_no_numbers_choose_outputs_all_the_same():
    from leone_amd import ops
    logits = torch.randn(6, 35)
    logits[1], logits[2, 4], logits[3] = math.nan, math.inf, -math.inf
    chosen, weight = ops.route_topk(logits.to(DEV), None, 4, 7, 4)
    for row in chosen.cpu().tolist():
        assert len(set(row)) == 4 and all(0 <= e < 35 for e in row)
    assert bool(torch.isfinite(weight[[0, 4, 5]]).all()) and bool(torch.isnan(weight[[1, 2, 3]]).all())


@pytest.mark.parametrize("experts,rows,top", [(1000, 40, 3), (65, 30, 2), (128, 64, 8), (3, 50, 2)])
def test_products_in_tiles_of_sixteen(experts, rows, top):
    """Up to 1,000 experts' tiles; experts with more pairs than a tile; inner sizes below, at and off a wave's share."""
    from leone_amd import ops
    gen = torch.Generator().manual_seed(experts)
    chosen = torch.stack([torch.randperm(experts, generator=gen)[:top] for _ in range(rows)]).to(torch.int32)
    weight = torch.rand(rows, top, generator=gen)
    for hidden, ff in ((8, 8), (40, 24), (136, 1000)) if experts < 200 else ((40, 24),):
        x = torch.randn(rows, hidden, generator=gen).bfloat16()
        up = (torch.randn(experts, 2, ff, hidden, generator=gen) / math.sqrt(hidden)).bfloat16()
        down = (torch.randn(experts, hidden, ff, generator=gen) / math.sqrt(ff)).bfloat16()
        got = ops.routed_experts(x.to(DEV), chosen.to(DEV), weight.to(DEV), up.to(DEV), down.to(DEV)).cpu().double()
        want = torch.zeros(rows, hidden, dtype=F)
        for t in range(rows):
            for e, a in zip(chosen[t].tolist(), weight[t].double()):
                g, u = (up[e, i].double() @ x[t].double() for i in (0, 1))
                want[t] += a * (down[e].double() @ (plain.silu(g) * u).bfloat16().double())
        # the middle is rounded to 8 bits on both sides, now and then to neighbours: 2^-8 of some elements of one place's sum
        assert float((got - want).norm() / want.norm()) < 2e-3


@pytest.mark.parametrize("counts,hidden,ff", [((63, 64, 65, 129, 0, 1), 8, 8), ((64, 128, 1), 64, 56), ((129, 2, 64), 72, 136),
                                              ((65, 63), 136, 64), ((200,), 200, 72), ((33,) + (0,) * 40, 264, 40)])
@pytest.mark.parametrize("gated", [True, False])
def test_products_in_tiles_of_sixty_four(counts, hidden, ff, gated):
    """Tiles just full, one short and one over; inner sizes below, at and off a chunk of 64, odd and even numbers of chunks; result
    rows off a workgroup's 64 and 128; the last case, few pairs for its experts, takes several tiles of 16 for one expert."""
    from leone_amd import ops
    experts, pairs = len(counts), sum(counts)
    top = 1 if pairs % 2 else 2
    gen = torch.Generator().manual_seed(pairs + hidden)
    which = torch.tensor([e for e, count in enumerate(counts) for _ in range(count)])[torch.randperm(pairs, generator=gen)]
    chosen = which.view(-1, top).to(torch.int32)
    weight = torch.rand(pairs // top, top, generator=gen) + 0.1
    x = torch.randn(pairs // top, hidden, generator=gen).bfloat16()
    up = (torch.randn(experts, 2 if gated else 1, ff, hidden, generator=gen) / math.sqrt(hidden)).bfloat16()
    down = (torch.randn(experts, hidden, ff, generator=gen) / math.sqrt(ff)).bfloat16()
    for weigh_input in (False,) if gated else (False, True):
        got = ops.routed_experts(x.to(DEV), chosen.to(DEV), weight.to(DEV), (up if gated else up[:, 0]).to(DEV), down.to(DEV),
                                 "silu" if gated else "relu2", weigh_input=weigh_input).cpu().double()
        rows = x.double().repeat_interleave(top, 0)
        a = weight.double().view(-1, 1)
        first = torch.stack([up[e, 0].double() @ r for e, r in zip(which, rows)])
        if gated:
            middle = plain.silu(first) * torch.stack([up[e, 1].double() @ r for e, r in zip(which, rows)])
        else:
            middle = (a * first if weigh_input else first).clamp(min=0).square()
        each = torch.stack([down[e].double() @ m for e, m in zip(which, middle.bfloat16().double())])
        want = (each if weigh_input else a * each).view(-1, top, hidden).sum(1)
        # as above: middles that are rounded to neighbours, 2^-8 of some elements of one place's sum
        assert float((got - want).norm() / want.norm()) < 2e-3


@pytest.mark.parametrize("counts,hidden,ff", [((127, 128, 129, 256, 0, 1, 300), 72, 136), ((65, 257), 136, 64), ((200,), 8, 200)])
@pytest.mark.parametrize("gated", [True, False])
def test_products_in_tiles_of_a_hundred_and_twenty_eight(counts, hidden, ff, gated, monkeypatch):
    """As above, at sizes too small for these tiles by the rule."""
    from leone_amd import ops
    kinds = []

    def tiles(x, rows, top, experts, hidden, ff):
        most = min(rows * top, rows * top // 128 + experts)
        kinds.append(most)
        return 128, most, torch.empty(most, dtype=torch.int32, device=DEV), torch.empty(most, 128, dtype=torch.int32, device=DEV)
    monkeypatch.setattr(ops, "_expert_tiles", tiles)
    test_products_in_tiles_of_sixty_four(counts, hidden, ff, gated)
    assert kinds


def test_tiles_by_pairs_and_width():
    """The size of a tile by the pairs an expert gets on average, the width, and whether tiles of 64 give every unit a workgroup."""
    from leone_amd import ops
    for hidden, experts, ff, lines in ((1024, 32, 512, (12, 1193)), (2048, 34, 768, (8, 374)), (4096, 8, 2048, (8, 299)), (1024, 8, 4096, (14, 597)),
                                       (2048, 128, 768, (8, 160))):
        for line, below, above in zip(lines, (16, 64), (64, 128)):
            x = torch.empty(1, hidden, dtype=torch.bfloat16, device=DEV)
            assert ops._expert_tiles(x, (line - 1) * experts, 1, experts, hidden, ff)[0] == below
            assert ops._expert_tiles(x, line * experts, 1, experts, hidden, ff)[0] == above


def _through_experts(x, which, weight, up, down, gated, weigh_input=False):
    """Pair by pair through the experts in 64 bits, the middle rounded as the kernels hand it on.  up: [experts, 1 or 2, ff, hidden]."""
    want = torch.empty(len(which), down.shape[1], dtype=F)
    for e in range(up.shape[0]):
        mine = which == e
        a, first = weight[mine].double(), x[mine].double() @ up[e, 0].double().T
        middle = plain.silu(first) * (x[mine].double() @ up[e, 1].double().T) if gated else (a * first if weigh_input else first).clamp(min=0).square()
        each = middle.bfloat16().double() @ down[e].double().T
        want[mine] = each if weigh_input else a * each
    return want


def _dealt(counts, hidden, ff, gated, seed):
    gen = torch.Generator().manual_seed(seed)
    which = torch.tensor([e for e, count in enumerate(counts) for _ in range(count)])[torch.randperm(sum(counts), generator=gen)]
    return (torch.randn(len(which), hidden, generator=gen).bfloat16(), which, torch.rand(len(which), 1, generator=gen) + 0.1,
            (torch.randn(len(counts), 2 if gated else 1, ff, hidden, generator=gen) / math.sqrt(hidden)).bfloat16(),
            (torch.randn(len(counts), hidden, ff, generator=gen) / math.sqrt(ff)).bfloat16())


def _check_pairs(counts, hidden, ff, gated, tile):
    from leone_amd import ops
    x, which, weight, up, down = _dealt(counts, hidden, ff, gated, hidden + ff)
    assert ops._expert_tiles(x.to(DEV), len(which), 1, len(counts), hidden, ff)[0] == tile
    for weigh_input in (False,) if gated else (False, True):
        got = ops.routed_experts(x.to(DEV), which.view(-1, 1).to(torch.int32).to(DEV), weight.to(DEV), (up if gated else up[:, 0]).to(DEV),
                                 down.to(DEV), "silu" if gated else "relu2", weigh_input=weigh_input).cpu().double()
        want = _through_experts(x, which, weight, up, down, gated, weigh_input)
        # as above: middles that are rounded to neighbours
        assert float((got - want).norm() / want.norm()) < 2e-3


@pytest.mark.parametrize("hidden,ff", [(264, 576), (328, 520), (392, 512), (448, 328), (512, 640), (520, 448), (576, 264), (704, 136)])
@pytest.mark.parametrize("gated", [True, False])
def test_tiles_of_sixty_four_over_many_chunks(hidden, ff, gated):
    """Inner sizes of 3 to 11 chunks of 64, on and off a whole one: the loop over two chunks none, one and several times and every
    number of chunks behind it, for the first product and the second."""
    _check_pairs([63, 64, 65, 130, 1], hidden, ff, gated, 64)


@pytest.mark.parametrize("hidden,ff", [(1032, 1408), (1408, 2056), (2048, 1032), (2056, 2568), (2568, 2048), (40, 4104), (4104, 24), (1984, 1000)])
@pytest.mark.parametrize("gated", [True, False])
def test_tiles_of_sixteen_over_long_rows(hidden, ff, gated):
    """Inner sizes whose share of a wave is one batch of eight steps and a remainder, two and more batches, and ends inside a step; of
    more than 2,048 by ordinary loads."""
    _check_pairs([5, 0, 17, 2], hidden, ff, gated, 16)


def test_products_with_one_chunk_ahead():
    """Experts whose matrices give every unit one workgroup, with rows whole multiples of 4 KB apart; some with more pairs than a tile."""
    from leone_amd.ops.library import library
    assert library().leone_moe_one_chunk_ahead(16, 1, 1024, 2048)
    _check_pairs([3, 64, 1, 65, 0, 130] + [20] * 10, 2048, 1024, True, 64)


@pytest.mark.parametrize("rows,total,top,always", [(1, 1, 1, 0), (8, 35, 4, 1), (17, 64, 12, 0), (64, 100, 9, 2), (256, 64, 8, 0), (256, 64, 9, 0),
                                                   (30, 300, 70, 1)])
@pytest.mark.parametrize("corrected", [None, torch.float32, torch.bfloat16])
def test_choice_and_tiles_in_one_launch(rows, total, top, always, corrected):
    """The choices and weights of route_topk and every pair once, in a tile of its expert, on both sides of what is handed on through
    shared memory (2,048 pairs) and of the launch's 16 rows at a time; outputs that stand for no matrix are numbered behind all."""
    from leone_amd import ops
    gen = torch.Generator().manual_seed(rows + total)
    logits = torch.randn(rows, total, generator=gen).to(DEV)
    correction = None if corrected is None else torch.randn(total, generator=gen).to(DEV).to(corrected)
    routed = max(1, total - 3)                             # three outputs stand for no matrix
    experts, places, tile = routed + always, top + always, ops.library().leone_moe_tile_pairs()
    want, want_weight = ops.route_topk(logits, correction, top)
    pairs = rows * places
    tiles = min(pairs // tile + experts, pairs)
    chosen = torch.empty(rows, places, dtype=torch.int32, device=DEV)
    weight = torch.empty(rows, places, device=DEV)
    tile_expert, tile_pairs = torch.empty(tiles, dtype=torch.int32, device=DEV), torch.empty(tiles, tile, dtype=torch.int32, device=DEV)
    ops.call("leone_route_plan", logits.data_ptr(), 0 if correction is None else correction.data_ptr(),
                     ops.BF16 if corrected == torch.bfloat16 else ops.F32, chosen.data_ptr(), weight.data_ptr(), rows, total, top,
                     1, 1, experts, tile_expert.data_ptr(), tile_pairs.data_ptr(), tiles, tile, always, *ops._DEFAULT_RULE.args(), ops._stream())
    torch.cuda.synchronize()
    assert torch.equal(chosen[:, :top], torch.where(want >= routed, want + always, want)) and torch.equal(weight[:, :top], want_weight)
    assert chosen[:, top:].tolist() == [list(range(routed, experts))] * rows and bool((weight[:, top:] == 1).all())
    of = chosen.flatten().tolist()
    found = [(pair, e) for e, held in zip(tile_expert.tolist(), tile_pairs.tolist()) for pair in held if pair >= 0]
    assert sorted(found) == [(pair, e) for pair, e in enumerate(of) if e < experts]
    held = [e for e in tile_expert.tolist() if e >= 0]
    assert len(held) == sum(math.ceil(of.count(e) / tile) for e in set(of) if e < experts)
