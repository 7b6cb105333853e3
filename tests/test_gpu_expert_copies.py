"""Experts' products from the matrices' second copies: of few pairs the bits of the products from the matrices themselves; of many pairs
against the same sums in 64 bits."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# inner sizes of fewer steps than waves, of one, of eight and more a wave, off whole shares; rows of one tile and of many
@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("experts,rows,top,hidden,ff", [(4, 1, 1, 32, 16), (6, 3, 2, 96, 32), (5, 20, 2, 288, 160), (34, 8, 6, 1056, 768),
                                                        (33, 8, 4, 2048, 768), (16, 9, 3, 4096, 1024)])
def test_the_same_bits(gated, experts, rows, top, hidden, ff):
    from leone_amd import ops
    gen = torch.Generator().manual_seed(experts + hidden)
    chosen = torch.stack([torch.randperm(experts + 1, generator=gen)[:top] for _ in range(rows)]).to(torch.int32).to(DEV)
    weight = torch.rand(rows, top, generator=gen).to(DEV)
    x = torch.randn(rows, hidden, generator=gen).bfloat16().to(DEV)
    up = (torch.randn(experts, *((2,) if gated else ()), ff, hidden, generator=gen) / math.sqrt(hidden)).bfloat16().to(DEV)
    down = (torch.randn(experts, hidden, ff, generator=gen) / math.sqrt(ff)).bfloat16().to(DEV)
    copies = (ops.tile_experts(up), ops.tile_experts(down))
    assert rows * top < 8 * experts or experts < 8                    # (tiles of 16 pairs whatever the matrices are read from)
    for options in (({}, {"activation": "gelu_tanh"}) if gated else ({"activation": "relu2"}, {"activation": "relu2", "weigh_input": True})):
        want = ops.routed_experts(x, chosen, weight, up, down, **options)
        assert torch.equal(ops.routed_experts(x, chosen, weight, up, down, copies=copies, **options), want)
        # a copy of more experts than take part
        fewer = ops.routed_experts(x, chosen, weight, up[:experts - 1], down[:experts - 1], **options)
        assert torch.equal(ops.routed_experts(x, chosen, weight, up[:experts - 1], down[:experts - 1], copies=copies, **options), fewer)


def test_where_there_is_no_copy():
    from leone_amd import ops
    assert ops.tile_experts(torch.zeros(2, 24, 32, dtype=torch.bfloat16)) is None
    assert ops.tile_experts(torch.zeros(2, 32, 48, dtype=torch.bfloat16)) is None
    assert ops.tile_experts(torch.zeros(2, 32, 32)) is None
    x = torch.randn(2, 64, device=DEV).bfloat16()
    up, down = torch.randn(3, 2, 32, 64, device=DEV).bfloat16(), torch.randn(3, 64, 32, device=DEV).bfloat16()
    chosen, weight = torch.zeros(2, 1, dtype=torch.int32, device=DEV), torch.ones(2, 1, device=DEV)
    with pytest.raises(ops.KernelError, match="does not belong"):
        ops.routed_experts(x, chosen, weight, up, down, copies=(ops.tile_experts(up)[:2], None))
    want = ops.routed_experts(x, chosen, weight, up, down)
    assert torch.equal(ops.routed_experts(x, chosen, weight, up, down, copies=(None, ops.tile_experts(down))), want)


@pytest.mark.parametrize("wanted,free,kept", [(None, 1 << 40, True), (False, 1 << 40, False), (True, 1 << 40, True), (None, 1 << 15, False), (True, 1 << 15, False)])
def test_a_model_keeps_the_copies_if_there_is_room(monkeypatch, wanted, free, kept):
    from leone_amd import ops
    from leone_amd.parts.base import FEED_FORWARDS, PartSpec
    from leone_amd.parts.model import DecoderModel
    part = FEED_FORWARDS.build(PartSpec("routed_glu", {"hidden": 64, "experts": 2, "top": 1, "intermediate": 32, "router": "r", "expert": "e{e}"}))
    made = {"r": torch.zeros(2, 64), **{f"e{e}.{n}": torch.randn(*shape) for e in range(2)
                                        for n, shape in (("gate", (32, 64)), ("up", (32, 64)), ("down", (64, 32)))}}
    part.bind({name: t.bfloat16().to(DEV) for name, t in made.items()})
    dense = torch.randn(64, 64, device=DEV).bfloat16()

    class Layer:
        parts = staticmethod(lambda: (part,))
        streamed_weights = staticmethod(lambda: [dense])
    model = DecoderModel.__new__(DecoderModel)
    model.layers, model.dtype, model.streamed_copy_bytes, model.head, model.embedding = [Layer], torch.bfloat16, None, None, None
    monkeypatch.setattr(DecoderModel, "streamed_weights", lambda self: [dense])
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda *a: (free, 1 << 40))
    assert model.keep_streamed_copies(wanted) == (0 if wanted is False else 64 * 64 * 2 + (part.expert_copy_bytes() if kept else 0))
    assert (part.copies[0] is not None) == kept
    ops.drop_streamed_copies()


@pytest.mark.parametrize("given", [False, True])
@pytest.mark.parametrize("room", [False, True])
def test_a_cache_is_no_smaller_for_the_copies(monkeypatch, room, given):
    """Memory that would hold the cache or the experts' copies holds the cache, of a size that is given or found; the copies come where there is
    room beside it."""
    from leone_amd import ops
    from leone_amd.api import Runtime, cache_bytes_per_token
    from leone_amd.benchmark import zukinex_shape
    from leone_amd.runtime import random_model
    model = random_model(zukinex_shape(512, 2, 512, 512), 3, "bfloat16")
    experts = sum(part.expert_copy_bytes() for layer in model.layers for part in layer.parts() if hasattr(part, "expert_copy_bytes"))
    dense = sum(-(-w.shape[0] // 16) * 16 * w.shape[1] * 2 for w in model.streamed_weights())
    free = 2 * (dense + experts) + (1 << 20)                 # of which all copies are no more than half
    page = 16 * cache_bytes_per_token(model)
    requests = int(0.7 * (free - dense) / page) // 64        # a cache for them: 64 pages each, most of what is left by the other copies
    limit = torch.cuda.memory_allocated() + free + (3 * experts if room else 0)
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda *a: (limit - torch.cuda.memory_allocated(), 1 << 40))
    runtime = Runtime(model, num_pages=64 * requests if given else None, page_tokens=16, max_requests=requests, max_context=1024)
    assert runtime.engine.cache.free_pages(0) == 64 * requests and torch.cuda.memory_allocated() < limit
    assert model.streamed_copy_bytes == dense + (experts if room else 0)
    assert model.keep_expert_copies() == model.keep_streamed_copies() == model.streamed_copy_bytes        # decided once
    ops.drop_streamed_copies()


@pytest.mark.parametrize("design", ["zukinex", "fosulix", "pamevik"])
def test_models_with_memories_keep_the_order_of_their_sums(design):
    """What a model says of its memories reaches every matrix and every expert's copy."""
    from leone_amd import benchmark, ops
    from leone_amd.runtime import random_model
    model = random_model(getattr(benchmark, design + "_shape")(512, 4, 512, 512), 3, "bfloat16")
    assert model.keep_streamed_copies(True) > 0
    copied = [w for w in model.streamed_weights() if ops.streamed_copy(w) is not None]
    assert copied and all(ops._any_order(w) == (not model.carries_memories()) == (design == "zukinex") for w in copied)
    routed = [part.copies for layer in model.layers for part in layer.parts() if hasattr(part, "expert_copy_bytes")]
    assert bool(routed) == (design != "pamevik") and all(copies[0] is not None and copies[2] == (design == "zukinex") for copies in routed)
    ops.drop_streamed_copies()


def test_copies_without_those_of_the_experts():
    from leone_amd import ops
    from leone_amd.api import Runtime
    from leone_amd.benchmark import zukinex_shape
    from leone_amd.runtime import random_model
    model = random_model(zukinex_shape(512, 2, 512, 512), 3, "bfloat16")
    dense = model.keep_streamed_copies(experts=False)
    Runtime(model, num_pages=8, page_tokens=16, max_requests=1)
    assert dense > 0 and model.streamed_copy_bytes == dense
    assert all(part.copies == (None, None) for layer in model.layers for part in layer.parts() if hasattr(part, "copies"))
    ops.drop_streamed_copies()


# tiles of 64 and 128 pairs, the last of an expert nearly empty or full, experts without pairs; one stage of the inner size, two, an odd number;
# rows of a matrix below, at and off what a workgroup takes, few and many workgroups
@pytest.mark.parametrize("mode", ["gated", "clamped", "plain", "weighed"])
@pytest.mark.parametrize("experts,rows,top,hidden,ff", [(2, 64, 1, 64, 64), (3, 129, 2, 128, 64), (4, 200, 2, 192, 448), (5, 333, 3, 320, 192),
                                                        (40, 1300, 4, 704, 1344), (3, 700, 2, 2048, 832)])
def test_many_pairs(mode, experts, rows, top, hidden, ff):
    of_many_pairs(mode, experts, rows, top, hidden, ff)


# every kind of tile whatever the rule takes for such sizes
@pytest.mark.parametrize("tile", [64, 128])
@pytest.mark.parametrize("mode", ["gated", "clamped", "plain", "weighed"])
@pytest.mark.parametrize("experts,rows,top,hidden,ff", [(2, 64, 1, 64, 64), (3, 129, 2, 128, 64), (4, 200, 2, 192, 448), (5, 333, 3, 320, 192), (3, 700, 2, 2048, 832)])
def test_every_tile_of_many_pairs(monkeypatch, tile, mode, experts, rows, top, hidden, ff):
    from leone_amd import ops
    monkeypatch.setattr(ops, "_copied_tile", lambda *sizes: tile)
    read = []
    monkeypatch.setattr(ops, "call", lambda name, *args, real=ops.call: (read.append(name), real(name, *args))[1])
    of_many_pairs(mode, experts, rows, top, hidden, ff)
    assert "leone_moe_product_tiles" in read and "leone_moe_product" not in read


# 256 rows of both matrices a workgroup, the second's end within one, below and above its half
@pytest.mark.parametrize("mode", ["gated", "plain", "weighed"])
@pytest.mark.parametrize("experts,rows,top,hidden,ff", [(40, 1300, 4, 832, 1344), (40, 1300, 4, 960, 1088), (12, 3100, 2, 1920, 1600)])
def test_twice_the_rows_a_workgroup_in_both_products(mode, experts, rows, top, hidden, ff):
    from leone_amd import ops
    assert hidden % 256 and ff % 128
    pairs, gated = rows * top, mode == "gated"
    assert ops._copied_tile(pairs, experts, hidden, ff, gated, 256) == 128
    tiles = min(pairs, pairs // 128 + experts)
    assert ops.library().leone_moe_many_rows(tiles, experts, ff, 1 if gated else 2) and ops.library().leone_moe_many_rows(tiles, experts, hidden, 0)
    of_many_pairs(mode, experts, rows, top, hidden, ff)


def of_many_pairs(mode, experts, rows, top, hidden, ff):
    from leone_amd import ops
    gen = torch.Generator(device=DEV).manual_seed(rows + ff)
    gated = mode in ("gated", "clamped")
    # the last expert gets nothing, the one before it hands rows on; the first is everybody's favourite
    liked = torch.rand(rows, experts, generator=gen, device=DEV)
    liked[:, 0] += 0.5
    liked[:, experts - 1] = -1.0
    chosen = liked.topk(min(top, experts - 1), dim=1).indices.to(torch.int32).contiguous()
    weight = torch.rand(rows, chosen.shape[1], generator=gen, device=DEV) + 0.1
    x = torch.randn(rows, hidden, generator=gen, device=DEV).bfloat16()
    up = (torch.randn(experts, *((2,) if gated else ()), ff, hidden, generator=gen, device=DEV) / math.sqrt(hidden)).bfloat16()
    down = (torch.randn(experts, hidden, ff, generator=gen, device=DEV) / math.sqrt(ff)).bfloat16()
    options = {"gated": {}, "clamped": {"activation": "clamped_swish", "limit": 0.8}, "plain": {"activation": "relu2"},
               "weighed": {"activation": "gelu_tanh", "weigh_input": True}}[mode]
    copies = (ops.tile_experts(up), ops.tile_experts(down))
    got = ops.routed_experts(x, chosen, weight, up, down, copies=copies, **options)
    want = torch.zeros(rows, hidden, dtype=torch.float64, device=DEV)
    for e in range(experts):
        row, place = (chosen == e).nonzero(as_tuple=True)
        if not len(row):
            continue
        a, t = weight[row, place].double()[:, None], x[row].double()
        if gated:
            g, u = t @ up[e, 0].double().T, t @ up[e, 1].double().T
            if mode == "clamped":
                g, u = g.clamp(max=0.8), u.clamp(-0.8, 0.8)
                h = g * torch.sigmoid(1.702 * g) * (u + 1)
            else:
                h = torch.nn.functional.silu(g) * u
        else:
            h = t @ up[e].double().T * (a if mode == "weighed" else 1.0)
            h = torch.relu(h).square() if mode == "plain" else torch.nn.functional.gelu(h, approximate="tanh")
        out = h.bfloat16().double() @ down[e].double().T
        want.index_add_(0, row, out if mode == "weighed" else a * out)
    # the middle is rounded to 8 bits on both sides, now and then to neighbours: 2^-8 of some elements
    assert float((got - want).norm() / want.norm()) < 2e-3
    assert torch.equal(ops.routed_experts(x, chosen, weight, up, down, copies=copies, **options), got)
    # a pair's result does not depend on the pairs beside it (tiles of the same size)
    some = torch.randperm(rows, generator=torch.Generator().manual_seed(1))[:rows - 3].to(DEV)
    if ops._expert_tiles(x, rows, chosen.shape[1], experts, hidden, ff, True)[0] == ops._expert_tiles(x, rows - 3, chosen.shape[1], experts, hidden, ff, True)[0]:
        assert torch.equal(ops.routed_experts(x[some].contiguous(), chosen[some].contiguous(), weight[some].contiguous(), up, down, copies=copies, **options),
                           got[some])


@pytest.mark.parametrize("experts,rows,top,hidden,ff", [(4, 3, 1, 64, 64), (4, 45, 2, 128, 64), (3, 700, 2, 2048, 832)])
def test_copies_for_sums_in_their_old_order(experts, rows, top, hidden, ff):
    """Few pairs, tiles of 64 and of 128: the bits of the products from the matrices themselves, whatever reads the copies."""
    from leone_amd import ops
    gen = torch.Generator(device=DEV).manual_seed(rows)
    chosen = torch.rand(rows, experts, generator=gen, device=DEV).topk(top, dim=1).indices.to(torch.int32).contiguous()
    weight = torch.rand(rows, top, generator=gen, device=DEV) + 0.1
    x = torch.randn(rows, hidden, generator=gen, device=DEV).bfloat16()
    up = (torch.randn(experts, 2, ff, hidden, generator=gen, device=DEV) / math.sqrt(hidden)).bfloat16()
    down = (torch.randn(experts, hidden, ff, generator=gen, device=DEV) / math.sqrt(ff)).bfloat16()
    copies = (ops.tile_experts(up), ops.tile_experts(down), False)
    assert torch.equal(ops.routed_experts(x, chosen, weight, up, down, copies=copies), ops.routed_experts(x, chosen, weight, up, down))
