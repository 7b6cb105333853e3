"""Decode attention over pages that hold whole tiles of keys (one address a tile) against pages of 16 tokens (an address a lane): the
same keys and queries, to the bit; the merge of key ranges against one range; the embedding in fours."""
import pytest
import torch

from tests.test_gpu_attention_f32 import pools

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TOKENS = 330


def made(kv_heads, size, requests, seed=3):
    gen = torch.Generator().manual_seed(seed)
    return [torch.randn(requests, TOKENS, kv_heads, size, generator=gen).bfloat16().float() for _ in range(2)]


def bits(pool):
    return pool.to(torch.bfloat16)


# (sixteen columns of 256 elements are more shared memory than a workgroup takes: refused)
@pytest.mark.parametrize("size,group,kv_heads", [(size, *heads) for size in (16, 64, 80, 128, 256) for heads in ((1, 2), (4, 2), (20, 1))
                                                 if (size, heads) != (256, (20, 1))])
def test_results_do_not_depend_on_the_pages(size, group, kv_heads):
    from leone_amd import ops
    places = [0, 1, 31, 32, 33, 127, 128, 200, 329]
    k, v = made(kv_heads, size, len(places))
    gen = torch.Generator().manual_seed(size)
    q = torch.randn(len(places), group * kv_heads * size, generator=gen).bfloat16().to(DEV)
    positions = torch.tensor(places, dtype=torch.int32, device=DEV)
    rows = torch.arange(len(places), dtype=torch.int32, device=DEV)
    for options in ({}, {"window": 40}, {"window": 33, "keep_first": 5}, {"chunk": 96}):
        for splits in (1, 3, 20):
            found = []
            for page_tokens in (16, 32, 64, 128):
                k_pool, v_pool, table = pools(k, v, page_tokens, page_tokens)
                found.append(ops.attention_decode(q, bits(k_pool), bits(v_pool), positions, rows, table, group * kv_heads, size ** -0.5,
                                                  max_context=TOKENS, splits=splits, **options))
            assert torch.isfinite(found[0]).all()
            for page_tokens, out in zip((32, 64, 128), found[1:]):
                assert torch.equal(out, found[0]), (options, splits, page_tokens)


@pytest.mark.parametrize("size", [64, 128])
@pytest.mark.parametrize("group,kv_heads", [(4, 2), (20, 1)])
def test_rows_that_bring_their_own_key_do_not_depend_on_the_pages(size, group, kv_heads):
    from leone_amd import ops
    places = [0, 1, 31, 32, 64, 127, 200, 329]
    k, v = made(kv_heads, size, len(places))
    gen = torch.Generator().manual_seed(size + group)
    qkv = torch.randn(len(places), (group + 2) * kv_heads * size, generator=gen).to(DEV)
    gain = (1.0 + 0.1 * torch.randn(2, size, generator=gen)).to(DEV)
    positions = torch.tensor(places, dtype=torch.int32, device=DEV)
    rows = torch.arange(len(places), dtype=torch.int32, device=DEV)
    cos, sin = ops.rope_table(1e4, size, 512, DEV)
    for projection in (qkv.bfloat16(), torch.stack([0.5 * qkv, 0.25 * qkv, 0.25 * qkv])):
        for gains in (gain, gain.bfloat16()):
            for splits in (1, 4, 19):
                found = []
                for page_tokens in (16, 32, 64):
                    k_pool, v_pool, table = pools(k, v, page_tokens, page_tokens)
                    k_pool, v_pool = bits(k_pool), bits(v_pool)
                    out = ops.attention_decode_projected(projection, group * kv_heads, kv_heads, size, gains[0].contiguous(), gains[1].contiguous(),
                                                         1e-6, cos, sin, k_pool, v_pool, positions, rows, table, size ** -0.5,
                                                         max_context=TOKENS, splits=splits)
                    pages = [int(table[r, p // page_tokens]) for r, p in enumerate(places)]
                    new = [k_pool[page, :, :, p % page_tokens].float() for page, p in zip(pages, places)]
                    found.append((out, torch.stack(new)))
                assert torch.isfinite(found[0][0]).all()
                for out, new in found[1:]:
                    assert torch.equal(out, found[0][0]) and torch.equal(new, found[0][1])


def test_rows_that_bring_their_own_key_are_cut_by_the_rule():
    """How many parts a row's keys are cut into decides in which order their results are added: the projected call's own number is
    ``choose_splits``'s, as it is for ``attention_decode``."""
    from leone_amd import ops
    heads, size, context = 8, 128, 2052
    gen = torch.Generator().manual_seed(5)
    k, v = (torch.randn(1, context, heads, size, generator=gen) for _ in range(2))
    qkv = torch.randn(1, 6 * heads * size, generator=gen).bfloat16().to(DEV)
    found = []
    for splits in (None, ops.choose_splits(1, heads, 4, context, ops.compute_units(torch.device(DEV)))):
        k_pool, v_pool, table = pools(k, v, 64, 2)
        found.append(ops.attention_decode_projected(qkv, 4 * heads, heads, size, None, None, 1e-6, None, None, bits(k_pool), bits(v_pool),
                                                    torch.tensor([context - 1], dtype=torch.int32, device=DEV),
                                                    torch.zeros(1, dtype=torch.int32, device=DEV), table, size ** -0.5,
                                                    max_context=context, splits=splits))
    assert torch.equal(*found)


def test_a_key_without_a_page_spoils_the_rows_that_see_it():
    from leone_amd import ops
    k, v = made(2, 128, 3)
    for page_tokens in (16, 64):
        k_pool, v_pool, table = pools(k, v, page_tokens, page_tokens)
        table[1, 64 // page_tokens:128 // page_tokens] = -1
        q = torch.ones(3, 8 * 128, device=DEV).bfloat16()
        positions = torch.tensor([200, 200, 200], dtype=torch.int32, device=DEV)
        out = ops.attention_decode(q, bits(k_pool), bits(v_pool), positions, torch.arange(3, dtype=torch.int32, device=DEV), table, 8, 0.1,
                                   max_context=TOKENS, splits=2)
        assert bool(torch.isnan(out[1]).all()) and bool(torch.isfinite(out[[0, 2]]).all())


@pytest.mark.parametrize("size", [16, 64, 80, 112, 128, 144, 256])
@pytest.mark.parametrize("splits", [2, 7, 8, 9, 17, 32, 63, 64, 65])
def test_ranges_are_merged_whatever_their_number(size, splits):
    """Up to 64 ranges by lanes, more through shared memory, all of them with keys (66 tiles); the shorter rows leave empty ones."""
    from leone_amd import ops
    places = [0, 40, 329, 65 * 32 + 19]
    tokens = places[-1] + 1
    gen = torch.Generator().manual_seed(3)
    k, v = [torch.randn(len(places), tokens, 2, size, generator=gen).bfloat16().float() for _ in range(2)]
    k_pool, v_pool, table = pools(k, v, 64, 1)
    q = torch.randn(len(places), 6 * size, generator=torch.Generator().manual_seed(1)).bfloat16().to(DEV)
    args = (q, bits(k_pool), bits(v_pool), torch.tensor(places, dtype=torch.int32, device=DEV),
            torch.arange(len(places), dtype=torch.int32, device=DEV), table, 6, size ** -0.5)
    whole = ops.attention_decode(*args, max_context=tokens, splits=1).float()
    cut = ops.attention_decode(*args, max_context=tokens, splits=splits).float()
    # the weights are the same numbers however the keys are cut; sums in another order round once more to bfloat16, row by row
    assert bool(((whole - cut).abs().amax(1) <= 2.0 ** -7 * whole.abs().amax(1)).all())


@pytest.mark.parametrize("hidden", [4, 6, 64, 1000, 1023, 4096])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_embedding_in_fours_and_element_by_element(hidden, dtype):
    from leone_amd import ops
    room = torch.randn(50 * hidden + 8, device=DEV).to(dtype)
    tokens = torch.tensor([0, 49, 7, 7], dtype=torch.int32, device=DEV)
    for shift in (0, 1, 4):
        table = room[shift:shift + 50 * hidden].view(50, hidden)
        assert torch.equal(ops.embed(table, tokens), table[tokens.long()].float())
