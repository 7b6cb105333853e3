"""Float attention on the matrix instructions against the kernel for any shape: the same rows over the same cache, once in
pages of 8 tokens (which only the latter takes) and once in pages of 16 and more."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def pools(k, v, page_tokens, seed):
    """k, v [requests, tokens, kv_heads, size] in pages that lie anywhere, pages of the pool nobody holds and places behind a
    request's end full of NaN; the block table [requests, blocks]."""
    from leone_amd import ops
    requests, tokens, heads, size = k.shape
    blocks = -(-tokens // page_tokens)
    places = torch.randperm(requests * blocks + 3, generator=torch.Generator().manual_seed(seed))[:requests * blocks].view(requests, blocks)
    out = []
    for t, pack in ((k, ops.pack_keys), (v, ops.pack_values)):
        filled = torch.full((requests, blocks * page_tokens, heads, size), float("nan"))
        filled[:, :tokens] = t
        pages = torch.full((requests * blocks + 3, heads, page_tokens, size), float("nan"))
        pages[places.reshape(-1)] = filled.view(requests, blocks, page_tokens, heads, size).transpose(2, 3).reshape(-1, heads, page_tokens, size)
        out.append(pack(pages).to(DEV))
    return out[0], out[1], places.to(torch.int32).to(DEV)


def both(rows, group, kv_heads, size, tokens=150, spoil=None, unmapped=None, **options):
    """``rows``: (request, position) of every row.  Results of the two kernels, pages of 16, 64 and 48 (no power of two) the second."""
    from leone_amd import ops
    gen = torch.Generator().manual_seed(17)
    requests = 1 + max(r for r, _ in rows)
    k, v = torch.randn(requests, tokens, kv_heads, size, generator=gen), torch.randn(requests, tokens, kv_heads, size, generator=gen)
    for request, position, value in spoil or []:
        v[request, position, 0, 5] = value
    q = (2.0 * torch.randn(len(rows), group * kv_heads * size, generator=gen)).to(DEV)
    entry = torch.tensor([r for r, _ in rows], dtype=torch.int32, device=DEV)
    positions = torch.tensor([p for _, p in rows], dtype=torch.int32, device=DEV)
    results = []
    for page_tokens in (8, 16, 64, *(() if unmapped else (48,))):          # (64 positions that are gone are no whole pages of 48)
        k_pool, v_pool, table = pools(k, v, page_tokens, page_tokens)
        for request, position in unmapped or []:        # 64 positions are gone, whatever the pages' size
            table[request, position // page_tokens:(position + 64) // page_tokens] = -1
        results.append(ops.attention_rows(q, k_pool, v_pool, positions, entry, table, group * kv_heads, size ** -0.5, **options))
    return results


def agree(results):
    for out in results[1:]:
        assert torch.equal(torch.isnan(out), torch.isnan(results[0])) and torch.equal(torch.isinf(out), torch.isinf(results[0]))
        fine = torch.isfinite(out)
        # each sums at most 150 weights of at most 1 in its own order, and rounds scores of up to 40 to 2e-6 of their weight
        assert float((out - results[0])[fine].abs().max()) < 2e-5


# single rows of different requests, a portion, portions cut where tiles of rows begin and end, and all of them in one step
DECODE = [(i, p) for i, p in enumerate((0, 1, 15, 16, 17, 63, 64, 149))]
PORTION = [(0, p) for p in range(100)]
MIXED = [(0, p) for p in range(3, 40)] + [(1, p) for p in range(90, 149)] + [(2, 149), (3, 7), (4, 0)] + [(5, p) for p in range(2)]


@pytest.mark.parametrize("size", [64, 128])
@pytest.mark.parametrize("group,kv_heads", [(1, 3), (3, 2), (4, 1), (16, 1)])
@pytest.mark.parametrize("rows", [DECODE, PORTION, MIXED, MIXED * 9], ids=["single", "portion", "mixed", "many"])
def test_both_kernels_agree(rows, group, kv_heads, size):
    if len(rows) > 800:                 # enough rows for the kernel with fewer waves: as many requests more
        rows = [(r + 6 * copy, p) for copy in range(9) for r, p in MIXED]
    agree(both(rows, group, kv_heads, size))


@pytest.mark.parametrize("options", [dict(window=20), dict(window=33, keep_first=5), dict(window=1, keep_first=40), dict(chunk=24),
                                     dict(query_factor=(0.3, 10))], ids=str)
def test_masks_and_factors(options):
    agree(both(MIXED, 4, 2, 128, **options))
    agree(both(DECODE, 2, 2, 64, **options))


def test_shapes_of_scores_and_gates():
    from leone_amd import ops
    heads, size, n = 8, 128, len(MIXED)
    gen = torch.Generator().manual_seed(3)
    angle = torch.rand(150, size // 2, generator=gen)
    cos, sin = angle.cos().to(DEV), angle.sin().to(DEV)
    sinks, slopes = torch.linspace(-2, 5, heads).to(DEV), torch.linspace(0, 0.5, heads).to(DEV)
    wide = torch.randn(n, heads * size + 4, generator=gen).to(DEV)
    for shape in (ops.ScoreShape(4.0), ops.ScoreShape(None, sinks), ops.ScoreShape(None, None, (cos, sin, "half_split")),
                  ops.ScoreShape(9.0, sinks, (cos, sin, "adjacent"))):
        agree(both(MIXED, 4, 2, size, shape=shape))
        agree(both(MIXED, 4, 2, size, shape=shape, slopes=slopes, gate=wide[:, 4:], gate_each=True, window=30))
        agree(both(MIXED, 4, 2, size, shape=shape, gate=wide[:, 4:4 + heads]))


def test_what_is_not_finite_stays_with_the_rows_that_see_it():
    inf, nan = float("inf"), float("nan")
    agree(both(MIXED, 4, 2, 64, spoil=[(0, 20, nan), (1, 100, inf), (1, 101, -inf), (2, 149, inf), (3, 8, nan)]))
    agree(both(MIXED, 4, 2, 64, unmapped=[(0, 0), (1, 64)], window=25))


@pytest.mark.parametrize("options", [dict(), dict(window=20), dict(window=33, keep_first=5), dict(window=130, keep_first=40), dict(chunk=24)], ids=str)
@pytest.mark.parametrize("size,group,kv_heads", [(64, 1, 3), (64, 4, 2), (128, 3, 2), (128, 16, 1)])
def test_a_row_is_the_same_whatever_rows_are_beside_it(size, group, kv_heads, options):
    """To the bit: each row alone, the rows of a step, and enough rows that other launches are taken; with values that are not finite
    behind some of them as well."""
    rows = [(r + 6 * copy, p) for copy in range(8) for r, p in MIXED]
    for spoil in (None, [(0, 20, float("nan")), (1, 145, float("inf"))]):
        many = both(rows, group, kv_heads, size, spoil=spoil, **options)
        # the rows' queries and requests' keys are made in order, so those of fewer rows have to be cut out of the many
        gen = torch.Generator().manual_seed(17)
        requests = 1 + max(r for r, _ in rows)
        k, v = (torch.randn(requests, 150, kv_heads, size, generator=gen) for _ in range(2))
        for request, position, value in spoil or []:
            v[request, position, 0, 5] = value
        q = (2.0 * torch.randn(len(rows), group * kv_heads * size, generator=gen)).to(DEV)
        from leone_amd import ops
        k_pool, v_pool, table = pools(k, v, 16, 16)
        for chosen in (range(len(MIXED)), range(5, 30), [0], [3], [40], [95], [99]):
            chosen = list(chosen)
            got = ops.attention_rows(q[chosen].contiguous(), k_pool, v_pool, torch.tensor([rows[i][1] for i in chosen], dtype=torch.int32, device=DEV),
                                     torch.tensor([rows[i][0] for i in chosen], dtype=torch.int32, device=DEV), table, group * kv_heads,
                                     size ** -0.5, **options)
            assert torch.equal(got.nan_to_num(7e7), many[1][chosen].nan_to_num(7e7)), chosen[:3]
