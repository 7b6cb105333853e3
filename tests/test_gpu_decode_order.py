"""Decoding with more workgroups than compute units: rows of every length, taken longest first or in pairs, come out where they
belong; and the row's own key and value at every place of a tile, whatever the cache holds there."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def projected(lengths, kv_heads, group, dim, planes, splits, seed=0):
    """(results of ``attention_decode_projected``, of the same rows one by one), the cache's places for the new tokens NaN."""
    from leone_amd import ops
    gen = torch.Generator(device=DEV).manual_seed(seed)
    rows, blocks = len(lengths), max(lengths) // 32 + 1
    table = torch.randperm(rows * blocks, generator=gen, device=DEV).view(rows, blocks).to(torch.int32)
    k = torch.randn(rows * blocks, kv_heads, dim // 8, 32, 8, generator=gen, device=DEV).bfloat16()
    v = torch.randn(rows * blocks, kv_heads, 4, dim, 8, generator=gen, device=DEV).bfloat16()
    positions = torch.tensor([n - 1 for n in lengths], dtype=torch.int32, device=DEV)
    for r, n in enumerate(lengths):
        page, at = int(table[r, (n - 1) // 32]), (n - 1) % 32
        k[page, :, :, at:] = float("nan")
        v[page, :, at // 8, :, at % 8:] = float("nan")
        v[page, :, at // 8 + 1:] = float("nan")
    heads = kv_heads * group
    width = (heads + 2 * kv_heads) * dim
    qkv = torch.randn(planes, rows, width, generator=gen, device=DEV) if planes else torch.randn(rows, width, generator=gen, device=DEV).bfloat16()
    gains = [1 + 0.1 * torch.randn(dim, generator=gen, device=DEV) for _ in range(2)]
    cos, sin = ops.rope_table(1e4, dim, max(lengths), DEV)
    entry = torch.arange(rows, dtype=torch.int32, device=DEV)

    def run(pick, splits):
        pools = k.clone(), v.clone()
        q = (qkv[:, pick] if planes else qkv[pick]).contiguous()
        out = ops.attention_decode_projected(q, heads, kv_heads, dim, *gains, 1e-6, cos, sin, *pools, positions[pick].contiguous(),
                                             entry[:len(pick)], table[pick].contiguous(), dim ** -0.5, max_context=max(lengths), splits=splits)
        return out, pools
    out, pools = run(list(range(rows)), splits)
    alone = [run([r], splits) for r in range(rows)]
    for r, n in enumerate(lengths):
        page, at = int(table[r, (n - 1) // 32]), (n - 1) % 32
        assert torch.equal(pools[0][page, :, :, at], alone[r][1][0][page, :, :, at]) and bool(torch.isfinite(pools[0][page, :, :, at].float()).all())
        assert torch.equal(pools[1][page, :, at // 8, :, at % 8], alone[r][1][1][page, :, at // 8, :, at % 8])
    return out, torch.cat([a[0] for a in alone])


# one workgroup a unit, two (paired), more (longest first), up to and past the rows that are ranked; equal rows
@pytest.mark.parametrize("rows,kv_heads", [(3, 1), (40, 8), (64, 8), (65, 5), (128, 8), (129, 4)])
@pytest.mark.parametrize("splits", [1, 3])
def test_rows_come_out_where_they_belong(rows, kv_heads, splits):
    gen = torch.Generator().manual_seed(rows)
    lengths = torch.randint(1, 200, (rows,), generator=gen).tolist()
    lengths[rows // 2:rows // 2 + 2] = [77] * len(lengths[rows // 2:rows // 2 + 2])
    got, want = projected(lengths, kv_heads, 2, 64, 0, splits)
    assert torch.equal(got, want)


@pytest.mark.parametrize("planes", [0, 1, 3, 7])
@pytest.mark.parametrize("dim,group", [(64, 1), (128, 4), (128, 16), (128, 17), (256, 3)])
def test_the_rows_own_key_at_every_place_of_a_tile(dim, group, planes):
    """What the cache held there before (NaN) must not come through; every row as it comes out alone."""
    lengths = list(range(1, 34)) + [63, 64, 65, 96, 97, 128, 129, 150]
    for splits in (1, 2):
        got, want = projected(lengths, 2, group, dim, planes, splits, seed=dim)
        assert bool(torch.isfinite(got.float()).all()) and torch.equal(got, want)


# ranked: up to two workgroups a unit and lengths more than 1,024 apart; one key less and it is not
@pytest.mark.parametrize("rows,kv_heads", [(33, 8), (64, 8), (65, 5), (128, 4)])
def test_rows_of_very_different_lengths(rows, kv_heads):
    gen = torch.Generator().manual_seed(rows)
    lengths = torch.randint(2, 1100, (rows,), generator=gen).tolist()
    lengths[rows // 2:rows // 2 + 2] = [77, 77]
    for longest in (1024, 1025, 1200):
        lengths[0], lengths[-1] = longest, 1
        lengths[1:-1] = [min(n, longest) for n in lengths[1:-1]]
        got, want = projected(lengths, kv_heads, 2, 64, 0, 1)
        assert torch.equal(got, want)
