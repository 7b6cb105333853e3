"""Float attention with a workgroup for every share of a row's keys: to the bit what one workgroup a row and kv head gives, and the rule
between them."""
import pytest
import torch

from leone_amd import ops
from leone_amd.engine.engine import DECODE_BUCKET_MIN
from tests.test_gpu_attention_f32 import DEV, pools

pytestmark = pytest.mark.gpu
# one tile, whole and not; a round of four tiles a share (512 keys), one over; two rounds and a part; rows of one request side by side
ROWS = [(0, 0), (0, 15), (0, 16), (1, 127), (1, 128), (1, 511), (1, 512), (1, 513), (2, 1100), (2, 1151), (2, 1152)]


def both(rows, group, kv_heads, size, page_tokens, spoil=(), unmapped=(), **options):
    gen = torch.Generator().manual_seed(23)
    tokens = 1 + max(p for _, p in rows)
    requests = 1 + max(r for r, _ in rows)
    k, v = torch.randn(requests, tokens, kv_heads, size, generator=gen), torch.randn(requests, tokens, kv_heads, size, generator=gen)
    for request, position, value in spoil:
        v[request, position, 0, 5] = value
    q = (2.0 * torch.randn(len(rows), group * kv_heads * size, generator=gen)).to(DEV)
    entry = torch.tensor([r for r, _ in rows], dtype=torch.int32, device=DEV)
    positions = torch.tensor([p for _, p in rows], dtype=torch.int32, device=DEV)
    k_pool, v_pool, table = pools(k, v, page_tokens, page_tokens)
    for request, page in unmapped:
        table[request, page] = -1
    return [ops.attention_rows(q, k_pool, v_pool, positions, entry, table, group * kv_heads, size ** -0.5, shares=shares, **options)
            for shares in (False, True)]


def same(pair):
    one, two = pair
    assert torch.equal(torch.isnan(one), torch.isnan(two))
    assert torch.equal(one.nan_to_num(7e7, 8e7, -8e7), two.nan_to_num(7e7, 8e7, -8e7))


@pytest.mark.parametrize("size,group,kv_heads", [(64, 1, 3), (64, 4, 2), (128, 3, 2), (128, 4, 1), (128, 16, 1)])
@pytest.mark.parametrize("options", [dict(), dict(window=20), dict(window=700, keep_first=40), dict(window=1, keep_first=200), dict(chunk=600),
                                     dict(query_factor=(0.3, 10))], ids=str)
def test_the_same_bits(size, group, kv_heads, options):
    for page_tokens in (16, 48, 64):
        same(both(ROWS, group, kv_heads, size, page_tokens, **options))


def test_shapes_of_scores_and_gates():
    heads, size = 8, 128
    gen = torch.Generator().manual_seed(3)
    angle = torch.rand(1200, size // 2, generator=gen)
    cos, sin = angle.cos().to(DEV), angle.sin().to(DEV)
    sinks, slopes = torch.linspace(-2, 5, heads).to(DEV), torch.linspace(0, 0.5, heads).to(DEV)
    wide = torch.randn(len(ROWS), heads * size + 4, generator=gen).to(DEV)
    for shape in (None, ops.ScoreShape(4.0), ops.ScoreShape(None, sinks), ops.ScoreShape(None, None, (cos, sin, "half_split")),
                  ops.ScoreShape(9.0, sinks, (cos, sin, "adjacent"))):
        same(both(ROWS, 4, 2, size, 64, shape=shape, slopes=slopes, gate=wide[:, 4:], gate_each=True, window=600))
        same(both(ROWS, 4, 2, size, 64, shape=shape, gate=wide[:, 4:4 + heads]))
    same(both(ROWS, 4, 2, 64, 64, shape=ops.ScoreShape(9.0, sinks, (cos[:, :32].contiguous(), sin[:, :32].contiguous(), "half_split"))))


def test_values_that_are_not_finite_and_pages_that_are_gone():
    inf, nan = float("inf"), float("nan")
    for size in (64, 128):
        same(both(ROWS, 4, 2, size, 64, spoil=[(0, 20, nan), (1, 100, inf), (1, 514, nan), (2, 1101, -inf)]))
        same(both(ROWS, 4, 2, size, 64, unmapped=[(1, 1), (2, 17)], window=500))


def test_more_tiles_than_a_wave_has_lanes():
    """Page numbers come 64 tiles of a share at a time: 8,192 keys and more."""
    same(both([(0, 8191), (0, 8192), (0, 8800)], 4, 1, 128, 64))
    same(both([(0, 8800)], 2, 1, 64, 16, window=8300, keep_first=30))


def test_the_rule():
    assert not any(ops.f32_attention_shares(rows, kv, size, 0) for rows in (1, 4) for kv in (1, 8) for size in (64, 128))
    for size in (64, 128):
        taken = [[ops.f32_attention_shares(units, 1, size, keys) for keys in (16, 128, 256, 512, 1024, 4096, 1 << 20)] for units in (1, 8, 16, 32, 64, 128, 4096)]
        assert all(line == sorted(line) for line in taken) and not any(taken[-1])          # more keys: rather; more rows: rather not
        assert all(column == sorted(column, reverse=True) for column in map(list, zip(*taken)))
    # steps of a few tokens' context are recorded for the first range, whose end says nothing of theirs
    assert not any(ops.f32_attention_shares(units, 1, size, DECODE_BUCKET_MIN) for units in (1, 4, 16, 64) for size in (64, 128))
    assert ops.f32_attention_shares(16, 1, 128, 2 * DECODE_BUCKET_MIN)
