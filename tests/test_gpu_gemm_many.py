"""Products of more rows than the weight-streaming kernels take, from the weight's tiled copy (``gemm_many``): every tile and output at the edges
of tiles, stages and ranges of K, against 64 bits; and the rule that hands products to it."""
import pytest
import torch

from leone_amd import ops

pytestmark = pytest.mark.gpu
TILES = [plan[:2] for plan in ops.MANY_TILES]


def _operands(m, n, k):
    gen = torch.Generator().manual_seed(m * 7 + n * 3 + k)
    x = torch.randn((m, k), generator=gen).bfloat16().cuda()
    weight = (torch.randn((n, k), generator=gen) / k ** 0.5).bfloat16().cuda()
    want = x.double() @ weight.double().t()
    # a float sum of k products is off by at most (k + 1) units of 2^-24 of the sum of their sizes (its planes' sum by a few more)
    bound = (k + 8) * 2.0 ** -24 * (x.double().abs() @ weight.double().abs().t())
    return x, weight, ops.tile_weight(weight), want, bound


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("m, n, k, splits", [
    (1, 16, 64, 1),             # the smallest: one row, half a part, one stage
    (129, 272, 192, 3),         # one over tiles; one stage a range
    (191, 1040, 320, 2),        # odd stages, a last range that is shorter
    (256, 512, 448, 1),         # whole tiles of rows and columns
    (1153, 2064, 128, 1),       # more than eight rows of tiles
])
def test_every_tile_and_output(tile, m, n, k, splits):
    x, weight, tiles, want, bound = _operands(m, n, k)
    planes = ops.gemm_many(x, tiles, n, torch.float32, plan=(*tile, splits))
    assert planes.dtype == torch.float32 and tuple(planes.shape) == ((splits, m, n) if splits > 1 else (m, n))
    got = (planes.sum(dim=0) if splits > 1 else planes).double()
    assert ((got - want).abs() <= bound).all()
    whole = ops.gemm_many(x, tiles, n, torch.float32, plan=(*tile, 1))
    assert torch.equal(ops.gemm_many(x, tiles, n, plan=(*tile, 1)), whole.bfloat16())
    stream = torch.randn((m, n), generator=torch.Generator().manual_seed(5)).cuda()
    added = stream.clone()
    assert ops.gemm_many(x, tiles, n, residual=added, plan=(*tile, 1)) is None
    assert torch.equal(added, stream + whole)
    for activation, limit in (("silu", None), ("gelu_tanh", None), ("clamped_swish", 0.5)):
        both = ops.gemm_many(x, tiles, n, gated=True, plan=(*tile, 1), activation=activation, limit=limit)
        assert torch.equal(both, ops.swiglu(whole.bfloat16(), activation=activation, limit=limit))


def test_rows_beyond_the_matrices_are_not_written():
    m, n, k = 130, 144, 128
    x, weight, tiles, want, bound = _operands(m, n, k)
    for tile in TILES:
        held = torch.full((m + 2, n), 7.0, device="cuda")
        ops.gemm_many(x, tiles, n, residual=held[1:-1], plan=(*tile, 1))
        assert (held[0] == 7).all() and (held[-1] == 7).all()
        assert ((held[1:-1].double() - 7 - want).abs() <= bound + 2.0 ** -23 * (want.abs() + 7)).all()


@pytest.mark.parametrize("m, n, k", [(129, 1024, 1024), (300, 1040, 4096), (640, 3072, 1088), (300, 3600, 2112)])
def test_products_with_a_copy_take_it_and_agree_with_those_without(m, n, k):
    x, weight, tiles, want, bound = _operands(m, n, k)
    plain = ops.linear(x, weight, out_dtype=torch.float32)
    gated = ops.linear(x, weight, gated=True)
    try:
        ops.keep_streamed_copy(weight)
        assert (ops._takes_many(x, weight, torch.float32, None, False) is not None) == ops.many_pays(m, n, k, False, False) == (n != 1040)
        assert ((ops.linear(x, weight, out_dtype=torch.float32).double() - want).abs() <= bound).all()
        assert ((plain.double() - want).abs() <= bound).all()
        stream = torch.zeros((m, n), device="cuda")
        left = ops.linear(x, weight, residual=stream)
        if left is not None:                             # planes for the caller to add
            assert left.dim() == 3 and left.shape[0] == ops.many_plan(m, n, k, True)[2]
            stream = left.sum(dim=0)
        assert ((stream.double() - want).abs() <= bound).all()
        # what the product's own launch makes of gate and up is what a launch of its own makes of the rounded sums, which no tile changes
        half = ops.linear(x, weight, gated=True)
        taken = ops._takes_many(x, weight, torch.bfloat16, None, True) is not None
        assert taken == ops.many_pays(m, n, k, False, True)
        assert torch.equal(half, ops.swiglu(ops.gemm_many(x, tiles, n, plan=ops.many_plan(m, n, k, False))) if taken else gated)
        # what it does not take stays with the library: other layouts, other types, products being noted
        assert ops._takes_many(x[:, ::2], weight[:, :k // 2], torch.float32, None, False) is None
        assert ops._takes_many(x, weight, torch.float16, None, False) is None
        assert ops._takes_many(x, weight, torch.float16, torch.zeros((m, n), device="cuda"), False) is None
        assert ops._takes_many(x, weight, torch.float32, torch.zeros((n, m), device="cuda").t(), False) is None
        with ops.record_library_products() as seen:
            ops.linear(x, weight, out_dtype=torch.float32)
        assert len(seen.problems) == 1
    finally:
        ops.drop_streamed_copies()


@pytest.mark.parametrize("m, n, k, gated, takes", [
    (256, 1024, 4096, False, False), (174, 1216, 6912, False, False), (160, 2304, 1536, False, True), (512, 2304, 1536, False, True),
    (320, 4608, 3072, False, True), (129, 1024, 2048, False, True), (256, 1024, 2112, False, False), (640, 8192, 2048, False, True), (2048, 2560, 1536, False, True),
    (1024, 6144, 1024, False, True), (273, 1408, 4352, True, False), (200, 2816, 2048, True, True), (576, 8192, 2048, True, True), (420, 12288, 2048, True, True),
    (300, 1536, 3072, True, False),
])
def test_products_in_one_range_whose_workgroups_are_few_stay_with_the_library(m, n, k, gated, takes):
    """A workgroup walks all of K: where it is long and there are few, the library is ahead by more than the host saves with the copy.  Into
    the stream, where planes fill the units, the copy is taken."""
    x, weight = torch.randn((m, k), device="cuda").bfloat16(), (torch.randn((n, k), device="cuda") / k ** 0.5).bfloat16()
    kind = torch.bfloat16 if gated else torch.float32
    plain = ops.linear(x, weight, out_dtype=kind, gated=gated)
    try:
        ops.keep_streamed_copy(weight)
        assert (ops._takes_many(x, weight, kind, None, gated) is not None) == takes
        if not takes:
            assert torch.equal(ops.linear(x, weight, out_dtype=kind, gated=gated), plain)
        assert gated or m * n * k > ops.MANY_MOST or ops._takes_many(x, weight, kind, torch.zeros((m, n), device="cuda"), False) is not None
    finally:
        ops.drop_streamed_copies()


@pytest.mark.parametrize("tile", list(ops.DEEP_TILES))
@pytest.mark.parametrize("m, n, k, splits", [
    (1, 16, 64, 1),             # the smallest: one row, half a part, one stage of the four that are asked for ahead
    (17, 80, 256, 1),           # one turn of four stages, and no second
    (32, 144, 320, 1),          # a turn and one stage
    (33, 1040, 704, 2),         # ranges of six stages and five
    (64, 512, 960, 3),          # ranges of five stages
    (65, 272, 1984, 4),         # ranges of eight stages, the last of seven; a second row of the smaller tiles
    (128, 256, 512, 1),         # whole tiles, whole turns
])
def test_every_deep_tile_and_output(tile, m, n, k, splits):
    x, weight, tiles, want, bound = _operands(m, n, k)
    planes = ops.gemm_many(x, tiles, n, torch.float32, plan=(*tile, splits, True))
    got = (planes.sum(dim=0) if splits > 1 else planes).double()
    assert ((got - want).abs() <= bound).all()
    whole = ops.gemm_many(x, tiles, n, torch.float32, plan=(*tile, 1, True))
    assert torch.equal(whole, ops.gemm_many(x, tiles, n, torch.float32, plan=(64, 128, 1)))       # the same sums as the other tiles
    assert torch.equal(ops.gemm_many(x, tiles, n, plan=(*tile, 1, True)), whole.bfloat16())
    stream = torch.randn((m, n), generator=torch.Generator().manual_seed(5)).cuda()
    added = stream.clone()
    assert ops.gemm_many(x, tiles, n, residual=added, plan=(*tile, 1, True)) is None
    assert torch.equal(added, stream + whole)
    gate, up = (p.reshape(m, n // 2).double() for p in whole.view(m, n // 16, 2, 8).unbind(2))
    for activation, limit in (("silu", None), ("gelu_tanh", None), ("clamped_swish", 0.5)):
        both = ops.gemm_many(x, tiles, n, gated=True, plan=(*tile, 1, True), activation=activation, limit=limit).double()
        if activation == "clamped_swish":
            low, held = gate.clamp(max=limit), up.clamp(-limit, limit)
            exact = low * torch.sigmoid(1.702 * low) * (held + 1.0)
        else:
            exact = (torch.nn.functional.silu(gate) if activation == "silu" else torch.nn.functional.gelu(gate, approximate="tanh")) * up
        # of the float sums, rounded once, at the end; of gelu's 1 + tanh, where that is small, float keeps a few 2^-24 of one
        cancelled = 2.0 ** -21 * (gate * up).abs() if activation == "gelu_tanh" else 0.0
        assert ((both - exact).abs() <= 2.0 ** -8 * exact.abs() * 1.01 + cancelled + 1e-30).all(), activation


@pytest.mark.parametrize("m, n, k", [(17, 1024, 1024), (64, 1040, 3072), (100, 3072, 1088), (128, 1024, 2048)])
def test_products_of_up_to_128_rows_take_the_copy(m, n, k):
    x, weight, tiles, want, bound = _operands(m, n, k)
    plain, gated = ops.linear(x, weight, out_dtype=torch.float32), ops.linear(x, weight, gated=True).double()
    assert ops._deep_choice(x, weight, torch.float32, None, False, False) is None                  # there is none yet
    try:
        ops.keep_streamed_copy(weight)
        assert ops._deep_choice(x, weight, torch.float32, None, False, False) is not None
        for got in (plain, ops.linear(x, weight, out_dtype=torch.float32)):
            assert ((got.double() - want).abs() <= bound).all()
        for stream in (torch.zeros((m, n), device="cuda"), None):
            left = ops.linear(x, weight, torch.float32, residual=stream, planes_ok=True)
            got = stream if left is None else left.sum(dim=0) if left.dim() == 3 else left
            assert left is None or left.dim() == 2 or left.shape[0] == ops.deep_plan(m, n, k, True, False)[2]
            assert ((got.double() - want).abs() <= bound).all()
        # the results of both round once, from sums that differ by their bounds at the most
        both = ops.linear(x, weight, gated=True).double()
        assert ((both - gated).abs() <= 2.0 ** -7 * both.abs() + 4 * bound.amax() * (1 + want.abs().amax())).all()
        assert ops._deep_choice(x[:, ::2], weight[:, :k // 2], torch.float32, None, False, False) is None
        assert ops._deep_choice(x[:16], weight, torch.float32, None, False, False) is None
        assert ops._deep_choice(x, weight, torch.float32, torch.zeros((n, m), device="cuda").t(), False, True) is None
        pieces = ops.linear_planes(torch.stack([x, x]), weight, [512, n - 512])
        assert ((torch.cat(pieces, 1).double() - want).abs() <= bound).all()
    finally:
        ops.drop_streamed_copies()


@pytest.mark.parametrize("m", [64, 300])
def test_a_copy_for_sums_in_their_old_order_is_left_alone_by_others(m):
    x, weight, tiles, want, bound = _operands(m, 1040, 1024)
    plain, parts = ops.linear(x, weight, out_dtype=torch.float32), ops.linear_planes(torch.stack([x, x]), weight, [16, 1024])
    try:
        ops.keep_streamed_copy(weight)
        held = ops.streamed_copy(weight)
        ops.keep_streamed_copy(weight, any_order=False)      # of a matrix that is kept in any order already: the stricter rule, the same copy
        ops.keep_streamed_copy(weight)
        assert ops.streamed_copy(weight) is held
        assert torch.equal(ops.linear(x, weight, out_dtype=torch.float32), plain)
        assert all(torch.equal(a, b) for a, b in zip(ops.linear_planes(torch.stack([x, x]), weight, [16, 1024]), parts))
    finally:
        ops.drop_streamed_copies()
