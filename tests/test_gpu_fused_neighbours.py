"""Few rows: the square behind a product and the rounding ahead of a pair of products, in the products' launches, to the bit what launches of
their own give."""
import pytest
import torch

from leone_amd import ops

pytestmark = pytest.mark.gpu


def some(*shape, seed=1):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed + sum(shape))).cuda()


@pytest.mark.parametrize("rows", [1, 2, 15, 16, 17, 40])
@pytest.mark.parametrize("n,k", [(16, 8), (40, 72), (256, 128), (1000, 1088), (4096, 64)])
def test_the_square_behind_a_product(rows, n, k):
    x, w = some(rows, k).bfloat16(), some(n, k, seed=2).bfloat16()
    x[0, 0] = float("nan")
    if rows > 1:
        x[1, 0], x[-1, 1] = float("inf"), 3e38
    for copied in (False, True):
        if copied:
            ops.keep_streamed_copy(w)
        assert torch.equal(ops.linear_relu_squared(x, w), ops.relu_squared(ops.linear(x, w)))
    ops.drop_streamed_copies()
    normed = ops.NormedRows(some(rows, k, seed=3), some(k).bfloat16(), 1e-5, torch.bfloat16)
    assert torch.equal(ops.linear_relu_squared(normed, w), ops.relu_squared(ops.linear(normed, w)))
    assert torch.equal(ops.linear_relu_squared(x.float(), w.float()).nan_to_num(1.5), ops.relu_squared(ops.linear(x.float(), w.float())).nan_to_num(1.5))


@pytest.mark.parametrize("rows", [1, 7, 16, 17, 130])
@pytest.mark.parametrize("parts,k", [((32, 32), 8), ((48, 48), 72), ((128, 64), 128), ((64, 128), 64), ((24, 24), 16), ((64, 64, 48), 64)])
def test_rounding_ahead_of_products_side_by_side(rows, parts, k):
    w = some(sum(parts), k, seed=4).bfloat16()
    wide = some(rows, 8 + len(parts) * k + 3, seed=5)
    even = some(rows, 8 + len(parts) * k + 4, seed=6)
    for proj, first in ((wide, 8), (even, 8), (even, 5), (even, 4)):          # rows and first columns that are 16-byte runs, and not
        x = proj[:, first:first + len(parts) * k].unflatten(1, (len(parts), k)).transpose(0, 1)
        want = ops.linear_planes(x.bfloat16().contiguous(), w, parts)
        got = ops.linear_planes_of_floats(x, w, parts)
        assert len(got) == len(want) and all(torch.equal(a, b) for a, b in zip(got, want))


def test_floats_that_lie_elsewhere_are_refused():
    """The kernel gets no address that the device does not have: what is on the host is refused, as by ``linear_planes``."""
    w = some(64, 32, seed=7).bfloat16()
    with pytest.raises(ops.KernelError, match="on cpu"):
        ops.linear_planes_of_floats(some(2, 3, 32, seed=8).cpu(), w, [32, 32])
