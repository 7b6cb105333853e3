"""Float products of few rows that norm their rows or add into the stream: the bits of the launches one by one."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def drawn(m, n, k, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    x, w = torch.randn(m, k, generator=gen, device=DEV) * 3.0, torch.randn(n, k, generator=gen, device=DEV) / math.sqrt(k)
    return x, w, 1.0 + 0.1 * torch.randn(k, generator=gen, device=DEV), torch.randn(m, n, generator=gen, device=DEV)


# inner sizes at both ends of every variant (four waves up to 511; whole rows of 512, 2,048 and 4,096; large matrices), ends of K off a
# pair of runs and off a segment; a last tile of a few columns, many workgroups
SIZES = [(4, 256), (13, 644), (2048, 576), (2049, 512), (16, 256), (40, 260), (96, 508), (512, 512), (48, 516), (1536, 1024), (530, 2044), (12288, 2048), (96, 2052), (33, 4092), (4096, 4096)]


@pytest.mark.parametrize("m", [1, 2, 5, 8])
@pytest.mark.parametrize("n,k", SIZES)
def test_the_same_bits(m, n, k):
    from leone_amd import ops
    x, w, gain, stream = drawn(m, n, k, m * n + k)
    normed = ops.NormedRows(x, gain, 1e-5, torch.float32)
    assert ops._folds_f32(normed, w, None, False) == (n * k <= ops.FOLDED_F32_NORM_ELEMENTS) and ops._folds_f32(x, w, stream, False)
    assert torch.equal(ops.gemm_f32_folded(normed, w), ops.gemm_f32(normed.materialize(), w))
    want = stream + ops.gemm_f32(x, w)
    assert ops.linear(x, w, residual=stream) is None and torch.equal(stream, want)
    if n % 16 == 0:
        for activation, limit in (("silu", None), ("gelu_tanh", None), ("clamped_swish", 0.7)):
            got = ops.gemm_f32_folded(normed, w, None, True, activation, limit)
            assert torch.equal(got, ops.gemm_f32_glu(normed.materialize(), w, activation, limit))


@pytest.mark.parametrize("n,k", [(48, 300), (96, 516), (64, 2048), (8200, 2048)])
def test_rows_that_are_no_numbers_or_out_of_range(n, k):
    """Rows that hold NaN, infinities, the smallest and the largest numbers, zeros: as the launches one by one, and nobody else's."""
    from leone_amd import ops
    x, w, gain, stream = drawn(8, n, k, 5)
    x[1, 3], x[2, k - 1] = math.nan, math.inf
    x[3] *= 1e-38
    x[4] *= 1e37
    x[5] = 0.0
    w[n - 1, 0], w[n - 2] = math.inf, 0.0
    w[n - 3] *= 1e-36
    normed = ops.NormedRows(x, gain, 1e-12, torch.float32)
    got, want = ops.gemm_f32_folded(normed, w), ops.gemm_f32(normed.materialize(), w)
    assert torch.equal(got.nan_to_num(7.5, 8.5, 9.5), want.nan_to_num(7.5, 8.5, 9.5)) and bool(torch.isfinite(got[6:, :n - 1]).all())
    want = stream + ops.gemm_f32(x, w)
    ops.gemm_f32_folded(x, w, stream)
    assert torch.equal(stream.nan_to_num(7.5, 8.5, 9.5), want.nan_to_num(7.5, 8.5, 9.5))


def test_what_is_left_to_launches_of_their_own():
    """More rows, picked rows, gains of another type, sizes and addresses off: the results are those of the separate kernels."""
    from leone_amd import ops
    x, w, gain, stream = drawn(9, 96, 512, 3)
    odd = torch.empty(8 * 512 + 1, device=DEV)[1:].view(8, 512).copy_(x[:8])
    for normed in (ops.NormedRows(x, gain, 1e-5, torch.float32), ops.NormedRows(x[:8], gain.bfloat16(), 1e-5, torch.float32),
                   ops.NormedRows(x, gain, 1e-5, torch.float32, torch.tensor([4, 0], dtype=torch.int32, device=DEV))):
        assert not ops._folds_f32(normed, w, None, False)
        assert torch.equal(ops.linear(normed, w), ops.gemm_f32(normed.materialize(), w))
    assert not ops._folds_f32(odd, w, stream[:8], False) and torch.equal(ops.linear(odd, w, residual=stream[:8]), ops.gemm_f32(odd, w))
    assert not ops._folds_f32(x, w, stream, False) and not ops._folds_f32(x[:8], w, stream.t()[:8], False)
    for n, k in ((96, 252), (96, 4100), (16400, 512)):
        x, w, gain, _ = drawn(2, n, k, 4)
        assert not ops._folds_f32(ops.NormedRows(x, gain, 1e-5, torch.float32), w, None, False)
    with pytest.raises(ops.KernelError):
        ops.gemm_f32_folded(x, w)


@pytest.mark.parametrize("n,k", [(1, 256), (7, 260), (9, 516), (40, 1000), (100, 2052), (2047, 640), (2048, 4100), (24, 6144)])
def test_eight_columns_a_workgroup_give_the_bits_of_many_rows(n, k):
    """Up to 2,048 columns and eight rows the instruction's columns are shared by two runs; ends of K off a pair of runs, columns off
    eight, columns and rows that are made again on the float instructions."""
    from leone_amd import ops
    gen = torch.Generator(device=DEV).manual_seed(n + k)
    a, b = torch.randn(64, k, generator=gen, device=DEV), torch.randn(n, k, generator=gen, device=DEV)
    a[1, k - 1], a[4] = math.nan, 0.0
    a[5] *= 1e-36
    b[n // 2] *= 1e30
    b[n - 1, k - 1] = math.inf
    many = ops.gemm_f32(a, b).nan_to_num(7.5, 8.5, 9.5)
    for m in (1, 3, 8):
        assert torch.equal(ops.gemm_f32(a[:m].contiguous(), b).nan_to_num(7.5, 8.5, 9.5), many[:m]), m


def test_a_product_is_not_added_into_what_it_reads():
    """The stream is the product's own operand, or overlaps it: the product comes back and the stream is as it was."""
    from leone_amd import ops
    x, w, _, _ = drawn(12, 512, 512, 6)
    kept = x.clone()
    for rows, stream in ((x[:8], x[:8]), (x[:8], x[2:10]), (x[3:8], x[:5])):
        want = ops.gemm_f32(rows, w)
        assert torch.equal(ops.linear(rows, w, residual=stream), want) and torch.equal(x, kept)
        with pytest.raises(ops.KernelError, match="made of"):
            ops.gemm_f32_folded(rows, w, stream)
    assert ops.linear(x[:4], w, residual=x[4:8]) is None and torch.equal(x[4:8], kept[4:8] + ops.gemm_f32(kept[:4], w))
    few = w[:8]                                            # the matrix itself
    assert torch.equal(ops.linear(kept[:8], w, residual=few), ops.gemm_f32(kept[:8], w))
    assert isinstance(ops.linear(kept[:8], w, residual=torch.zeros(8, 512)), torch.Tensor)          # a stream that lies elsewhere
