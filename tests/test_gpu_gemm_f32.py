"""The single-precision product: both kernels, their tiles' edges, the cut of the inner size, operands off 16 bytes."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def worst(m, n, k, shift=0, seed=1):
    """The largest error of the product over what its sums can be off by (``shift``: elements the operands are moved by)."""
    from leone_amd import ops
    gen = torch.Generator(device=DEV).manual_seed(seed)
    a = torch.randn(m * k + shift, generator=gen, device=DEV)[shift:].view(m, k)
    b = torch.randn(n * k + shift, generator=gen, device=DEV)[shift:].view(n, k)
    got = ops.gemm_f32(a, b)
    want = a.double() @ b.double().T
    # every product and every addition of a chain of k is off by at most 2^-24 of the running sum's size, whose root mean
    # square is sqrt(k); the errors add up like a random walk, and none of so many is beyond eight times its deviation
    bound = 8.0 * 2.0 ** -24 * math.sqrt(k) * math.sqrt(k + math.log2(k + 1))
    return float((got.double() - want).abs().max()) / bound


# rows: every number of row tiles of the streaming kernel and its edges, then the tiled kernel with both tiles; columns off 16
# and 64; inner sizes below a run, off a run, off 4, and long enough to be cut
@pytest.mark.parametrize("m", [1, 2, 15, 16, 17, 32, 33, 63, 64, 65, 127, 130, 777])
@pytest.mark.parametrize("n,k", [(16, 8), (17, 60), (96, 64), (130, 333), (2048, 512), (520, 2052), (1536, 6144)])
def test_sizes(m, n, k):
    assert worst(m, n, k) < 1.0


def test_many_tiles():
    assert worst(1500, 6144, 256) < 1.0 and worst(1025, 8200, 100) < 1.0


@pytest.mark.parametrize("m", [3, 40, 200])
def test_operands_off_sixteen_bytes(m):
    assert worst(m, 100, 512, shift=1) < 1.0 and worst(m, 100, 512, shift=3) < 1.0


def test_rows_do_not_depend_on_their_neighbours():
    """A row that holds infinities and NaN spoils its own results only."""
    from leone_amd import ops
    for m, n, k in ((5, 70, 96), (130, 70, 1000)):
        a, b = torch.randn(m, k, device=DEV), torch.randn(n, k, device=DEV)
        clean = ops.gemm_f32(a, b)
        a[1, 3], a[2, k - 1] = math.inf, math.nan
        spoilt = ops.gemm_f32(a, b)
        keep = [i for i in range(m) if i not in (1, 2)]
        assert torch.equal(clean[keep], spoilt[keep])
        assert bool(torch.isinf(spoilt[1]).all()) and bool(torch.isnan(spoilt[2]).all())


@pytest.mark.parametrize("n,k", [(40, 200), (96, 256), (70, 333), (512, 512), (100, 1000), (530, 2052), (2048, 2048), (256, 6144)])
def test_a_row_is_the_same_whatever_rows_are_beside_it(n, k):
    """To the bit, over both kernels, their tiles and cuts of K, and whether the operands are aligned."""
    from leone_amd import ops
    gen = torch.Generator(device=DEV).manual_seed(k)
    a, b = torch.randn(1024, k, generator=gen, device=DEV), torch.randn(n, k, generator=gen, device=DEV)
    alone = torch.cat([ops.gemm_f32(a[i:i + 1].contiguous(), b) for i in (0, 1, 15)])
    for m in (16, 17, 32, 33, 64, 65, 128, 200, 300, 777, 1024):
        together = ops.gemm_f32(a[:m].contiguous(), b)
        assert torch.equal(together[[0, 1, 15]], alone), m
        moved = torch.empty(m * k + 1, device=DEV)[1:].view(m, k).copy_(a[:m])
        assert torch.equal(ops.gemm_f32(moved, b), together), m


@pytest.mark.parametrize("n,k", [(33, 257), (40, 511), (40, 520), (40, 545), (96, 577), (16401, 512), (16400, 515), (16392, 2048), (8200, 2084)])
def test_few_rows_give_the_bits_of_many(n, k):
    """Two runs an instruction (up to eight rows) and two tiles a workgroup (many of them): ends of K off a pair of runs, a last tile
    alone, and rows whose sums are made again beside others."""
    from leone_amd import ops
    gen = torch.Generator(device=DEV).manual_seed(k)
    a, b = torch.randn(64, k, generator=gen, device=DEV), torch.randn(n, k, generator=gen, device=DEV)
    a[1, k - 1], a[4] = math.nan, 0.0
    a[5] *= 1e-36
    b[n - 1, 0], b[n - 2] = math.inf, 0.0
    many = ops.gemm_f32(a, b).nan_to_num(7.5, 8.5, 9.5)
    for m in (1, 2, 7, 8, 9, 16, 17):
        for shift in (0, 1):
            rows = torch.empty(m * k + shift, device=DEV)[shift:].view(m, k).copy_(a[:m])
            assert torch.equal(ops.gemm_f32(rows, b).nan_to_num(7.5, 8.5, 9.5), many[:m]), (m, shift)


def test_results_off_sixteen_bytes():
    """Where K is cut, the sum over its parts writes a result that lies anywhere."""
    from leone_amd import ops
    m, n, k = 40, 128, 2048
    assert ops.library().leone_gemm_f32_planes(m, n, k) > 1
    a, b = torch.randn(m, k, device=DEV), torch.randn(n, k, device=DEV)
    want = ops.gemm_f32(a, b)
    for shift in (1, 2, 3):
        room = torch.full((m * n + 8,), 7.0, device=DEV)
        ops.gemm_f32(a, b, out=room[shift:shift + m * n].view(m, n))
        assert torch.equal(room[shift:shift + m * n].view(m, n), want)
        assert bool((room[:shift] == 7.0).all()) and bool((room[shift + m * n:] == 7.0).all())


@pytest.mark.parametrize("m,n,k", [(1, 17, 257), (16, 129, 511), (33, 128, 513), (65, 130, 609), (200, 127, 1100), (70, 300, 2048)])
@pytest.mark.parametrize("scale", [1e-37, 1e-30, 1e-12, 1.0, 1e12])
def test_numbers_of_every_size(m, n, k, scale):
    """Numbers in three parts: none of their 24 bits is lost, whatever the size of A's numbers and wherever the row ends."""
    from leone_amd import ops
    gen = torch.Generator(device=DEV).manual_seed(n)
    a, b = torch.randn(m, k, generator=gen, device=DEV) * scale, torch.randn(n, k, generator=gen, device=DEV)
    want = a.double() @ b.double().T
    error = float((ops.gemm_f32(a, b).double() - want).norm() / want.norm())
    # a product that loses more than a float's last bit is off by 2^-24 of itself, at random; sums round as sums of floats do
    assert error < 2.0 ** -24 * (1.0 + math.sqrt(math.log2(k))), error


@pytest.mark.parametrize("m,n,k", [(1, 4096, 256), (16, 999, 513), (32, 2048, 2048), (200, 1001, 1001), (300, 512, 6144)])
def test_a_lone_product_is_rounded_as_a_float_product_is(m, n, k):
    """All that is left out of a product and lost on the way is below 2^-8 of a float's last bit: the product of both last parts (2^-32)
    and what the sums of the lower ones round."""
    from leone_amd import ops
    gen = torch.Generator(device=DEV).manual_seed(n)
    a, b = torch.zeros(m, k, device=DEV), torch.randn(n, k, generator=gen, device=DEV)
    at, value = torch.randint(0, k, (m,), generator=gen, device=DEV), torch.randn(m, generator=gen, device=DEV)
    a[torch.arange(m, device=DEV), at] = value
    want = value.double()[:, None] * b[:, at].double().T
    got = ops.gemm_f32(a, b)
    assert float(((got.double() - want) / want).abs().max()) < 2.0 ** -24 * (1.0 + 2.0 ** -7)
    assert float((got != want.float()).double().mean()) < 2.0 ** -7


# scales of A and B: below bfloat16's least number, 2^-133, a number's parts are lost, which counts where the other factor is large; the
# last two bring numbers that are no normal floats, and sums of products that are none
@pytest.mark.parametrize("m,n,k", [(1, 17, 257), (16, 129, 511), (33, 128, 513), (40, 130, 2048), (300, 127, 1100), (70, 300, 6144)])
@pytest.mark.parametrize("sizes", [(-110, 80), (80, -110), (-124, 70), (-122, 62), (62, -122), (-126, 100), (-70, -20), (-140, 100), (100, -140), (-75, -50)])
def test_small_numbers_against_large_ones(m, n, k, sizes):
    from leone_amd import ops
    gen = torch.Generator(device=DEV).manual_seed(n)
    a, b = (torch.randn(rows, k, generator=gen, device=DEV) * 2.0 ** (size / 2) * 2.0 ** (size / 2) for rows, size in zip((m, n), sizes))
    want = a.double() @ b.double().T
    got = ops.gemm_f32(a, b)
    # as in test_numbers_of_every_size; a product or a sum below the least normal float is off by half of 2^-149 at most
    bound = 2.0 ** -24 * (1.0 + math.sqrt(math.log2(k))) * float(want.norm()) + 2.0 ** -150 * (2 * k) * math.sqrt(m * n)
    assert float((got.double() - want).norm()) < bound
    alone = torch.cat([ops.gemm_f32(a[i:i + 1].contiguous(), b) for i in (0, m - 1)])
    assert torch.equal(got[[0, m - 1]], alone)             # whether a sum is made again is its own two rows' matter


@pytest.mark.parametrize("m", [3, 40, 300])
def test_a_lone_small_number_against_a_large_one(m):
    """2^-140 x 2^100 is an ordinary number, and so is what a row holds of both kinds; rows of zeros give zeros."""
    from leone_amd import ops
    n, k = 140, 600
    a, b = torch.zeros(m, k, device=DEV), torch.zeros(n, k, device=DEV)
    a[0, 5], b[:, 5] = 2.0 ** -140, 2.0 ** 100
    a[1, 7], b[:, 7] = 1.2345678 * 2.0 ** -126, 2.0 ** 100
    a[2, 7], a[2, 590] = 2.0 ** -120 * (1 + 2.0 ** -14), -1.5 * 2.0 ** -60
    b[:, 590] = 3.0 * 2.0 ** 40
    got = ops.gemm_f32(a, b)
    assert bool((got[0] == 2.0 ** -40).all()) and not bool(got[3:].any())
    assert torch.equal(got[1], (a[1, 7] * 2.0 ** 100).expand(n))
    assert torch.equal(got[2], (a[2, 7].double() * 2.0 ** 100 - 4.5 * 2.0 ** -20).float().expand(n))


def test_numbers_that_are_no_sums_of_parts():
    """The largest numbers round to infinity in 16 bits and an infinity has nothing left over: plain sums all the same."""
    from leone_amd import ops
    for m, n, k in ((3, 20, 300), (40, 140, 600), (300, 70, 512)):
        a, b = torch.zeros(m, k, device=DEV), torch.randn(n, k, device=DEV)
        a[0, 5], a[1, k - 1], a[2, 7] = 3.4e38, -3.4028234e38, math.inf
        b[:, 5] = b[:, k - 1] = 0.25
        b[:, 7] = 1.0 + 2.0 ** -20
        b[3, 7] = 0.0
        got = ops.gemm_f32(a, b)
        assert torch.equal(got[0], torch.full_like(got[0], 3.4e38) * 0.25)
        assert torch.equal(got[1], torch.full_like(got[1], -3.4028234e38) * 0.25)
        keep = [j for j in range(n) if j != 3]
        assert bool((got[2, keep] == math.inf).all()) and bool(torch.isnan(got[2, 3])) and not bool(got[3:].any())


@pytest.mark.parametrize("m,n,k", [(1, 2048, 2048), (24, 3072, 512), (200, 3072, 2048)])
def test_rows_that_are_no_numbers_do_not_hold_up_a_launch(m, n, k):
    """What it costs beside the product of ordinary numbers is bounded: such sums are made by the float instructions (measured 1.0 to 1.7
    times, of all rows 1.0 to 3.6; a loop over K for each of them was 1.0 to 9 times, of all rows 12 to 92)."""
    from leone_amd import ops
    a, b = torch.randn(m, k, device=DEV), torch.randn(n, k, device=DEV)
    spoilt = torch.full_like(a, math.nan)

    def took(x):
        best = math.inf
        for _ in range(5):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(50):
                ops.gemm_f32(x, b)
            end.record()
            end.synchronize()
            best = min(best, start.elapsed_time(end))
        return best

    took(a)
    assert took(spoilt) < 8.0 * took(a)


@pytest.mark.parametrize("n,k", [(16, 256), (48, 511), (144, 520), (1040, 1024), (96, 255), (3072, 2048)])
def test_gates_and_ups_in_the_products_own_launch(n, k):
    """To the bit what the product and the activation behind it give, in every kernel, also where K is cut or too short."""
    from leone_amd import ops
    b = torch.randn(n, k, device=DEV) / math.sqrt(k)
    for m in (1, 5, 16, 17, 33, 64, 130, 300):
        a = torch.randn(m, k, device=DEV)
        for options in ({}, {"activation": "gelu_tanh"}, {"activation": "clamped_swish", "limit": 0.5}):
            assert torch.equal(ops.gemm_f32_glu(a, b, **options), ops.swiglu(ops.gemm_f32(a, b), **options)), (m, options)
    a[0, 3], a[1, 5] = math.inf, math.nan
    got, want = ops.gemm_f32_glu(a, b), ops.swiglu(ops.gemm_f32(a, b))
    assert torch.equal(torch.nan_to_num(got, 1.0, 2.0, 3.0), torch.nan_to_num(want, 1.0, 2.0, 3.0))
