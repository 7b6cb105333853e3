"""What the attention of decoded tokens writes into the cache when it makes the new key itself."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("planes", [1, 3])
@pytest.mark.parametrize("dim", [64, 128])
def test_new_keys_are_those_of_the_separate_kernel(dim, planes):
    """The same bits whichever of the two kernels wrote a key, over 16,384 heads: with the squares of a head added in another order
    about one key in 3,000 rounds to another bfloat16 element, which a few heads do not show."""
    from leone_amd import ops
    q_heads, kv_heads, page, rows = 8, 8, 16, 128
    gen = torch.Generator(device=DEV).manual_seed(dim + planes)
    rand = lambda *size: torch.randn(*size, generator=gen, device=DEV)
    table = torch.arange(rows, dtype=torch.int32, device=DEV).view(rows, 1)
    entry = torch.arange(rows, dtype=torch.int32, device=DEV)
    cos, sin = ops.rope_table(1e6, dim, 64, DEV)
    width = (q_heads + 2 * kv_heads) * dim
    for _ in range(16):
        positions = torch.randint(0, page, (rows,), generator=gen, device=DEV, dtype=torch.int32)
        qkv = rand(rows, width).bfloat16() if planes == 1 else rand(planes, rows, width) * torch.tensor([1.0, 0.02, 3e-4], device=DEV).view(3, 1, 1)
        q_gain, k_gain = ((1 + 0.1 * rand(dim)).bfloat16() for _ in range(2))
        k_pool, v_pool = rand(rows, kv_heads, dim // 8, page, 8).bfloat16(), rand(rows, kv_heads, page // 8, dim, 8).bfloat16()
        k_apart, v_apart = k_pool.clone(), v_pool.clone()
        ops.qk_norm_rope_write(qkv, q_heads, kv_heads, dim, q_gain, k_gain, 1e-6, cos, sin, positions, entry, table, k_apart, v_apart,
                               out_dtype=torch.bfloat16)
        ops.attention_decode_projected(qkv, q_heads, kv_heads, dim, q_gain, k_gain, 1e-6, cos, sin, k_pool, v_pool, positions, entry, table,
                                       dim ** -0.5, 0, max_context=page)
        assert torch.equal(k_pool, k_apart) and torch.equal(v_pool, v_apart)
