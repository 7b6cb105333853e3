"""How the delta rule's low-rank halves lie in memory."""
import pytest
import torch


@pytest.mark.parametrize("heads,dim,vdim,a_rank,g_rank", [(1, 6, 5, 3, 3), (3, 4, 4, 12, 12), (1, 6, 6, 8, 8), (2, 16, 16, 24, 24), (2, 16, 16, 8, 16)])
@pytest.mark.parametrize("kind", [torch.bfloat16, torch.float32])
def test_halves_begin_at_sixteen_bytes(heads, dim, vdim, a_rank, g_rank, kind):
    from leone_amd.parts.base import MIXERS, PartSpec
    hidden = 16
    names = {n: n for n in ("q", "k", "v", "b", "A_log", "dt_bias", "a1", "a2", "g1", "g2", "norm", "o", "q_conv", "k_conv", "v_conv")}
    mixer = MIXERS.build(PartSpec("channel_delta", {"hidden": hidden, "heads": heads, "kv_heads": heads, "dim": dim, "vdim": vdim, "taps": 4,
                                                    "eps": 1e-5, "a_rank": a_rank, "g_rank": g_rank, **names}))
    tensors = {spec.name: torch.randn(spec.shape).to(kind) for spec in mixer.tensor_specs()}
    a2, g2 = tensors["a2"], tensors["g2"]
    mixer.bind(tensors)
    assert torch.equal(mixer.w_a2, a2) and torch.equal(mixer.w_g2, g2)
    assert mixer.w_a2.data_ptr() % 16 == 0 and mixer.w_g2.data_ptr() % 16 == 0
    # the second operand of the one launch lies a whole number of rows of the rank behind the first
    assert mixer.w_low is None or a_rank * 2 % 16 == 0
