"""Request slots of several state tensors cleared, copied, saved and put back in one launch."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("shapes", [[(1,)], [(3, 5), (4096,), (4097,)], [(2, 16 * 24 + 16 + 1), (7,), (3, 1000), (5, 2048, 4), (1, 1, 4)],
                                    [(n,) for n in range(1, 70)]])
@pytest.mark.parametrize("slots", [2, 9, 70])
def test_moves(shapes, slots):
    from leone_amd.ops.state import StateSlots
    gen = torch.Generator(device=DEV).manual_seed(slots)
    tensors = [torch.randn((slots, *shape), generator=gen, device=DEV) for shape in shapes]
    want = [t.clone() for t in tensors]
    held = StateSlots(tensors)

    def same():
        return all(torch.equal(a, b) for a, b in zip(tensors, want))

    held.copy(0, slots - 1)
    for t in want:
        t[slots - 1] = t[0]
    assert same()
    some = list(range(1, slots))
    packed = held.save(some)
    assert same()
    held.zero(some)
    kept = [t.clone() for t in want]
    for t in want:
        t[1:] = 0
    assert same()
    held.restore(some, packed)
    want = kept
    assert same()


def test_refusals():
    from leone_amd.ops import KernelError
    from leone_amd.ops.state import StateSlots
    held = StateSlots([torch.zeros(4, 6, device=DEV)])
    for slots in ([4], [-1]):
        with pytest.raises(KernelError):
            held.zero(slots)
    with pytest.raises(KernelError):
        held.restore([0, 1], held.save([0]))
    with pytest.raises(KernelError):
        StateSlots([torch.zeros(4, 6, device=DEV), torch.zeros(3, 6, device=DEV)])
    assert not StateSlots.takes(torch.zeros(4, 6)) and not StateSlots.takes(torch.zeros(6, 4, device=DEV).T)
    assert not StateSlots.takes(torch.zeros(4, 3, dtype=torch.bfloat16, device=DEV))
