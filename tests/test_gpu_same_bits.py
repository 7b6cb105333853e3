"""Kernels in runs and in registers against the general ones they stand in for, which take operands that do not lie so: the same bits."""
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _off(t):
    """The same values one element past an aligned address."""
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=DEV)[1:]
    flat.copy_(t.reshape(-1))
    return flat.view(t.shape)


def _single_rows(n, generator):
    slots = torch.randperm(n + 2, generator=generator)[:n].to(torch.int32)
    return SimpleNamespace(decode_only=True, rows=n, positions=torch.randint(0, 6, (n,), generator=generator, dtype=torch.int32).to(DEV),
                           row_entry=torch.arange(n, dtype=torch.int32, device=DEV), entry_slots=slots.to(DEV))


@pytest.mark.parametrize("rows", [5, 300, 515])
@pytest.mark.parametrize("hidden", [8, 1000, 1024, 1032, 2048, 2056, 4096])
@pytest.mark.parametrize("weights,out", [(torch.bfloat16, torch.bfloat16), (torch.float32, torch.float32)])
def test_layer_norms(rows, hidden, weights, out):
    """Few rows in runs or element by element, many rows a wave each, against the kernels for any address; with and without a norm of the
    delta, rows that are picked, and for few rows a filter of four taps and its state."""
    from leone_amd import ops
    gen = torch.Generator().manual_seed(rows + hidden)
    x, delta = torch.randn(rows, hidden, generator=gen).to(DEV) * 2 + 0.5, torch.randn(rows, hidden, generator=gen).to(DEV)
    gain, bias, dgain, dbias = (torch.randn(hidden, generator=gen).to(weights).to(DEV) for _ in range(4))
    picked = torch.randint(0, rows, (rows,), generator=gen, dtype=torch.int32).to(DEV)
    filters, kept = torch.randn(hidden, 4, generator=gen).to(weights).to(DEV), torch.randn(rows + 2, 3, hidden, generator=gen).to(DEV)
    step = _single_rows(rows, gen)
    for normed, which, taps in ((False, None, False), (True, None, False), (True, picked, False)) + (((True, None, True),) if rows < 512 else ()):
        found = []
        for place in (torch.clone, _off):
            stream, state = place(x), kept.clone()
            y = ops.add_layernorm(stream, delta, gain, bias, 1e-5, out, which, (dgain, dbias, 1e-6) if normed else None,
                                  (filters, state, step, True) if taps else None)
            found.append((y, stream, state))
        assert all(torch.equal(a, b) for a, b in zip(*found)), (normed, which is not None, taps)


@pytest.mark.parametrize("channels", [4, 1028, 2048])
def test_filters_of_many_rows(channels):
    from leone_amd import ops
    gen = torch.Generator().manual_seed(channels)
    spans = [(0, 500), (7, 2), (2, 11), (900, 90)]
    entries, first = [], 0
    for slot, (start, count) in enumerate(spans):
        entries.append(SimpleNamespace(first_row=first, count=count, start=start, slot=slot))
        first += count
    step = SimpleNamespace(decode_only=False, rows=first, positions=torch.cat([torch.arange(p, p + n) for p, n in spans]).to(torch.int32).to(DEV),
                           row_entry=torch.cat([torch.full((n,), i) for i, (_, n) in enumerate(spans)]).to(torch.int32).to(DEV), entries=entries,
                           entry_slots=torch.arange(len(spans), dtype=torch.int32, device=DEV), plan=None, device=torch.device(DEV))
    state, weight = torch.randn(4, 3, channels, generator=gen).to(DEV), torch.randn(channels, 4, generator=gen).bfloat16().to(DEV)
    for kind in (torch.float32, torch.bfloat16):
        x = torch.randn(first, channels, generator=gen).to(kind).to(DEV)
        for out in (torch.float32, torch.bfloat16):
            got, want = (ops.causal_conv(place(x), weight, state, step, out, add_input=True, activation="silu", write_state=False) for place in (torch.clone, _off))
            assert torch.equal(got, want)


@pytest.mark.parametrize("rows", [3, 700])
@pytest.mark.parametrize("hidden", [4, 1020, 1024, 1028, 2048, 2052, 4096])
def test_norms_behind_a_sublayer(rows, hidden):
    """One delta, planes, and experts' places, which the general path sums in a launch of its own; with and without a second norm.  Gains
    that are not aligned take the kernel that holds no row, in the same runs of four."""
    from leone_amd import ops
    gen = torch.Generator().manual_seed(rows + hidden)
    draw = lambda *size: torch.randn(*size, generator=gen).to(DEV)     # noqa: E731
    x, gain, gain2 = draw(rows, hidden), draw(hidden).bfloat16(), draw(hidden)
    chosen = torch.randint(-1, 7, (rows, 5), generator=gen, dtype=torch.int32).to(DEV)
    paired = ops.PairedRows(draw(rows * 5, hidden), chosen, draw(rows, 5).abs(), draw(rows, hidden).bfloat16(), draw(rows, hidden), 5)
    for delta in (draw(rows, hidden), draw(3, rows, hidden), paired):
        for then in (None, (gain2, 1e-5, torch.bfloat16)):
            found = []
            for place in (torch.clone, _off):
                stream = x.clone()
                found.append((ops.add_normed(stream, delta, place(gain), 1e-6, out_dtype=None if then else torch.bfloat16, then=then), stream))
            assert torch.equal(found[0][0], found[1][0]) and torch.equal(found[0][1], found[1][1])


@pytest.mark.parametrize("kind", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads,vdim", [(2048, 1), (16, 128), (3, 24)])
def test_gates_on_attentions_output(kind, heads, vdim):
    from leone_amd import ops
    gen = torch.Generator().manual_seed(heads)
    rows = 300
    out, gate = torch.randn(rows, heads * vdim, generator=gen).to(kind).to(DEV), torch.randn(rows, heads, generator=gen).to(DEV) * 3
    got, want = (ops.head_gate(place(out), gate, heads, vdim) for place in (torch.clone, _off))
    assert torch.equal(got, want)
