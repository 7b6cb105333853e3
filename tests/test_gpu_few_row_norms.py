"""Layer norms of few rows whose elements stay in registers, and the per-head norm with its gate, at the sizes where a lane's or a
thread's share changes."""
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _norm(v, gain, bias, eps):
    mean = v.mean(-1, keepdim=True)
    return (v - mean) / (((v - mean) ** 2).mean(-1, keepdim=True) + eps).sqrt() * gain.double() + bias.double()


def _close(got, want, out):
    # float sums of up to 5,000 terms over a thousand threads, a few roundings behind them; results in
    # bfloat16 have eight significant bits, so up to 2^-8 of the value more
    err = (got.cpu().double() - want).abs()
    assert float((err / (want.abs() + 1.0)).max()) < (2.0 ** -8 + 4e-6 if out == torch.bfloat16 else 4e-6)


@pytest.mark.parametrize("hidden", [1, 63, 1024, 1025, 2048, 2049, 4096, 4097])
@pytest.mark.parametrize("weights,out", [(torch.bfloat16, torch.bfloat16), (torch.float32, torch.bfloat16), (torch.float32, torch.float32),
                                         (torch.bfloat16, torch.float32)])
def test_layer_norms_of_few_rows(hidden, weights, out):
    """Rows just filling the threads' registers, one element over and too long for them, with every set of operands."""
    from leone_amd import ops
    gen = torch.Generator().manual_seed(hidden)
    n = 5
    draw = lambda *size: torch.randn(*size, generator=gen)     # noqa: E731
    x, delta = draw(n, hidden) * 2 + 0.5, draw(n, hidden) - 0.25
    gain, bias, dgain, dbias = (draw(hidden).to(weights) for _ in range(4))
    dev = lambda *ts: [t.to(DEV) for t in ts]                  # noqa: E731
    for with_delta, normed, picked in ((False, False, False), (True, False, False), (True, True, False), (True, True, True)):
        rows = torch.tensor([3, 0, 3], dtype=torch.int32) if picked else None
        stream = x.to(DEV).clone()
        y = ops.add_layernorm(stream, delta.to(DEV) if with_delta else None, *dev(gain, bias), 1e-5, out, rows.to(DEV) if picked else None,
                              (*dev(dgain, dbias), 1e-6) if normed else None)
        more = (_norm(delta.double(), dgain, dbias, 1e-6) if normed else delta.double()) if with_delta else 0.0
        total = x.double() + more
        want = _norm(total, gain, bias, 1e-5)
        _close(y, want[rows.long()] if picked else want, out)
        assert torch.equal(stream.cpu(), x) if picked or not with_delta else float((stream.cpu().double() - total).abs().max()) < 2e-5
    stream = x.to(DEV).clone()
    assert ops.add_layernorm(stream, delta.to(DEV), None, None, 1e-5, None) is None and torch.equal(stream.cpu(), x + delta)


@pytest.mark.parametrize("hidden", [1, 1025, 2049, 4097])
@pytest.mark.parametrize("taps,filters", [(2, torch.bfloat16), (3, torch.bfloat16), (4, torch.bfloat16), (5, torch.bfloat16), (4, torch.float32)])
def test_layer_norms_of_few_rows_with_a_folded_filter(hidden, taps, filters):
    """Requests at their first inputs (what the state holds does not count) and later ones, slots in another order than rows; more taps
    than are held, and filters of another type than the norm's vectors, take the other kernel."""
    from leone_amd import ops
    gen = torch.Generator().manual_seed(hidden + taps)
    n = 4
    x = torch.randn(n, hidden, generator=gen)
    gain, bias = torch.randn(hidden, generator=gen).bfloat16(), torch.randn(hidden, generator=gen).bfloat16()
    weight = torch.randn(hidden, taps, generator=gen).to(filters)
    state = torch.randn(6, taps - 1, hidden, generator=gen)
    positions, slots = torch.tensor([0, 1, taps - 1, 50], dtype=torch.int32), torch.tensor([4, 1, 5, 0], dtype=torch.int32)
    step = SimpleNamespace(decode_only=True, rows=n, positions=positions.to(DEV), row_entry=torch.arange(n, dtype=torch.int32, device=DEV),
                           entry_slots=slots.to(DEV))
    h = _norm(x.double(), gain, bias, 1e-5)
    for write in (False, True):
        kept = state.to(DEV).clone()
        y = ops.add_layernorm(x.to(DEV), None, gain.to(DEV), bias.to(DEV), 1e-5, torch.float32, conv=(weight.to(DEV), kept, step, write))
        after = state.clone().double()
        for r in range(n):
            s, p = int(slots[r]), int(positions[r])
            old = torch.stack([state[s, j].double() * (p - (taps - 1 - j) >= 0) for j in range(taps - 1)] + [h[r]])
            want = h[r] + (weight.double().T * old).sum(0)
            # taps products behind the norm, each as large as the largest of their sum's terms
            scale = 1.0 + h[r].abs() + (weight.double().T * old).abs().sum(0)
            assert float(((y[r].cpu().double() - want).abs() / scale).max()) < 4e-6
            if write:
                after[s] = old[1:]
        assert float((kept.cpu().double() - after).abs().max()) < 4e-5
        assert write or torch.equal(kept.cpu(), state)


@pytest.mark.parametrize("vdim", [1, 63, 64, 65, 512, 513, 1024])
@pytest.mark.parametrize("act,gate_first", [("sigmoid", False), ("silu", True), (None, False)])
def test_head_norms_of_few_rows(vdim, act, gate_first):
    from leone_amd import ops
    gen = torch.Generator().manual_seed(vdim)
    rows, heads = 3, 5
    o, gate = torch.randn(rows, heads, vdim, generator=gen), torch.randn(rows, heads * vdim + 8, generator=gen)
    for weights, out in ((torch.bfloat16, torch.bfloat16), (torch.float32, torch.float32)):
        for per_head in (False, True):
            gain = torch.randn(heads * vdim if per_head else vdim, generator=gen).to(weights)
            more = {"gate": gate.to(DEV)[:, :heads * vdim], "activation": act} if act else {}
            got = ops.head_norm_gate(o.view(rows, -1).to(DEV), heads, vdim, 1e-5, out, gain=gain.to(DEV), gate_first=gate_first, **more)
            g = gate.double()[:, :heads * vdim].view(rows, heads, vdim)
            g = torch.sigmoid(g) * (g if act == "silu" else 1) if act else torch.ones_like(g)
            v = o.double() * (g if gate_first else 1)
            v = v / ((v ** 2).mean(-1, keepdim=True) + 1e-5).sqrt() * gain.double().view(*((heads, vdim) if per_head else (vdim,)))
            _close(got.view(rows, heads, vdim), v if gate_first else v * g, out)


@pytest.mark.parametrize("hidden", [4, 1020, 1024, 2048, 2052, 4096, 4100])
@pytest.mark.parametrize("places", [1, 4, 8, 9])
def test_norms_behind_a_sublayer_that_sum_their_places(hidden, places):
    """The norm of a delta in planes, and of what routed experts left row by row (some places handing the row on, some empty), at the
    sizes where registers no longer hold a row and where places come in several turns."""
    from leone_amd import ops
    gen = torch.Generator().manual_seed(hidden + places)
    n, experts = 6, 5
    draw = lambda *size: torch.randn(*size, generator=gen)     # noqa: E731
    x, pairs, extra = draw(n, hidden), draw(n * places, hidden), draw(n, hidden)
    chosen = torch.randint(-1, experts + 2, (n, places), generator=gen, dtype=torch.int32)
    weight, gain, gain2 = torch.rand(n, places, generator=gen), draw(hidden), draw(hidden).bfloat16()
    for kind, out, planes in ((torch.bfloat16, torch.bfloat16, False), (torch.float32, torch.float32, False), (None, torch.bfloat16, True)):
        for picked in (False, True):
            rows = torch.tensor([3, 0, 5], dtype=torch.int32) if picked else None
            stream = x.to(DEV).clone()
            if planes:
                delta, total = pairs.view(places, n, hidden).to(DEV), pairs.view(places, n, hidden).double().sum(0)
            else:
                came = draw(n, hidden).to(kind)
                with_extra = extra if kind == torch.float32 else None
                delta = ops.PairedRows(pairs.to(DEV), chosen.to(DEV), weight.to(DEV), came.to(DEV), with_extra.to(DEV) if with_extra is not None else None, experts)
                each = torch.where((chosen >= experts)[..., None], weight.double()[..., None] * came.double()[:, None], pairs.view(n, places, hidden).double())
                total = (each * (chosen >= 0)[..., None]).sum(1) + (with_extra.double() if with_extra is not None else 0)
                assert float((delta.sum().cpu().double() - total).abs().max()) < 1e-5
            normed = lambda v, g, eps: v / ((v ** 2).mean(-1, keepdim=True) + eps).sqrt() * g.double()      # noqa: E731
            after = x.double() + normed(total, gain, 1e-6)
            then = (gain2.to(DEV), 1e-5, out) if picked else None
            y = ops.add_normed(stream, delta, gain.to(DEV), 1e-6, out_dtype=None if picked else out, then=then, rows=rows.to(DEV) if picked else None)
            _close(y, normed(after, gain2, 1e-5)[rows.long()] if picked else after, out)
            assert torch.equal(stream.cpu(), x) if picked else float((stream.cpu().double() - after).abs().max()) < 4e-5
