"""Row-wise kernels at the sizes where many rows, whole runs or several trips of a workgroup take another path: filters of four taps
with a window in registers, the exponential gates of long portions."""
import math
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _step(spans, slots):
    """A step of entries with rows [first position, count] each."""
    positions = torch.cat([torch.arange(p, p + n) for p, n in spans]).to(torch.int32)
    entry = torch.cat([torch.full((n,), i) for i, (_, n) in enumerate(spans)]).to(torch.int32)
    entries, first = [], 0
    for (p, n), slot in zip(spans, slots):
        entries.append(SimpleNamespace(first_row=first, count=n, start=p, slot=slot))
        first += n
    return SimpleNamespace(decode_only=False, rows=first, positions=positions.to(DEV), row_entry=entry.to(DEV), entries=entries,
                           entry_slots=torch.tensor(slots, dtype=torch.int32, device=DEV), plan=None, device=torch.device(DEV))


@pytest.mark.parametrize("channels", [4, 1020, 1028, 1030])
@pytest.mark.parametrize("kind,out,filters", [(torch.float32, torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32, torch.float32),
                                              (torch.float32, torch.float32, torch.bfloat16)])
def test_filters_of_many_rows(channels, kind, out, filters):
    """Requests of a row, a few and many, at their start and later, boundaries inside a workgroup's rows; inputs that are columns of
    wider rows (1,030 channels: not in runs of four)."""
    from leone_amd import ops
    gen = torch.Generator().manual_seed(channels)
    spans, slots, taps = [(0, 1), (7, 2), (0, 3), (1, 5), (0, 500), (2, 11), (900, 9)], [3, 0, 6, 1, 5, 2, 4], 4
    step = _step(spans, slots)
    wide = torch.randn(step.rows, channels + 8, generator=gen).to(kind)
    weight, bias = torch.randn(channels, taps, generator=gen).to(filters), torch.randn(channels, generator=gen).to(filters)
    state = torch.randn(8, taps - 1, channels, generator=gen)
    kept = state.to(DEV).clone()
    x = wide.to(DEV)[:, 4:4 + channels]
    got = ops.causal_conv(x, weight.to(DEV), kept, step, out, add_input=True, bias=bias.to(DEV)).cpu().double()
    first, want, after = 0, [], state.double().clone()
    for (p, n), slot in zip(spans, slots):
        rows = wide[first:first + n, 4:4 + channels].double()
        before = state[slot].double() * (torch.arange(p - 3, p) >= 0)[:, None]
        full = torch.cat([before, rows])
        want.append(rows + bias.double() + sum(full[j:j + n] * weight.double()[:, j] for j in range(taps)))
        after[slot] = full[-3:]
        first += n
    want = torch.cat(want)
    # six float operations on values of up to some 20; results in bfloat16 have eight significant bits
    assert float(((got - want).abs() / (want.abs() + 10.0)).max()) < (2.0 ** -8 if out == torch.bfloat16 else 2e-6)
    assert torch.equal(kept.cpu().double(), after)


@pytest.mark.parametrize("counts", [(1, 1), (64, 1), (65, 3), (256, 257), (1024, 1025), (2111,), (300,) + (1,) * 130, (1100,) + (1, 2) * 520])
def test_exponential_gates(counts):
    """One wave's rows, a workgroup's and one over, from a state and from a sequence's start; long entries beside many short ones, with
    every number of threads."""
    from leone_amd import ops
    gen = torch.Generator().manual_seed(sum(counts))
    heads, dim, vdim = 2, 32, 64
    starts = [0 if i % 2 else 5 for i in range(len(counts))]
    step = _step(list(zip(starts, counts)), list(range(1, len(counts) + 1)))
    step.decode_only = all(n == 1 for n in counts)
    width = 2 * heads * dim + heads * vdim + 2 * heads
    proj = torch.randn(step.rows, width, generator=gen)
    columns = {"q": 0, "k": heads * dim, "v": 2 * heads * dim, "i": width - 2 * heads, "f": width - heads}
    bias = {"i": torch.randn(heads, generator=gen), "f": torch.randn(heads, generator=gen) + 2}
    per = dim * vdim + dim + 1
    state = torch.zeros(len(counts) + 1, heads, per)
    state[:, :, -1] = torch.randn(len(counts) + 1, heads, generator=gen)
    kept = state.to(DEV).clone()
    _, (_, top) = ops.outer_scan(proj.to(DEV), columns, kept, step, heads, dim, vdim,
                                 gates={"i_bias": bias["i"].to(DEV), "f_bias": bias["f"].to(DEV), "cap": 15.0})
    top, first = top.cpu().double(), 0
    for e, n in enumerate(counts):
        raw = proj[first:first + n].double()
        li = 15 * torch.tanh((raw[:, columns["i"]:columns["i"] + heads] + bias["i"].double()) / 15)
        lf = torch.nn.functional.logsigmoid(15 * torch.tanh((raw[:, columns["f"]:] + bias["f"].double()) / 15))
        m = torch.zeros(heads, dtype=torch.float64) if starts[e] == 0 else state[e + 1, :, -1].double()
        for t in range(n):
            m = torch.maximum(lf[t] + m, li[t])
            # sums of up to 64 gates of float a wave, each off by 2^-24 of values up to 100
            assert float((top[first + t] - m).abs().max()) < 1e-4, (e, t)
        assert float((kept[e + 1, :, -1].cpu().double() - m).abs().max()) < 1e-4
        first += n


def test_exponential_gates_of_an_entry_without_rows():
    """The maximum goes from the state that is read to the one that is written, nothing is read of the rows, and no row's gates change."""
    from leone_amd import ops
    from leone_amd.ops.library import call
    gen = torch.Generator().manual_seed(3)
    heads, rows = 3, 70
    proj, bias = torch.randn(rows, 2 * heads, generator=gen).to(DEV), torch.randn(2, heads, generator=gen).to(DEV)
    state = torch.randn(5, heads, 4, generator=gen)

    def gates(spans, longest):
        spans, kept = torch.tensor(spans, dtype=torch.int32, device=DEV), state.to(DEV).clone()
        coef, top = torch.zeros(rows, heads, 2, device=DEV), torch.zeros(rows, heads, device=DEV)
        call("leone_exp_gates", proj.data_ptr(), 2 * heads, 0, heads, bias[0].data_ptr(), bias[1].data_ptr(), ops.F32, 15.0, spans.data_ptr(),
             spans.shape[0], kept.data_ptr(), kept.stride(0), 4, 3, 1, coef.data_ptr(), top.data_ptr(), longest, heads, torch.cuda.current_stream().cuda_stream)
        return kept, coef, top

    for longest in (1, rows, 300):                       # a wave an entry, a few, and as many as a workgroup may have
        want = gates([[0, rows, 1, 1]], longest)
        got = gates([[0, 0, 0, 3], [0, rows, 1, 1], [0, 0, -1, 4]], longest)
        assert torch.equal(got[1], want[1]) and torch.equal(got[2], want[2])
        want[0][3, :, 3], want[0][4, :, 3] = state[0, :, 3].to(DEV), 0.0
        assert torch.equal(got[0], want[0])


@pytest.mark.parametrize("hidden", [8, 1016, 1032, 2048, 2056, 4096])
@pytest.mark.parametrize("weights,out", [(torch.bfloat16, torch.bfloat16), (torch.float32, torch.float32), (torch.bfloat16, torch.float32)])
def test_layer_norms_of_many_rows(hidden, weights, out):
    """A wave a row, at the lengths where its registers change and where a row ends inside a run of 256, with every set of operands."""
    from leone_amd import ops
    gen = torch.Generator().manual_seed(hidden)
    n = 515
    x, delta = torch.randn(n, hidden, generator=gen) * 2 + 0.5, torch.randn(n, hidden, generator=gen) - 0.25
    gain, bias, dgain, dbias = (torch.randn(hidden, generator=gen).to(weights) for _ in range(4))

    def norm(v, g, b, eps):
        off = v - v.mean(-1, keepdim=True)
        return off / ((off ** 2).mean(-1, keepdim=True) + eps).sqrt() * g.double() + b.double()

    for with_delta, normed, picked in ((False, False, False), (True, False, False), (True, True, False), (True, True, True)):
        rows = torch.randint(0, n, (n - 2,), generator=gen, dtype=torch.int32) if picked else None
        stream = x.to(DEV).clone()
        y = ops.add_layernorm(stream, delta.to(DEV) if with_delta else None, gain.to(DEV), bias.to(DEV), 1e-5, out,
                              rows.to(DEV) if picked else None, (dgain.to(DEV), dbias.to(DEV), 1e-6) if normed else None)
        more = (norm(delta.double(), dgain, dbias, 1e-6) if normed else delta.double()) if with_delta else 0.0
        total = x.double() + more
        want = norm(total, gain, bias, 1e-5)
        want = want[rows.long()] if picked else want
        # float sums of up to 4,096 terms over 64 lanes, a few roundings behind them; bfloat16 results have eight significant bits (a
        # row of 8 elements may vary little beside its mean)
        assert float(((y.cpu().double() - want).abs() / (want.abs() + 1.0)).max()) < (2.0 ** -8 if out == torch.bfloat16 else 0.0) + (4e-6 if hidden > 8 else 2e-5)
        assert torch.equal(stream.cpu(), x) if picked or not with_delta else float((stream.cpu().double() - total).abs().max()) < 4e-5


@pytest.mark.parametrize("kind", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads,vdim", [(16, 1), (20, 1), (1312, 1), (1316, 1), (5, 8), (3, 24), (7, 6)])
def test_gates_on_attentions_output(kind, heads, vdim):
    """A gate an element, of few and of many values, and a gate a head, in runs of eight and where a row does not lie in such runs."""
    from leone_amd import ops
    gen = torch.Generator().manual_seed(heads * vdim)
    rows = 300
    out, gate = torch.randn(rows, heads * vdim, generator=gen).to(kind), torch.randn(rows, heads + 12, generator=gen) * 3
    for first in (0, 4, 5):
        got = ops.head_gate(out.to(DEV).clone(), gate.to(DEV)[:, first:first + heads], heads, vdim).cpu().double()
        want = out.double() * torch.sigmoid(gate.double()[:, first:first + heads]).repeat_interleave(vdim, 1)
        assert float(((got - want).abs() / (want.abs() + 1e-3)).max()) < (2.0 ** -8 if kind == torch.bfloat16 else 2e-6)


@pytest.mark.parametrize("rows", [256, 259])
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("turned,pairing,normed", [(1.0, "half_split", True), (1.0, "adjacent", True), (0.5, "adjacent", True), (0.0, "adjacent", False)])
def test_heads_in_runs_of_eight(rows, dim, turned, pairing, normed):
    """Norms, rotation and cache write in runs of eight against the kernel a wave a head, which takes rows that do not lie in such runs:
    the same bits, for prompts and decoded tokens at odd places, unmapped pages, layers that bring queries only."""
    from leone_amd import ops
    gen = torch.Generator(device=DEV).manual_seed(rows + dim)
    rand = lambda *size: torch.randn(*size, generator=gen, device=DEV)     # noqa: E731
    q_heads, kv_heads, page = 18, 2, 16                  # enough heads for the kernel in runs with and without keys and values
    assert ops.library().leone_heads_in_pairs(rows, q_heads, 0) and ops.library().leone_heads_in_pairs(rows, q_heads + 2 * kv_heads, 1)
    heads = (q_heads + 2 * kv_heads) * dim
    positions = 5 + torch.arange(rows, dtype=torch.int32, device=DEV)
    entry = torch.zeros(rows, dtype=torch.int32, device=DEV)
    if rows > 256:                                       # two requests, the second one from a run's start on
        positions[33:] = torch.arange(8, 8 + rows - 33, dtype=torch.int32, device=DEV)
        entry[33:] = 1
    table = torch.randperm(40, generator=gen, device=DEV).view(2, 20).to(torch.int32)
    table[1, 2] = -1
    cos, sin = ops.rope_table(1e6, int(dim * turned), 300, DEV) if turned else (None, None)
    for kind in (torch.float32, torch.bfloat16):
        for given in {torch.float32, kind}:
            gains = [(1 + 0.1 * rand(dim)).to(kind) for _ in range(2)] if normed else [None, None]
            data = rand(rows, heads + 8).to(given)
            pools = rand(40, kv_heads, dim // 8, page, 8).to(kind), rand(40, kv_heads, page // 8, dim, 8).to(kind)
            for queries_only in (False, True):
                found = []
                for width in (heads + 8, heads + 4):     # rows that lie in runs, and rows that do not
                    k_pool, v_pool = (p.clone() for p in pools)
                    q = ops.qk_norm_rope_write(data[:, :width].contiguous(), q_heads, kv_heads, dim, *gains, 1e-6, cos, sin, positions, entry, table,
                                               k_pool, v_pool, write_cache=not queries_only, out_dtype=kind, pairing=pairing, value_dim=dim,
                                               queries_only=queries_only)
                    found.append((q, k_pool, v_pool))
                assert all(torch.equal(a, b) for a, b in zip(*found)), (kind, given, queries_only)
                assert queries_only or not torch.equal(found[0][1], pools[0])


@pytest.mark.parametrize("dim,q_heads,kv_heads,rows", [(16, 32, 4, 1050), (32, 30, 2, 1089), (16, 16, 4, 600)])
def test_two_key_ranges_of_small_heads(dim, q_heads, kv_heads, rows):
    """Key ranges of a long portion merged two rows a wave, the last tile not full, and of a shorter one a row a wave."""
    from leone_amd import ops
    gen = torch.Generator().manual_seed(dim + rows)
    page = 16
    pages = -(-rows // page)
    keys, values = (torch.randn(pages * page, kv_heads, dim, generator=gen).bfloat16() for _ in range(2))
    k_pool = keys.view(pages, page, kv_heads, dim // 8, 8).permute(0, 2, 3, 1, 4).contiguous()
    v_pool = values.view(pages, page // 8, 8, kv_heads, dim).permute(0, 3, 1, 4, 2).contiguous()
    q = torch.randn(rows, q_heads, dim, generator=gen).bfloat16()
    out = torch.empty(rows, q_heads * dim, dtype=torch.bfloat16, device=DEV)
    table = torch.arange(pages, dtype=torch.int32, device=DEV).view(1, -1)
    ops.attention_prefill(q.view(rows, -1).to(DEV), out, k_pool.to(DEV), v_pool.to(DEV), torch.arange(rows, dtype=torch.int32, device=DEV),
                          ops.prefill_tiles([(0, 0, rows)]).to(DEV), table, q_heads, dim ** -0.5, splits=2)
    hidden = torch.triu(torch.ones(rows, rows, dtype=torch.bool), 1)
    for h in range(q_heads):
        scores = (q[:, h].double() @ keys[:rows, h * kv_heads // q_heads].double().T) * dim ** -0.5
        want = torch.softmax(scores.masked_fill(hidden, -math.inf), -1) @ values[:rows, h * kv_heads // q_heads].double()
        # weights and results are rounded to eight bits: 2^-8 of the largest value, a few times over
        assert float((out.view(rows, q_heads, dim)[:, h].cpu().double() - want).abs().max()) < 0.03
