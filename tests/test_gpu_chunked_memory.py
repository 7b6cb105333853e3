"""Matrix memories over long portions as products over chunks of 64 rows, with gates, with a rotation, and with a decay for every
key channel, against the recurrence token by token in double precision."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
F = torch.float64
# portions (rows, position they start at): below, at and above a chunk, a last chunk of one row, and a single token beside them
ENTRIES = [[(70, 0)], [(64, 5), (3, 0), (129, 0)], [(33, 3), (1, 9), (200, 40)]]


def step_of(entries):
    from leone_amd.parts.context import EntryInfo, StepContext
    slots = [2, 0, 3][:len(entries)]
    infos, positions, owners = [], [], []
    for i, (slot, (count, start)) in enumerate(zip(slots, entries)):
        infos.append(EntryInfo(f"r{i}", slot, len(positions), count, start))
        positions += range(start, start + count)
        owners += [i] * count
    on = lambda values: torch.tensor(values, dtype=torch.int32, device=DEV)
    return slots, StepContext(rows=len(positions), dtype=torch.float32, device=torch.device(DEV), positions=on(positions), row_entry=on(owners),
                              entries=infos, entry_slots=on(slots), want_rows=None)


def close(got, want, what):
    # float sums of up to 260 products and decays of as many rows, each rounded to 2^-24 and growing like a random walk: a few
    # 1e-6 of the result's size; five times that
    error = float((got.to(F) - want).norm() / (want.norm() + 1e-30))
    assert error < 2e-5, (what, error)


def turned(x, positions, cos, sin):
    half = cos.shape[1]
    c, s = cos[positions].to(F), sin[positions].to(F)
    a, b = x[:, :half], x[:, half:2 * half]
    return torch.cat([a * c - b * s, b * c + a * s, x[:, 2 * half:]], 1)


@pytest.mark.parametrize("entries", ENTRIES, ids=str)
@pytest.mark.parametrize("heads,dim,vdim,rot", [(2, 256, 64, 0), (1, 24, 17, 8), (3, 64, 15, 64), (2, 130, 16, 130), (1, 200, 500, 0)])
@pytest.mark.parametrize("gated", [True, False])
def test_gates_and_rotations(gated, heads, dim, vdim, rot, entries):
    from leone_amd import ops
    gen = torch.Generator().manual_seed(dim + rot)
    slots, step = step_of(entries)
    rows = step.rows
    width = 2 * heads * dim + heads * vdim
    x = torch.randn(rows, width + 2 * heads, generator=gen)
    x[:, width + heads:] += 2.0
    x[rows // 3, width + heads:] = -30.0                      # a row that forgets, and one that writes with all its might
    x[rows // 2, width:width + heads] = 12.0
    per_head = dim * vdim + (dim + 1 if gated else 0)
    state = torch.randn(4, heads, per_head, generator=gen)
    for slot, (_, start) in zip(slots, entries):
        if start == 0:
            state[slot] = math.nan
    bias = torch.randn(2, heads, generator=gen)
    decay = torch.tensor([0.97, 0.0, 1.0])[:heads]
    cos, sin = ops.rope_table(1e4, rot, 300, DEV) if rot else (None, None)
    columns = {"q": 0, "k": heads * dim, "v": 2 * heads * dim, "i": width, "f": width + heads}
    dev_state = state.to(DEV)
    out, under = ops.outer_scan(x.to(DEV), columns, dev_state, step, heads, dim, vdim, q_scale=dim ** -0.5, k_scale=0.7, cos=cos, sin=sin,
                                **(dict(gates={"i_bias": bias[0].to(DEV), "f_bias": bias[1].to(DEV), "cap": 15.0}) if gated
                                   else dict(decay=decay.to(DEV))))
    out, x = out.view(rows, heads, vdim).cpu(), x.to(F)
    at = 0
    for slot, (count, start) in zip(slots, entries):
        span = slice(at, at + count)
        at += count
        for h in range(heads):
            q, k = (x[span, b + h * dim:b + (h + 1) * dim] for b in (0, heads * dim))
            if rot:
                q, k = (turned(t, range(start, start + count), cos.cpu(), sin.cpu()) for t in (q, k))
            q, k, v = q * dim ** -0.5, k * 0.7, x[span, 2 * heads * dim + h * vdim:2 * heads * dim + (h + 1) * vdim]
            before = state[slot, h].to(F) if start else torch.zeros(per_head, dtype=F)
            memory, norm, top = before[:dim * vdim].view(dim, vdim), before[dim * vdim:dim * vdim + dim], before[-1] if gated else None
            li = 15.0 * torch.tanh((x[span, width + h] + bias[0, h].to(F)) / 15.0)
            lf = torch.nn.functional.logsigmoid(15.0 * torch.tanh((x[span, width + heads + h] + bias[1, h].to(F)) / 15.0))
            want, dots, tops = [], [], []
            for t in range(count):
                a, b = decay[h].to(F), 1.0
                if gated:
                    new = torch.maximum(lf[t] + top, li[t])
                    a, b, top = torch.exp(lf[t] + top - new), torch.exp(li[t] - new), new
                    norm = a * norm + b * k[t]
                    dots.append(norm @ q[t])
                    tops.append(top)
                memory = a * memory + b * torch.outer(k[t], v[t])
                want.append(memory.T @ q[t])
            close(out[span, h], torch.stack(want), "out")
            close(dev_state[slot, h, :dim * vdim].cpu(), memory.reshape(-1), "state")
            if gated:
                close(under[0][span, h].cpu(), torch.stack(dots), "normaliser's read-out")
                close(under[1][span, h].cpu(), torch.stack(tops), "running maximum")
                close(dev_state[slot, h, dim * vdim:dim * vdim + dim].cpu(), norm, "normaliser")


@pytest.mark.parametrize("entries", ENTRIES, ids=str)
@pytest.mark.parametrize("heads,kv_heads,dim,vdim", [(2, 1, 128, 128), (3, 3, 7, 11), (2, 2, 64, 40), (4, 2, 100, 130)])
@pytest.mark.parametrize("kind", ["mild", "strong", "extreme"])
def test_a_decay_for_every_channel(kind, heads, kv_heads, dim, vdim, entries):
    """Decays near 1, decays that leave nothing after a few rows, and channels that forget everything at one row beside ones
    that keep everything (which the rows before must not blur)."""
    from leone_amd import ops
    gen = torch.Generator().manual_seed(dim)
    slots, step = step_of(entries)
    rows, kv = step.rows, kv_heads * dim
    x = torch.randn(rows, 2 * kv + heads * vdim, generator=gen)
    beta, size = torch.randn(rows, heads, generator=gen), torch.randn(rows, heads * dim, generator=gen)
    rate_log, bias = torch.rand(heads, generator=gen) - 1.0, torch.rand(heads * dim, generator=gen) * 3 - 4
    if kind == "strong":
        rate_log = rate_log + 3.0
    if kind == "extreme":
        size = torch.where(torch.rand(rows, heads * dim, generator=gen) < 0.1, 300.0, -40.0)
    state = torch.randn(4, heads, dim, vdim, generator=gen)
    for slot, (_, start) in zip(slots, entries):
        if start == 0:
            state[slot] = math.nan
    dev_state = state.to(DEV)
    wide = torch.cat([size, beta], 1).to(DEV)                   # both as slices of wider rows
    out = ops.delta_scan(x.to(DEV), {"q": 0, "k": kv, "v": 2 * kv}, wide[:, heads * dim:], wide[:, :heads * dim], rate_log.to(DEV), bias.to(DEV),
                         dev_state, step, heads, kv_heads, dim, vdim, dim ** -0.5, 1e-6).view(rows, heads, vdim).cpu()
    x, at = x.to(F), 0
    for slot, (count, start) in zip(slots, entries):
        span = slice(at, at + count)
        at += count
        for h in range(heads):
            g = (h // (heads // kv_heads)) * dim
            q, k = (t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6) for t in (x[span, g:g + dim], x[span, kv + g:kv + g + dim]))
            v = x[span, 2 * kv + h * vdim:2 * kv + (h + 1) * vdim]
            mine = slice(h * dim, (h + 1) * dim)
            decay = torch.exp(-torch.exp(rate_log[h].to(F)) * torch.nn.functional.softplus((size[span, mine] + bias[mine]).to(F)))
            strength = torch.sigmoid(beta[span, h].to(F))
            memory = state[slot, h].to(F) if start else torch.zeros(dim, vdim, dtype=F)
            want = []
            for t in range(count):
                memory = decay[t][:, None] * memory
                memory = memory + torch.outer(k[t], strength[t] * (v[t] - memory.T @ k[t]))
                want.append(memory.T @ q[t] * dim ** -0.5)
            close(out[span, h], torch.stack(want), "out")
            close(dev_state[slot, h].cpu(), memory, "state")


PLANTS = ["v inf", "v nan", "k nan", "q nan", "gate nan", "strength nan"]


@pytest.mark.parametrize("at", [0, 15, 16, 37, 63, 64, 100, 129])
@pytest.mark.parametrize("plant", PLANTS)
@pytest.mark.parametrize("kind", ["gates", "fixed", "one", "channel"])
def test_what_is_not_finite_reaches_no_row_before_it(kind, plant, at, monkeypatch):
    """An infinity or a NaN in one row of a portion: the rows before it keep their bits, and from it on the same read-outs and
    states are finite as when the rows are walked one by one."""
    from leone_amd import ops
    heads, dim, vdim = 2, 40, 24
    gen = torch.Generator().manual_seed(5)
    slots, step = step_of([(130, 3)])
    rows, width = 130, heads * (2 * dim + vdim)
    x = torch.randn(rows, width + 2 * heads, generator=gen)
    beta, size = torch.randn(rows, heads, generator=gen), torch.randn(rows, heads * (dim if kind == "channel" else 1), generator=gen)
    first = torch.randn(4, heads, dim * vdim + (dim + 1 if kind == "gates" else 0), generator=gen)

    def run(spoilt):
        rows_in, gate, strength, state = x.clone(), size.clone(), beta.clone(), first.to(DEV)
        if spoilt:
            value = math.inf if plant.endswith("inf") else math.nan
            if plant[0] in "qkv":
                rows_in[at, {"q": 0, "k": heads * dim, "v": 2 * heads * dim}[plant[0]] + 7] = value       # of head 0
            elif plant == "gate nan":
                gate[at, 0], rows_in[at, width + heads] = value, value
            else:
                strength[at, 0], rows_in[at, width] = value, value
        columns = {"q": 0, "k": heads * dim, "v": 2 * heads * dim, "i": width, "f": width + heads}
        if kind in ("one", "channel"):
            state = state.view(4, heads, dim, vdim)
            out = ops.delta_scan(rows_in.to(DEV), columns, strength.to(DEV), gate.to(DEV), torch.zeros(heads, device=DEV),
                                 torch.zeros(gate.shape[1], device=DEV), state, step, heads, heads, dim, vdim, dim ** -0.5, 1e-6)
            return out, state.reshape(4, -1), out
        if kind == "gates":
            bias = torch.zeros(2, heads, device=DEV)
            out, under = ops.outer_scan(rows_in.to(DEV), columns, state, step, heads, dim, vdim, q_scale=dim ** -0.5,
                                        gates={"i_bias": bias[0], "f_bias": bias[1], "cap": 15.0})
            return out, state.view(4, -1), under[0]
        cos, sin = ops.rope_table(1e4, 16, 300, DEV)
        out, _ = ops.outer_scan(rows_in.to(DEV), columns, state, step, heads, dim, vdim, q_scale=dim ** -0.5, cos=cos, sin=sin,
                                decay=torch.tensor([0.97, 0.9], device=DEV))
        return out, state.view(4, -1), out

    clean, spoilt = run(False), run(True)
    monkeypatch.setattr(ops, "MEMORY_CHUNKS_FROM", 1 << 30)
    walked = run(True)
    for now, was, by_rows in zip(spoilt, clean, walked):
        assert torch.equal(torch.isfinite(now), torch.isfinite(by_rows))
    for i in (0, 2):
        assert torch.equal(spoilt[i][:at], clean[i][:at])


@pytest.mark.parametrize("dim", [40, 128, 256])
def test_chunks_are_as_exact_as_rows(dim, monkeypatch):
    """Gated memories: what the read-outs are off 64 bits by, in chunks and walked row by row, over several inputs (the ratio of
    the means comes out between 0.93 and 0.96; sums over 256 channels in one chain gave 1.12)."""
    from leone_amd import ops
    heads, vdim, rows, off = 4, 64, 200, {"chunks": 0.0, "rows": 0.0}
    for seed in range(6):
        gen = torch.Generator(device=DEV).manual_seed(seed)
        width = heads * (2 * dim + vdim)
        x = torch.randn(rows, width + 2 * heads, generator=gen, device=DEV)
        x[:, width + heads:] += 2.0
        bias = torch.zeros(2, heads, device=DEV)
        columns = {"q": 0, "k": heads * dim, "v": 2 * heads * dim, "i": width, "f": width + heads}
        q, k = (x[:, b:b + heads * dim].to(F).view(rows, heads, dim).transpose(0, 1) for b in (0, heads * dim))
        v = x[:, 2 * heads * dim:width].to(F).view(rows, heads, vdim).transpose(0, 1)
        li, lf = (15.0 * torch.tanh(x[:, width + i * heads:width + (i + 1) * heads].to(F) / 15.0).T for i in (0, 1))
        total = torch.nn.functional.logsigmoid(lf).cumsum(1)
        entry = li - total
        top = total + entry.cummax(1).values.clamp_min(0)
        weight = ((total - top)[:, :, None] + entry[:, None, :]).masked_fill(torch.ones(rows, rows, device=DEV).triu(1) > 0, -math.inf).exp()
        want = ((q @ k.transpose(1, 2)) * dim ** -0.5 * weight) @ v
        for how in off:
            monkeypatch.setattr(ops, "MEMORY_CHUNKS_FROM", 32 if how == "chunks" else 1 << 30)
            state = torch.zeros(4, heads, dim * vdim + dim + 1, device=DEV)
            out, _ = ops.outer_scan(x, columns, state, step_of([(rows, 0)])[1], heads, dim, vdim, q_scale=dim ** -0.5,
                                    gates={"i_bias": bias[0], "f_bias": bias[1], "cap": 15.0})
            off[how] += float((out.view(rows, heads, vdim).transpose(0, 1).to(F) - want).norm() / want.norm()) / 6
    assert off["rows"] < 4e-7 and off["chunks"] <= 1.02 * off["rows"], off


@pytest.mark.parametrize("dim,from_rows", [(64, 32), (72, 64), (128, 64)])
def test_where_channel_wise_portions_go_in_chunks(dim, from_rows, monkeypatch):
    """Shorter portions are walked, which is faster there, and come out the same."""
    from leone_amd import ops
    seen, through = [], ops.chunked_memory
    monkeypatch.setattr(ops, "chunked_memory", lambda *a, **b: (seen.append(1), through(*a, **b)))
    for rows, chunked in ((from_rows - 1, False), (from_rows, True)):
        x, beta, size = (torch.randn(rows, n, device=DEV) for n in (3 * dim, 1, dim))
        state = torch.zeros(4, 1, dim, dim, device=DEV)
        seen.clear()
        ops.delta_scan(x, {"q": 0, "k": dim, "v": 2 * dim}, beta, size, torch.zeros(1, device=DEV), torch.zeros(dim, device=DEV), state,
                       step_of([(rows, 0)])[1], 1, 1, dim, dim, dim ** -0.5, 1e-6)
        assert bool(seen) == chunked
