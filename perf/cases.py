"""The work this engine is measured by: decoding and prompts through ``Engine.step``, generation through ``Runtime``.

A case is one pass of a user's program over a model it has loaded: ``steps`` decode steps of a batch whose requests stand at
their contexts, the prompts of some requests in one step, a prompt portion beside decoding requests (continuous batching),
greedy decoding behind a prompt, or whole generations with sampling.  The models are the layer sizes ``leone_amd.benchmark``
measures (``DESIGN_SIZES``; width 4,096 is the layer of the Qwen3-8B shape): Qwen3, Pamevik (per-request state: mLSTM,
retention and delta-rule memories beside attention) and Zukinex (windowed attention, mixtures of experts), with weights made
here from the seed.  Tokens of the bfloat16 models are given, as a scoring or replaying program gives them: the results are
logits, which a near tie between two tokens does not turn into another sequence.
"""
import math
import zlib

import torch

from leone_amd import ops
from leone_amd.api import Runtime, sampling_params
from leone_amd.architectures import config_from_dict, model_spec_for
from leone_amd.benchmark import QWEN3_8B, pamevik_shape, zukinex_shape
from leone_amd.engine.engine import StepEntry
from leone_amd.engine.scheduler import SchedulerPolicy
from leone_amd.parts.model import DecoderModel
from leone_amd.weights import loader

DEVICE = "cuda:0"
PAGE = 64
VOCAB = 32768
F64 = torch.float64


def _case(name, design, width, work, dtype="bfloat16", batch=1, shortest=0, longest=0, steps=1, portion=0, start=0):
    case = {"design": design, "width": width, "layers": 8 if width >= 1024 else 4, "dtype": dtype, "work": work,
            "batch": batch, "shortest": shortest, "longest": longest, "steps": steps, "portion": portion, "start": start}
    return {"name": name, **case} if name else case


def listed():
    return [
        # one user's chat, a few thousand tokens in
        _case("qwen3 decode 1", "qwen3", 4096, "decode", batch=1, shortest=2048, longest=2048, steps=8),
        # the benchmark's headline: eight requests at a context of 8,192
        _case("qwen3 decode 8", "qwen3", 4096, "decode", batch=8, shortest=8176, longest=8176, steps=8),
        # a full serving batch whose requests have come to different lengths
        _case("qwen3 decode 64", "qwen3", 4096, "decode", batch=64, shortest=300, longest=2304, steps=8),
        # the smallest step: a short question to a small model, where launches and latency are what is waited for
        _case("qwen3 decode short", "qwen3", 1024, "decode", batch=2, shortest=77, longest=120, steps=8),
        # the benchmark's prompt
        _case("qwen3 prompt 2048", "qwen3", 4096, "prompt", batch=1, shortest=2048, longest=2048),
        # continuous batching: a late portion of a long prompt, eleven other requests decoding beside it
        _case("qwen3 portion", "qwen3", 4096, "mixed", batch=11, shortest=150, longest=3000, portion=501, start=6000),
        # the true 32-bit engine: a prompt and the tokens behind it, chosen on the device
        _case("qwen3 float32", "qwen3", 2048, "greedy", dtype="float32", batch=1, shortest=777, longest=777, steps=8),
        # the entry point whole: scheduler, prompts, decoding, and samplers that cut
        _case("qwen3 generate", "qwen3", 512, "generate", dtype="float32", batch=5, shortest=40, longest=300, steps=24),
        # recurrent mixers: a long prompt in one portion
        _case("pamevik prompt 2048", "pamevik", 2048, "prompt", batch=1, shortest=2048, longest=2048),
        # recurrent mixers: requests that go on from prompts they have in the cache
        _case("pamevik decode 8", "pamevik", 2048, "decode", batch=8, shortest=700, longest=1472, steps=12),
        # mixtures of experts: a few prompts of odd lengths arriving together
        _case("zukinex prompts", "zukinex", 2048, "prompt", batch=3, shortest=211, longest=901),
        # mixtures of experts: a small batch decoding past its window
        _case("zukinex decode 8", "zukinex", 2048, "decode", batch=8, shortest=1100, longest=1984, steps=8),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["qwen3 decode", "qwen3 decode", "qwen3 decode", "qwen3 prompt", "qwen3 prompt", "qwen3 mixed",
                       "qwen3 greedy", "qwen3 generate", "pamevik prompt", "pamevik decode", "zukinex prompt", "zukinex decode"])
    design, work = kind.split()
    width = {"qwen3": rng.choice([1024, 1536, 2048, 3072, 4096]), "pamevik": rng.choice([1024, 2048, 2048]),
             "zukinex": rng.choice([1024, 2048, 2048])}[design]
    if work == "decode":
        batch = _log(rng, 1, 64)
        longest = _log(rng, 64, min(8176, 64 * 1024 // batch) if design == "qwen3" else 2048 // (1 + batch // 16))
        shortest = rng.randint(max(32, longest // 4), longest)
        return _case(None, design, width, work, batch=batch, shortest=shortest, longest=longest, steps=rng.choice([4, 6, 8]))
    if work == "prompt":
        batch = rng.choice([1, 1, 2, 3, 4])
        longest = _log(rng, 17, 2048 // batch)
        return _case(None, design, width, work, batch=batch, shortest=rng.randint(max(9, longest // 3), longest), longest=longest)
    if work == "mixed":
        longest = _log(rng, 100, 3000)
        return _case(None, design, width, work, batch=rng.randint(1, 24), shortest=rng.randint(64, longest), longest=longest,
                     portion=_log(rng, 33, 1024), start=_log(rng, 128, 6000))
    if work == "greedy":
        longest = _log(rng, 16, 1024)
        return _case(None, design, rng.choice([512, 1024, 2048]), work, dtype="float32", batch=1, shortest=longest,
                     longest=longest, steps=rng.randint(2, 8))
    longest = _log(rng, 40, 300)
    return _case(None, design, rng.choice([512, 1024]), work, dtype="float32", batch=rng.randint(1, 6),
                 shortest=rng.randint(20, longest), longest=longest, steps=rng.randint(8, 24))


def lengths(case):
    """The requests' contexts (or prompts), spread from ``shortest`` to ``longest``; contexts that are gone on from by another
    request are whole pages."""
    low, high, n = case["shortest"], case["longest"], case["batch"]
    spread = [high - int(round((high - low) * ((i * 0.6180339887) % 1.0))) for i in range(n)]
    return [max(1, s // PAGE) * PAGE for s in spread] if continues(case) else spread


def continues(case):
    """Whether the decoding requests are continuations of the ones held: neither a request's state nor the keys a window has
    passed can be cut back to, so that a pass forks what it decodes."""
    return case["work"] == "decode" and case["design"] != "qwen3"


# ---- models -------------------------------------------------------------------------------------------------------------
def config_of(case):
    width, layers = case["width"], case["layers"]
    if case["design"] == "qwen3":
        return dict(QWEN3_8B, num_hidden_layers=layers, hidden_size=width, num_attention_heads=width // 128,
                    num_key_value_heads=width // 512, intermediate_size=3 * width, vocab_size=VOCAB, max_position_embeddings=16384)
    shape = {"pamevik": pamevik_shape, "zukinex": zukinex_shape}[case["design"]]
    return shape(width, layers, VOCAB, 4096)


def tensor_shapes(c):
    """Name -> shape of every tensor of a model's checkpoint."""
    out = {}
    if "hidden_size" in c:
        w, d, ff = c["hidden_size"], c["head_dim"], c["intermediate_size"]
        hq, hk = c["num_attention_heads"] * d, c["num_key_value_heads"] * d
        out["model.embed_tokens.weight"] = (c["vocab_size"], w)
        for i in range(c["num_hidden_layers"]):
            p = f"model.layers.{i}."
            out.update({p + "input_layernorm.weight": (w,), p + "post_attention_layernorm.weight": (w,),
                        p + "self_attn.q_proj.weight": (hq, w), p + "self_attn.k_proj.weight": (hk, w),
                        p + "self_attn.v_proj.weight": (hk, w), p + "self_attn.o_proj.weight": (w, hq),
                        p + "self_attn.q_norm.weight": (d,), p + "self_attn.k_norm.weight": (d,),
                        p + "mlp.gate_proj.weight": (ff, w), p + "mlp.up_proj.weight": (ff, w), p + "mlp.down_proj.weight": (w, ff)})
        out.update({"model.norm.weight": (w,), "lm_head.weight": (c["vocab_size"], w)})
        return out
    w = c["width"]
    out["embed"] = (c["vocab"], w)
    if c["architecture"] == "Zukinex":
        out["pos"] = (c["max_positions"], w)
        for i, layer in enumerate(c["layers"]):
            m, f, x, y = layer["mixer"], layer["mlp"], f"l{i}.mix.", f"l{i}.mlp."
            out.update({f"l{i}.norm1": (w,), f"l{i}.norm2": (w,), x + "q": (m["heads"] * m["dim"], w), x + "q.norm": (m["dim"],),
                        x + "g": (m["heads"] * m["vdim"], w), x + "o": (w, m["heads"] * m["vdim"])})
            if m.get("kv_from") is None:
                out.update({x + "k": (m["kv_heads"] * m["dim"], w), x + "v": (m["kv_heads"] * m["vdim"], w), x + "k.norm": (m["dim"],)})
            parts = {"": f["ff"]} if f["kind"] == "dense" else {
                **{f"e{e}.": f["expert"]["ff"] for e in range(f["router"]["experts"])}, "shared.": f["shared"]["ff"]}
            for part, ff in parts.items():
                out.update({y + part + "gate": (ff, w), y + part + "up": (ff, w), y + part + "down": (w, ff)})
            if f["kind"] == "moe":
                total = f["router"]["experts"] + f["router"]["identity"]
                out.update({y + "router": (total, w), y + "correction": (total,)})
        out.update({"final.norm": (w,), "head": (c["vocab"], w)})
        return out
    for i, layer in enumerate(c["layers"]):
        p, x, m = f"l{i}.", f"l{i}.mix.", layer["mixer"]
        for n in ["1"] + (["2"] if layer["mlp"] else []):
            for part in (f"norm{n}", f"norm{n}b"):
                out.update({p + part: (w,), p + part + ".b": (w,)})
            out[p + "canon" + n] = (w, c["canon"]["taps"])
        if layer["mlp"]:
            out.update({p + "mlp.up": (layer["mlp"]["ff"], w), p + "mlp.down": (w, layer["mlp"]["ff"])})
        if layer["type"] == "mlstm":
            qk, vv = m["heads"] * m["dim"], m["heads"] * m["vdim"]
            out.update({x + "q": (qk, w), x + "k": (qk, w), x + "v": (vv, w), x + "g": (vv, w), x + "o": (w, vv), x + "norm": (vv,),
                        x + "i": (m["heads"], w), x + "i.b": (m["heads"],), x + "f": (m["heads"], w), x + "f.b": (m["heads"],)})
        elif layer["type"] == "channel_delta":
            qk, vv, hd = m["kv_heads"] * m["dim"], m["heads"] * m["vdim"], m["heads"] * m["dim"]
            out.update({x + "q": (qk, w), x + "k": (qk, w), x + "v": (vv, w), x + "q.conv": (qk, m["conv"]), x + "k.conv": (qk, m["conv"]),
                        x + "v.conv": (vv, m["conv"]), x + "b": (m["heads"], w), x + "A_log": (m["heads"],), x + "dt_bias": (hd,),
                        x + "a1": (m["a_rank"], w), x + "a2": (hd, m["a_rank"]), x + "g1": (m["g_rank"], w), x + "g2": (vv, m["g_rank"]),
                        x + "norm": (m["vdim"],), x + "o": (w, vv)})
        else:
            a, r = m["left"], m["right"]
            out.update({x + "left.q": (a["heads"] * a["dim"], w), x + "left.k": (a["kv_heads"] * a["dim"], w),
                        x + "left.v": (a["kv_heads"] * a["vdim"], w), x + "left.g": (a["heads"], w),
                        x + "left.o": (w, a["heads"] * a["vdim"]), x + "left.out": (w,),
                        x + "right.q": (r["heads"] * r["dim"], w), x + "right.k": (r["heads"] * r["dim"], w),
                        x + "right.v": (r["heads"] * r["vdim"], w), x + "right.g": (r["heads"] * r["vdim"], w),
                        x + "right.o": (w, r["heads"] * r["vdim"]), x + "right.out": (w,)})
    out.update({"final.norm": (w,), "final.norm.b": (w,), "head": (c["vocab"], w)})
    return out


def make_weights(case, seed):
    """Weights of the kind training leaves: activations of order one through every layer, gains around their design's size,
    decays away from 0 and 1, and a router that is sure of its experts (each token's vector lies near one of 64 centres, and
    every centre has four experts)."""
    c, dtype = config_of(case), getattr(torch, case["dtype"])
    gen = torch.Generator(device=DEVICE)

    def normal(name, *shape):
        gen.manual_seed((int(seed) * 1000003 + zlib.crc32(name.encode())) & 0x7FFFFFFFFFFFFFFF)
        return torch.randn(shape, generator=gen, device=DEVICE)

    zukinex = c.get("architecture") == "Zukinex"
    centres = normal("centres", 64, case["width"]) if zukinex else None
    weights = {}
    for name, shape in tensor_shapes(c).items():
        last = name.split(".")[-1]
        t = normal(name, *shape)
        if zukinex and name == "embed":
            t = centres[torch.arange(shape[0], device=DEVICE) % 64] + 0.3 * t
        elif zukinex and name == "pos":
            t = 0.1 * t
        elif last == "router":
            gen.manual_seed((int(seed) * 31 + zlib.crc32(name.encode())) & 0x7FFFFFFF)
            liked = torch.rand((64, shape[0]), generator=gen, device=DEVICE).topk(4, dim=1).indices
            sure = 2.4 + 1.2 * torch.rand((64, 4), generator=gen, device=DEVICE)
            t = torch.zeros((64, shape[0]), device=DEVICE).scatter_(1, liked, sure).T @ centres / centres.square().sum(1).mean()
        elif last == "correction":
            t = 0.01 * t
        elif name.endswith("f.b"):
            t = t + 2.0
        elif last == "A_log":
            t = 0.5 * t - 1.0
        elif last in ("canon1", "canon2", "conv"):
            t = 0.4 * t
        elif last == "b" and "norm" in name:
            t = 0.1 * t
        elif zukinex and last in ("norm1", "norm2"):
            t = 0.25 + 0.02 * t
        elif len(shape) == 1 and last not in ("b", "dt_bias"):
            t = 1.0 + 0.1 * t
        elif len(shape) == 2 and last != "embed" and "embed_tokens" not in name:
            t = t / math.sqrt(shape[1])
        weights[name] = t.to(dtype)
    return weights


def tokens_of(case, seed):
    """Given tokens: for every request its context or prompt and ``steps`` tokens behind it; the prompt that comes in portions."""
    gen = torch.Generator().manual_seed(int(seed) * 7919 + 13)

    def some(n):
        return torch.randint(0, VOCAB, (n,), generator=gen).tolist()

    requests = [(some(n), some(case["steps"])) for n in lengths(case)]
    return requests, some(case["start"] + case["portion"])


def feed(engine, request, tokens):
    for at in range(0, len(tokens), 2048):
        engine.step([StepEntry(request, tokens[at:at + 2048])])


def prepare(case, seed):
    config = config_from_dict(config_of(case))
    dtype = getattr(torch, case["dtype"])
    model = DecoderModel(model_spec_for(config), dtype, torch.device(DEVICE))
    model.config = config
    model.bind(loader.load_from_tensors(make_weights(case, seed), model.tensor_specs(), dtype, DEVICE, source="made weights"))
    requests, long_prompt = tokens_of(case, seed)
    work, longest = case["work"], max(lengths(case))
    room = max(longest + case["steps"], len(long_prompt)) + PAGE
    pages = 2 * sum((n + case["steps"]) // PAGE + 2 for n in lengths(case)) + len(long_prompt) // PAGE + 2
    state = {"case": case, "requests": requests, "long": long_prompt}
    prompt_rows = sum(len(p) for p, _ in requests)
    runtime = Runtime(model, num_pages=pages, page_tokens=PAGE, max_requests=2 * case["batch"] + 1, max_context=room,
                      policy=SchedulerPolicy(max_live_requests=case["batch"], prefill_chunk_tokens=512, max_step_tokens=512))
    state["runtime"], state["engine"] = runtime, runtime.engine
    if work in ("decode", "mixed"):
        for i, (context, _) in enumerate(requests):
            feed(runtime.engine, ("held", i), context)
        if work == "mixed":
            feed(runtime.engine, "long", long_prompt[:case["start"]])
    if work == "generate":
        state["prompts"] = [p for p, _ in requests]
        kinds = [sampling_params(), sampling_params(temperature=0.8, seed=int(seed) % 1000 + 7),
                 sampling_params(temperature=0.8, top_k=40, top_p=0.9, seed=int(seed) % 1000 + 11)]
        state["sampling"] = [kinds[i % 3] for i in range(case["batch"])]
    if work in ("decode", "generate"):
        run(state)            # a serving program has its recordings of decode steps from its start
    return state


def run(state):
    case, engine, requests = state["case"], state["engine"], state["requests"]
    work = case["work"]
    if work == "generate":
        results = state["runtime"].generate_tokens(state["prompts"], case["steps"], state["sampling"], eos_token_id=None)
        return [torch.tensor(r.tokens) for r in results]
    if work == "prompt":
        out = engine.step([StepEntry(i, prompt, [len(prompt) - 1]) for i, (prompt, _) in enumerate(requests)])
        for i in range(len(requests)):
            engine.release(i)
        return {"logits": out.logits}
    if work == "mixed":
        portion = state["long"][case["start"]:]
        entries = [StepEntry("long", portion, [len(portion) - 1])]
        entries += [StepEntry(("held", i), new[:1], [0]) for i, (_, new) in enumerate(requests)]
        out = engine.step(entries)
        engine.truncate("long", case["start"])
        for i, (context, _) in enumerate(requests):
            engine.truncate(("held", i), len(context))
        return {"logits": out.logits}
    if work == "greedy":
        prompt = requests[0][0]
        logits = [engine.step([StepEntry(0, prompt, [len(prompt) - 1])]).logits]
        tokens = [ops.argmax(logits[0])]
        for _ in range(case["steps"]):
            logits.append(engine.step([StepEntry(0, [0], [0])], device_tokens=tokens[-1]).logits)
            tokens.append(ops.argmax(logits[-1]))
        engine.release(0)
        return {"logits": logits, "tokens": tokens}
    live = [("held", i) for i in range(len(requests))]
    if continues(case):
        live = [("going", i) for i in range(len(requests))]
        for i, request in enumerate(live):
            engine.fork(("held", i), request)
    logits = []
    for s in range(case["steps"]):
        logits.append(engine.step([StepEntry(r, [new[s]], [0]) for r, (_, new) in zip(live, requests)]).logits)
    for r, (context, _) in zip(live, requests):
        if continues(case):
            engine.release(r)
        else:
            engine.truncate(r, len(context))
    return {"logits": logits}


# ---- what a pass cannot do without ----------------------------------------------------------------------------------------
def work(case):
    """Matrices read once a step (of the experts, as many as the step's rows are expected to meet), the cache and the state
    of the live requests, logits written; two operations for every product a row takes part in."""
    c, size = config_of(case), 2 if case["dtype"] == "bfloat16" else 4
    dense = expert = experts = top = 0
    for name, shape in tensor_shapes(c).items():
        if len(shape) != 2 or name.split(".")[-1] in ("embed", "pos", "canon1", "canon2", "conv") or "embed_tokens" in name:
            continue
        if ".mlp.e" in name:
            expert += shape[0] * shape[1]
        elif name not in ("head", "lm_head.weight"):
            dense += shape[0] * shape[1]
    head = VOCAB * case["width"]
    if c.get("architecture") == "Zukinex":
        r = c["layers"][-1]["mlp"]["router"]
        experts, top = r["experts"] + r["identity"], r["top"]
    paged, state, window = [], 0, None
    if case["design"] == "qwen3":
        paged = [(c["num_attention_heads"], 2 * c["num_key_value_heads"] * 128)] * case["layers"]
    elif case["design"] == "zukinex":
        window = 1024 + 4
        paged = [(layer["mixer"]["heads"], 2 * layer["mixer"]["kv_heads"] * 128) for layer in c["layers"]]
    else:
        for layer in c["layers"]:
            m = layer["mixer"]
            if layer["type"] == "parallel":
                paged.append((m["left"]["heads"], 2 * m["left"]["kv_heads"] * 128))
                m = m["right"]
            state += m["heads"] * m["dim"] * m["vdim"]
    everyone = lengths(case)
    if case["work"] == "prompt":
        steps = [[(n, 0, 1) for n in everyone]]
    elif case["work"] == "mixed":
        steps = [[(case["portion"], case["start"], 1)] + [(1, n, 1) for n in everyone]]
    else:
        steps = [[(1, n + s, 1) for n in everyone] for s in range(case["steps"])]
        if case["work"] in ("greedy", "generate"):
            steps = [[(n, 0, 1) for n in everyone]] + steps[:case["steps"] - (case["work"] == "generate")]
    bytes_, flops = 0.0, 0.0
    for step in steps:
        rows, wanted = sum(n for n, _, _ in step), sum(w for _, _, w in step)
        met = 1.0 - (1.0 - top / experts) ** rows if experts else 0.0
        bytes_ += size * (dense + head + met * expert) + 4.0 * wanted * VOCAB + size * rows * case["width"]
        flops += 2.0 * rows * (dense + (expert * top / experts if experts else 0.0)) + 2.0 * wanted * head
        for n, start, _ in step:
            keys = start + n if window is None else min(start + n, window + n)
            pairs = n * start + n * (n + 1) / 2.0 if window is None else sum(min(start + i + 1, window) for i in range(n))
            for heads, row in paged:
                bytes_ += size * row * keys
                flops += 4.0 * heads * 128 * pairs
            bytes_ += (2 if start else 1) * 4.0 * state
            flops += 4.0 * n * state
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    """About four times what these paths are off ``exact`` (measured: 3e-6 in float32; in bfloat16 0.003 to 0.006, Pamevik 0.015 to
    0.022, whose read-outs are divided by their own root mean square); the largest of a million such values is some five
    times their root mean square."""
    if case["dtype"] == "float32":
        return {"rel": 1.2e-5, "max": 1e-4, "differ": 0.01}
    return {"rel": 0.03, "max": 0.5} if case["design"] == "pamevik" else {"rel": 0.02, "max": 0.15}


# ---- the same in 64 bits --------------------------------------------------------------------------------------------------
def _unit(x, eps):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps)


def _turn(x, dims, base, adjacent=False):
    """The first ``dims`` elements of x [requests, steps, heads, size] turned by their position, pairs half a turn apart or adjacent."""
    half = dims // 2
    freq = torch.tensor([base ** (-2.0 * i / dims) for i in range(half)], dtype=F64, device=x.device)
    angle = torch.arange(x.shape[1], dtype=F64, device=x.device)[:, None] * freq
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]
    a, b = (x[..., 0:dims:2], x[..., 1:dims:2]) if adjacent else (x[..., :half], x[..., half:dims])
    first, second = a * cos - b * sin, b * cos + a * sin
    turned = torch.stack([first, second], -1).flatten(-2) if adjacent else torch.cat([first, second], -1)
    return torch.cat([turned, x[..., dims:]], -1)


def _attend(q, k, v, scale, window=None, keep_first=0):
    """Causal softmax attention, [requests, steps, heads, size] each; a slice of the queries at a time."""
    share, out = q.shape[2] // k.shape[2], torch.empty_like(q)
    at = torch.arange(q.shape[1], device=q.device)
    for r in range(q.shape[0]):
        for g in range(k.shape[2]):
            for i in range(0, q.shape[1], 1024):
                mine, seen = q[r, i:i + 1024, g * share:(g + 1) * share], at[:min(i + 1024, q.shape[1])]
                score = torch.matmul(mine.transpose(0, 1), k[r, :len(seen), g].T) * scale
                gap = at[i:i + 1024, None] - seen[None]
                hidden = gap < 0
                if window is not None:
                    hidden |= (gap >= window) & (seen[None] >= keep_first)
                weights = torch.softmax(score.masked_fill_(hidden, -math.inf), -1)
                out[r, i:i + 1024, g * share:(g + 1) * share] = torch.matmul(weights, v[r, :len(seen), g]).transpose(0, 1)
    return out


def _qwen3(c, w, tokens):
    eps, d = c["rms_norm_eps"], c["head_dim"]
    x = w("model.embed_tokens.weight")[tokens]
    for i in range(c["num_hidden_layers"]):
        p = f"model.layers.{i}."
        h = _unit(x, eps) * w(p + "input_layernorm.weight")
        q, k, v = ((h @ w(p + f"self_attn.{n}_proj.weight").T).unflatten(-1, (-1, d)) for n in "qkv")
        q, k = (_turn(_unit(t, eps) * w(p + f"self_attn.{n}_norm.weight"), d, c["rope_theta"]) for t, n in ((q, "q"), (k, "k")))
        x = x + _attend(q, k, v, d ** -0.5).flatten(-2) @ w(p + "self_attn.o_proj.weight").T
        h = _unit(x, eps) * w(p + "post_attention_layernorm.weight")
        x = x + (torch.nn.functional.silu(h @ w(p + "mlp.gate_proj.weight").T) * (h @ w(p + "mlp.up_proj.weight").T)) @ w(p + "mlp.down_proj.weight").T
    return _unit(x, eps) * w("model.norm.weight"), w("lm_head.weight")


def _mixture(h, f, w, p):
    r = f["router"]
    rows = h.flatten(0, 1)
    score = torch.softmax(rows @ w(p + "router").T, -1)
    choice, count = score + w(p + "correction"), r["groups"]["count"]
    open_ = choice.unflatten(-1, (count, -1)).max(-1).values.topk(r["groups"]["keep"], -1).indices
    allowed = torch.zeros((len(rows), count), dtype=torch.bool, device=h.device).scatter_(1, open_, True)
    allowed = allowed.repeat_interleave(score.shape[1] // count, 1)
    chosen = choice.masked_fill(~allowed, -math.inf).topk(r["top"], -1).indices
    share = score.gather(1, chosen)
    share = torch.zeros_like(score).scatter_(1, chosen, share / (share.sum(-1, keepdim=True) + 1e-20))
    silu = torch.nn.functional.silu
    out = rows * share[:, r["experts"]:].sum(-1, keepdim=True) + \
        (silu(rows @ w(p + "shared.gate").T) * (rows @ w(p + "shared.up").T)) @ w(p + "shared.down").T
    for e in range(r["experts"]):
        at = share[:, e].nonzero().flatten()
        g = silu(rows[at] @ w(f"{p}e{e}.gate").T) * (rows[at] @ w(f"{p}e{e}.up").T)
        out.index_add_(0, at, share[at, e:e + 1] * (g @ w(f"{p}e{e}.down").T))
    return out.view_as(h)


def _zukinex(c, w, tokens):
    eps = c["norm"]["eps"]
    x = w("embed")[tokens] + w("pos")[:tokens.shape[1]]
    held = {}
    for i, layer in enumerate(c["layers"]):
        m, f, p, y = layer["mixer"], layer["mlp"], f"l{i}.mix.", f"l{i}.mlp."
        dims, base = m["rot"]["dims"], m["rot"]["base"]

        def heads(n):
            return (x @ w(p + n).T).unflatten(-1, (-1, m["dim"]))

        if m.get("kv_from") is None:
            held[i] = _turn(_unit(heads("k"), eps) * w(p + "k.norm"), dims, base, True), heads("v")
        k, v = held[m.get("kv_from", i)]
        q = _turn(_unit(heads("q"), eps) * w(p + "q.norm"), dims, base, True)
        a = _attend(q, k, v, m["scale"], m["mask"]["size"], m["mask"]["keep_first"]).flatten(-2) * torch.sigmoid(x @ w(p + "g").T)
        x = x + _unit(a @ w(p + "o").T, eps) * w(f"l{i}.norm1")
        if f["kind"] == "dense":
            b = (torch.nn.functional.gelu(x @ w(y + "gate").T, approximate="tanh") * (x @ w(y + "up").T)) @ w(y + "down").T
        else:
            b = _mixture(x, f, w, y)
        x = x + _unit(b, eps) * w(f"l{i}.norm2")
    return _unit(x, eps) * w("final.norm"), w("head")


def _taps(h, taps):
    """Causal convolution of every column over the rows; the last tap meets the row itself."""
    n, out = taps.shape[1], torch.zeros_like(h)
    for j in range(n):
        back = n - 1 - j
        out[:, back:] += h[:, :h.shape[1] - back] * taps[:, j]
    return out


def _decayed(q, k, v, log_w):
    """sum over s <= t of exp(log_w[t, s]) (q_t . k_s) v_s and of the same without v; log_w [requests, heads, steps, steps]."""
    seen = torch.ones(q.shape[1], q.shape[1], dtype=torch.bool, device=q.device).tril()
    mix = torch.einsum("rthd,rshd->rhts", q, k) * torch.where(seen, log_w, -math.inf).exp()
    return torch.einsum("rhts,rshv->rthv", mix, v), mix.sum(-1).transpose(1, 2)


def _mlstm(h, w, p, m, eps):
    dim, cap = m["dim"], m["gate_cap"]
    q, k, v = ((h @ w(p + n).T).unflatten(-1, (m["heads"], -1)) for n in "qkv")
    log_i, pre_f = (cap * torch.tanh((h @ w(p + n).T + w(p + n + ".b")) / cap) for n in "if")
    total = torch.nn.functional.logsigmoid(pre_f).cumsum(1).transpose(1, 2)                       # [requests, heads, steps]
    entry = log_i.transpose(1, 2) - total
    top = total + entry.cummax(-1).values.clamp_min(0.0)
    read, norm = _decayed(q * dim ** -0.5, k, v, (total - top)[..., :, None] + entry[..., None, :])
    floor = torch.maximum(norm.abs(), (-top).exp().transpose(1, 2))
    out = _unit(read / (floor[..., None] + 1e-6), eps).flatten(-2) * w(p + "norm")
    return (out * torch.sigmoid(h @ w(p + "g").T)) @ w(p + "o").T


def _side_by_side(h, w, p, m, eps):
    a, r = m["left"], m["right"]
    q, k, v = ((h @ w(p + "left." + n).T).unflatten(-1, (-1, 128)) for n in "qkv")
    q, k = (_turn(t, a["rot"]["dims"], a["rot"]["base"]) for t in (q, k))
    left = _attend(q, k, v, a["scale"]) * torch.sigmoid(h @ w(p + "left.g").T)[..., None]
    q, k, v = ((h @ w(p + "right." + n).T).unflatten(-1, (r["heads"], -1)) for n in "qkv")
    q, k = (_turn(t, r["rot"]["dims"], r["rot"]["base"]) for t in (q, k))
    at = torch.arange(h.shape[1], dtype=F64, device=h.device)
    rate = torch.tensor(r["decay"], dtype=F64, device=h.device).log()[None, :, None, None]
    right, _ = _decayed(q, k * r["dim"] ** -0.5, v, rate * (at[:, None] - at[None]))
    right = _unit(right, eps).flatten(-2) * torch.nn.functional.silu(h @ w(p + "right.g").T)
    return 0.5 * (_unit(left.flatten(-2) @ w(p + "left.o").T, eps) * w(p + "left.out")
                  + _unit(right @ w(p + "right.o").T, eps) * w(p + "right.out"))


def _channel_delta(h, w, p, m, eps):
    heads, share = m["heads"], m["heads"] // m["kv_heads"]
    q, k, v = (torch.nn.functional.silu(_taps(h @ w(p + n).T, w(p + n + ".conv"))) for n in "qkv")
    q, k = (t.unflatten(-1, (m["kv_heads"], -1)).repeat_interleave(share, 2) for t in (q, k))
    q, k = (t / torch.sqrt(t.square().sum(-1, keepdim=True) + 1e-6) for t in (q, k))
    q, v = q * m["dim"] ** -0.5, v.unflatten(-1, (heads, -1))
    beta = torch.sigmoid(h @ w(p + "b").T)
    step = torch.nn.functional.softplus((h @ w(p + "a1").T) @ w(p + "a2").T + w(p + "dt_bias")).unflatten(-1, (heads, -1))
    decay = torch.exp(-w(p + "A_log").exp()[:, None] * step)
    memory = torch.zeros(h.shape[0], heads, m["dim"], m["vdim"], dtype=F64, device=h.device)
    out = torch.empty_like(v)
    for t in range(h.shape[1]):
        memory *= decay[:, t, :, :, None]
        write = beta[:, t, :, None] * (v[:, t] - torch.matmul(k[:, t, :, None], memory)[:, :, 0])
        memory += k[:, t, :, :, None] * write[:, :, None]
        out[:, t] = torch.matmul(q[:, t, :, None], memory)[:, :, 0]
    gate = torch.sigmoid((h @ w(p + "g1").T) @ w(p + "g2").T).unflatten(-1, (heads, -1))
    return (_unit(out, eps) * w(p + "norm") * gate).flatten(-2) @ w(p + "o").T


def _pamevik(c, w, tokens):
    eps = c["norm"]["eps"]

    def norm(x, n):
        dev = x - x.mean(-1, keepdim=True)
        return dev / torch.sqrt(dev.square().mean(-1, keepdim=True) + eps) * w(n) + w(n + ".b")

    x = w("embed")[tokens]
    mixers = {"mlstm": _mlstm, "parallel": _side_by_side, "channel_delta": _channel_delta}
    for i, layer in enumerate(c["layers"]):
        p = f"l{i}."
        h = norm(x, p + "norm1")
        h = h + _taps(h, w(p + "canon1"))
        x = x + norm(mixers[layer["type"]](h, w, p + "mix.", layer["mixer"], eps), p + "norm1b")
        if layer["mlp"]:
            h = norm(x, p + "norm2")
            h = h + _taps(h, w(p + "canon2"))
            x = x + norm(torch.relu(h @ w(p + "mlp.up").T).square() @ w(p + "mlp.down").T, p + "norm2b")
    return norm(x, "final.norm"), w("head")


def exact(case, seed):
    if case["work"] == "generate":
        return None                     # tokens only
    weights, c = make_weights(case, seed), config_of(case)
    forward = {"qwen3": _qwen3, "pamevik": _pamevik, "zukinex": _zukinex}[case["design"]]

    def logits(sequences, last):
        """Logits of the last ``last`` positions of every sequence, [sequences, last, vocab]."""
        found = [None] * len(sequences)
        order = sorted(range(len(sequences)), key=lambda i: len(sequences[i]))
        while order:
            group, longest = [], len(sequences[order[-1]])
            while order and (not group or (len(group) + 1) * longest <= 8192):
                group.append(order.pop())
            padded = [sequences[i] + [0] * (longest - len(sequences[i])) for i in group]      # nothing looks ahead
            y, head = forward(c, lambda n: weights[n].to(F64), torch.tensor(padded, device=DEVICE))
            for row, i in enumerate(group):
                n = len(sequences[i])
                found[i] = y[row, n - last:n] @ head.T
        return torch.stack(found)

    requests, long_prompt = tokens_of(case, seed)
    if case["work"] == "prompt":
        return {"logits": logits([p for p, _ in requests], 1)[:, 0]}
    if case["work"] == "mixed":
        return {"logits": logits([long_prompt] + [p + new[:1] for p, new in requests], 1)[:, 0]}
    if case["work"] == "greedy":
        tokens, found, chosen = list(requests[0][0]), [], []
        for _ in range(case["steps"] + 1):
            found.append(logits([tokens], 1)[0])
            chosen.append(found[-1].argmax(-1).to(torch.int32))
            tokens.append(int(chosen[-1]))
        return {"logits": found, "tokens": chosen}
    found = logits([p + new for p, new in requests], case["steps"])
    return {"logits": [found[:, s] for s in range(case["steps"])]}
