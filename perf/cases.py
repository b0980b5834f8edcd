"""What a user of this engine has it do, as cases that can be timed and checked.

A case is a model, a precision and a set of sequences taken through the engine's public entry points: prompts in one step
(``prefill``), prompts and then greedy decoding with the tokens fed back on the device (``generate``), prompts that arrive while
others decode (``serve``), and prompts followed by tokens that are given (``follow``, what a trace replay and a scoring program
do). The models are the GPT-2 shapes (small, medium, XL) and three of the other designs at GPT-2 small's width and depth, all with
random weights; token ids are uniform. Every pass opens its sequences and gives them back, so a pass can be repeated.

``exact`` is the same in 64 bits, whole sequences, written out in torch."""

from __future__ import annotations

import math

import numpy as np
import torch

from mini_llm_amd.config import config_from_dict
from mini_llm_amd.engine import StepEntry
from mini_llm_amd.engine.engine import Engine, EngineOptions
from mini_llm_amd.engine.loading import build_model
from mini_llm_amd.weights import bind_tensors

DEVICE = "cuda:0"
VOCAB, POSITIONS, SESSIONS = 50257, 1024, 64
STEP_TOKENS = 2048    # tokens of a step that reads prompts (the engine's own default)
SERVE_TOKENS = 512    # the same where prompts arrive beside decoding requests, which should not wait long


# ---- models ---------------------------------------------------------------------------------------------------------------
def _gpt2(layers: int, width: int) -> dict:
    return {"architectures": ["GPT2LMHeadModel"], "n_layer": layers, "n_embd": width, "n_head": width // 64, "n_inner": 4 * width,
            "vocab_size": VOCAB, "n_positions": POSITIONS, "layer_norm_epsilon": 1e-5, "activation_function": "gelu_new"}


def _gimozen(width: int, layers: int) -> dict:
    """Attention with normed heads; every fourth layer attention over a latent, every second of those over the rows of the one before."""
    heads, ff = width // 64, -(-(8 * width // 3) // 64) * 64
    rot = {"dims": 32, "base": 10000.0, "scaling": {"factor": 4.0, "original": 1024, "fast": 32.0, "slow": 1.0}}
    out, latent_at = [], None
    for index in range(layers):
        if index % 4 == 2:
            mixer = {"heads": heads, "dim": 64, "rot_dim": 32, "vdim": 64, "kv_rank": 256, "rot": rot, "scale": 96 ** -0.5}
            if latent_at is not None:
                mixer["kv_from"], latent_at = latent_at, None
            else:
                latent_at = index
            out.append({"type": "latent_attention", "mixer": mixer, "mlp": {"kind": "dense", "ff": ff}})
        else:
            out.append({"type": "attention", "mlp": {"kind": "dense", "ff": ff},
                        "mixer": {"heads": heads, "kv_heads": heads, "dim": 64, "vdim": 64, "scale": 0.125, "q_temp": {"coef": 0.1, "every": 256}}})
    return {"architecture": "Gimozen", "vocab": VOCAB, "width": width, "embedding": {"scale": width ** 0.5}, "norm": {"eps": 1e-5},
            "postln_alpha": 1.0, "layers": out}


def _ketolix(width: int, layers: int) -> dict:
    """In fours: a matrix memory, two layers of attention over a window, attention beside a decayed recurrence."""
    heads, wide = width // 64, max(1, width // 128)
    mlp = {"kind": "dense", "ff": -(-(8 * width // 3) // 64) * 64}
    rot = {"dims": 64, "base": 500000.0, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 512}}
    attention = {"type": "attention", "mlp": mlp, "mixer": {"heads": heads, "kv_heads": max(1, heads // 4), "dim": 64, "vdim": 64, "scale": 0.125,
                                                           "softcap": 30.0, "mask": {"size": 512}, "rot": rot, "v_mix": True}}
    memory = {"type": "mlstm", "mlp": mlp, "mixer": {"heads": wide, "dim": 64, "vdim": 128, "gate_cap": 15.0}}
    parallel = {"type": "parallel", "mlp": mlp, "mixer": {
        "left": {"heads": heads, "kv_heads": max(1, heads // 4), "dim": 64, "vdim": 64, "scale": 0.125, "conv": 4, "mask": {"size": 512},
                 "rot": {"dims": 32, "base": 500000.0}},
        "right": {"heads": wide, "dim": 64, "vdim": 128, "decay": [1.0 - 0.1 ** (1.0 + 2.0 * i / max(1, wide - 1)) for i in range(wide)]},
        "left_scale": 0.7, "right_scale": 0.7}}
    pattern = [memory, attention, attention, parallel]
    return {"architecture": "Ketolix", "vocab": VOCAB, "width": width, "norm": {"eps": 1e-5}, "layers": [pattern[i % 4] for i in range(layers)]}


def _goletar(width: int, layers: int) -> dict:
    """In turn: a gated recurrence, and attention over a latent; eight routed experts of which two are picked."""
    mlp = {"kind": "moe", "expert": {"ff": -(-(4 * width // 3) // 64) * 64, "limit": 7.0}, "router": {"experts": 8, "top": 2}}
    latent = {"heads": width // 64, "dim": 64, "rot_dim": 32, "vdim": 64, "kv_rank": 256, "rot": {"dims": 32, "base": 10000.0}, "scale": 96 ** -0.5}
    return {"architecture": "Goletar", "vocab": VOCAB, "width": width, "embedding": {"bigram": {"buckets": 65521, "mul_prev": 7919, "mul_cur": 104729}},
            "norm": {"eps": 1e-5},
            "layers": [{"type": "latent_attention", "mixer": latent, "mlp": mlp} if index % 2 else {"type": "mingru", "mixer": {"width": 5 * width // 4}, "mlp": mlp}
                       for index in range(layers)]}


MODELS = {"gpt2-small": _gpt2(12, 768), "gpt2-medium": _gpt2(24, 1024), "gpt2-xl": _gpt2(48, 1600),
          "gimozen": _gimozen(768, 12), "ketolix": _ketolix(768, 12), "goletar": _goletar(768, 12)}


# ---- cases ----------------------------------------------------------------------------------------------------------------
def _case(name, model, dtype, kind, sequences, shortest, longest, new=0) -> dict:
    case = {"name": name} if name else {}
    case.update(model=model, dtype=dtype, kind=kind, sequences=sequences, shortest=shortest, longest=longest, new=new)
    return case


def listed() -> list:
    return [
        # one short completion on the command line: latency of single tokens, and the smallest prompt step
        _case("complete-small-bf16", "gpt2-small", "bfloat16", "generate", 1, 17, 17, 16),
        # the headline: eight sequences from 512-token prompts, greedy, and the same in 32-bit
        _case("generate-small-bf16-b8", "gpt2-small", "bfloat16", "generate", 8, 512, 512, 48),
        _case("generate-small-f32-b8", "gpt2-small", "float32", "generate", 8, 512, 512, 32),
        # a full house of short conversations on the medium shape
        _case("generate-medium-bf16-b64", "gpt2-medium", "bfloat16", "generate", 64, 65, 190, 32),
        # the largest model at the largest batch: weights and products of 64 rows
        _case("generate-xl-bf16-b64", "gpt2-xl", "bfloat16", "generate", 64, 33, 96, 16),
        # documents read in one step: two whole contexts, and ragged ones in 32-bit
        _case("prefill-small-bf16", "gpt2-small", "bfloat16", "prefill", 2, 1024, 1024),
        _case("prefill-small-f32-ragged", "gpt2-small", "float32", "prefill", 5, 67, 1001),
        _case("prefill-xl-bf16", "gpt2-xl", "bfloat16", "prefill", 2, 1024, 1024),
        # continuous batching: prompts of 32 to 768 arrive in portions beside the requests that already decode
        _case("serve-medium-bf16", "gpt2-medium", "bfloat16", "serve", 24, 32, 768, 8),
        # the other designs: a long document, a replayed trace over a matrix memory and windows, and a ragged one through experts
        _case("prefill-gimozen-bf16", "gimozen", "bfloat16", "prefill", 2, 1024, 1024),
        _case("follow-ketolix-f32-b8", "ketolix", "float32", "follow", 8, 300, 513, 16),
        _case("follow-goletar-f32-ragged", "goletar", "float32", "follow", 6, 19, 640, 16),
    ]


def _seconds(case) -> float:
    """A rough guess of a pass's cost, to compare cases by."""
    w = work(case)
    return w["bytes"] / 3e12 + w["flops"] / (4e14 if case["dtype"] == "bfloat16" else 6e13) + len(_plan(case)) * _depth(case["model"]) * 40e-6


def draw(rng) -> dict:
    most = max(_seconds(c) for c in listed())
    spread = lambda lo, hi: min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))
    while True:
        model = rng.choice(["gpt2-small", "gpt2-small", "gpt2-small", "gpt2-medium", "gpt2-medium", "gpt2-xl", "gimozen", "ketolix", "goletar"])
        gpt2 = model.startswith("gpt2")
        # random routers have close calls that bfloat16 decides either way, and Ketolix's norms behind every branch make bfloat16's
        # rounding several percent of its logits: these two run in 32-bit, where outputs can be compared
        dtype = "float32" if model in ("goletar", "ketolix") else rng.choice(["bfloat16", "bfloat16", "float32"]) if model != "gpt2-xl" else "bfloat16"
        kind = rng.choice(["generate", "generate", "prefill", "serve"] if gpt2 else ["prefill", "follow"])
        sequences = spread(4, 48) if kind == "serve" else spread(1, 12) if kind == "prefill" else spread(1, 64)
        longest = spread(8, 1000 if kind != "serve" else 768)
        shortest = rng.choice([longest, spread(min(5, longest), longest)])
        case = _case(None, model, dtype, kind, sequences, shortest, longest, 0 if kind == "prefill" else spread(4, 24) if kind != "serve" else spread(2, 8))
        total = sum(_lengths(case))
        if total <= (4096 if kind == "prefill" else 16384) and _seconds(case) <= most:
            return case


def _lengths(case) -> list:
    """Prompt lengths between the shortest and the longest, in no order of size; the longest is among them."""
    n, lo, hi = case["sequences"], case["shortest"], case["longest"]
    if n == 1:
        return [hi]
    even = [int(round(lo + (hi - lo) * k / (n - 1))) for k in range(n)]
    stride = next(s for s in range(max(1, (2 * n) // 3), 2 * n + 2) if math.gcd(s, n) == 1)
    return [even[(n - 1 + k * stride) % n] for k in range(n)]


def _plan(case) -> list:
    """The steps of a pass: per step the portions [(sequence, from, to)] of prompts it reads and the sequences that bring one token more."""
    lengths, steps = _lengths(case), []
    serving = case["kind"] == "serve"
    budget = SERVE_TOKENS if serving else STEP_TOKENS if case["kind"] != "prefill" else 1 << 30
    at, done, running = 0, 0, []
    while at < len(lengths):
        room, portions, beside = budget - (len(running) if serving else 0), [], list(running) if serving else []
        while at < len(lengths) and room > 0:
            take = min(room, lengths[at] - done)
            portions.append((at, done, done + take))
            done, room = done + take, room - take
            if done == lengths[at]:
                running.append(at)
                at, done = at + 1, 0
        steps.append((portions, beside))
    steps += [([], list(range(len(lengths))))] * case["new"]
    return steps


# ---- one pass -------------------------------------------------------------------------------------------------------------
_engines: dict = {}


def _tensors(model, name: str, dtype: str) -> dict:
    """Random weights of the model's own recipe, as a file in the precision holds them. GPT-2's token table alone is drawn as wide as the
    trained one is (0.14): a greedy choice then is as clear as a trained model's, and not a matter of the last bit of 50,257 sums."""
    generator = torch.Generator(device=DEVICE).manual_seed(1000 + sorted(MODELS).index(name))
    out = {}
    for tensor, spec in model.named_tensor_specs().items():
        std = 0.14 if tensor == "wte.weight" else spec.init.std
        values = torch.randn(tuple(spec.shape), generator=generator, device=DEVICE) * std + spec.init.mean
        if dtype == "bfloat16" and spec.role in ("matrix", "table"):
            values = values.bfloat16().float()
        out[tensor] = values
    return out


def _engine(name: str, dtype: str) -> Engine:
    """A program holds its model for as long as it runs; inputs come and go."""
    if (name, dtype) not in _engines:
        model = build_model(config_from_dict(MODELS[name]), dtype)
        bind_tensors(model, _tensors(model, name, dtype), torch.device(DEVICE))
        _engines[name, dtype] = Engine(model=model, options=EngineOptions(dtype=dtype, max_sessions=SESSIONS, max_tokens=SESSIONS * POSITIONS, max_length=POSITIONS))
    return _engines[name, dtype]


def _tokens(case, seed: int) -> list:
    """Per sequence its prompt and, where tokens are given, those behind it."""
    rng = np.random.default_rng([seed, 77])
    more = case["new"] if case["kind"] == "follow" else 0
    return [rng.integers(0, VOCAB, n + more).astype(np.int32) for n in _lengths(case)]


def prepare(case, seed):
    return {"engine": _engine(case["model"], case["dtype"]), "kind": case["kind"], "lengths": _lengths(case), "plan": _plan(case), "tokens": _tokens(case, seed)}


def run(state):
    engine, kind, lengths, tokens = state["engine"], state["kind"], state["lengths"], state["tokens"]
    greedy = kind in ("generate", "serve")
    handles = [engine.try_take_cache() for _ in lengths]
    chosen, ahead, queued, fed = [], None, 0, list(lengths)
    for number, (portions, beside) in enumerate(state["plan"]):
        last = number == len(state["plan"]) - 1
        if greedy and not portions and not last:   # plain decoding: queued, its tokens taken from the device
            engine.decode_batch_enqueue(handles)
            queued += 1
            if ahead is not None:
                chosen += ahead.tolist()
                ahead = None
            if queued > 1:
                chosen += engine.take()
                queued -= 1
            continue
        entries = []
        for i in beside:
            if greedy:
                entries.append(StepEntry(handles[i], [0], [0], from_slot=True))
            else:
                entries.append(StepEntry(handles[i], [int(tokens[i][fed[i]])], [0]))
                fed[i] += 1
        for i, lo, hi in portions:
            entries.append(StepEntry(handles[i], tokens[i][lo:hi], [hi - lo - 1] if hi == lengths[i] else []))
        result = engine.runner.step(entries, choose=greedy and not last)
        if ahead is not None:
            chosen += ahead.tolist()
            ahead = None
        if greedy and not last:
            ahead = result   # read once the next step is under way
        elif last:
            logits = result
    for _ in range(queued):
        chosen += engine.take()
    for handle in handles:
        engine.release_cache(handle)
    return {"tokens": np.asarray(chosen, dtype=np.int32), "logits": logits} if greedy else {"logits": logits}


# ---- what a pass cannot do without ------------------------------------------------------------------------------------------
def _depth(name: str) -> int:
    raw = MODELS[name]
    return raw.get("n_layer") or len(raw["layers"])


def _shape(name: str):
    """(matrix elements every token needs, expert elements, share of them a token picks, head elements, [(pair flops, row elements,
    window)] per layer that keeps keys, state elements and flops a token of the recurrences)."""
    raw = MODELS[name]
    if "n_layer" in raw:
        d, ff, n = raw["n_embd"], raw["n_inner"], raw["n_layer"]
        return n * (4 * d * d + 2 * d * ff), 0, 1.0, VOCAB * d, [(4 * d, 2 * d, None)] * n, 0, 0
    d, common, experts, share, layers, state, state_flops = raw["width"], 0, 0, 1.0, [], 0, 0

    def memory(m):
        nonlocal common, state, state_flops
        common += d * (2 * m["heads"] * m["dim"] + 3 * m["heads"] * m["vdim"])
        state += m["heads"] * m["dim"] * m["vdim"]
        state_flops += 4 * m["heads"] * m["dim"] * m["vdim"]

    def attend(m):
        nonlocal common
        H, G = m["heads"], m["kv_heads"]
        own_values = "conv" not in m
        common += d * (H * m["dim"] + G * m["dim"] + (G * m["vdim"] if own_values else 0) + H * m["vdim"])
        layers.append((2 * H * (m["dim"] + m["vdim"]), G * (m["dim"] + m["vdim"]), (m.get("mask") or {}).get("size")))

    for layer in raw["layers"]:
        m, mlp = layer["mixer"], layer["mlp"]
        if layer["type"] == "latent_attention":
            H, r, dim, rot, vdim = m["heads"], m["kv_rank"], m["dim"], m["rot_dim"], m["vdim"]
            gate = d * H * (vdim if raw["architecture"] == "Gimozen" else 1)
            common += d * H * (dim + rot) + (0 if "kv_from" in m else d * (r + rot)) + H * r * (dim + vdim) + gate + d * H * vdim
            layers.append((2 * H * (dim + rot + vdim), r + rot, None))
        elif layer["type"] == "attention":
            attend(m)
        elif layer["type"] == "mlstm":
            memory(m)
        elif layer["type"] == "parallel":
            attend(m["left"])
            memory(m["right"])
        else:   # mingru
            common += 4 * d * m["width"]
            state += m["width"]
        if mlp["kind"] == "dense":
            common += 3 * d * mlp["ff"]
        else:
            E = mlp["router"]["experts"]
            common += d * E
            experts += E * 3 * d * mlp["expert"]["ff"]
            share = mlp["router"]["top"] / E
    return common, experts, share, VOCAB * d, layers, state, state_flops


def work(case) -> dict:
    """Per step: the weights it uses once, the cached rows its tokens attend to once, its new rows written once, states read and
    written; the multiply-adds of the products, of the pairs a mask shows and of the logits that are asked for."""
    common, experts, share, head, layers, state, state_flops = _shape(case["model"])
    e = 2 if case["dtype"] == "bfloat16" else 4
    lengths, stored = _lengths(case), [0] * case["sequences"]
    flops = bytes_ = 0.0
    for portions, beside in _plan(case):
        parts = [(i, hi - lo) for i, lo, hi in portions] + [(i, 1) for i in beside]
        rows = sum(n for _, n in parts)
        wanted = len(beside) + sum(1 for i, lo, hi in portions if hi == lengths[i])
        flops += 2.0 * rows * (common + experts * share) + rows * state_flops + 2.0 * wanted * head
        bytes_ += e * (common + experts * (1.0 - (1.0 - share) ** rows) + (head if wanted else 0)) + 4.0 * wanted * VOCAB
        bytes_ += len(parts) * 2 * 4.0 * state
        for i, n in parts:
            for pair, row, window in layers:
                seen = [min(k + 1, window or k + 1) for k in (stored[i], stored[i] + n - 1)]
                flops += pair * n * (seen[0] + seen[1]) / 2
                reach = stored[i] + n if window is None else min(stored[i] + n, window + n)
                bytes_ += e * row * (reach + n)
            stored[i] += n
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    """Four times the distance from ``exact`` that was measured: in 32-bit 1 to 3e-6 (sums of up to 6,400 in some order), 7e-6 behind
    Ketolix's norms on every branch; in bfloat16, whose rows between kernels are rounded to 8 bits at every layer, 4e-3 for GPT-2 and 1.4e-2
    for Gimozen. The largest single difference is some five times the mean one over millions of logits."""
    if case["dtype"] == "float32":
        rel = 3e-5 if case["model"] == "ketolix" else 1e-5
    else:
        rel = 3e-2 if case["model"] == "gimozen" else 1.6e-2
    return {"rel": rel, "max": 8 * rel, "differ": 0.005}


# ---- the same in 64 bits ----------------------------------------------------------------------------------------------------
def exact(case, seed):
    raw, name = MODELS[case["model"]], case["model"]
    model = build_model(config_from_dict(raw), "float32")   # for the tensors' names and shapes alone
    w = {k: v.double() for k, v in _tensors(model, name, case["dtype"]).items()}
    sequences, lengths = _tokens(case, seed), _lengths(case)
    if "n_layer" in raw:
        steps = [0] * len(lengths)   # greedy tokens each sequence is fed
        for _, beside in _plan(case):
            for i in beside:
                steps[i] += 1
        return {"tokens": None, "logits": _exact_gpt2(raw, w, sequences, steps)} if case["kind"] != "prefill" else {"logits": _exact_gpt2(raw, w, sequences, steps)}
    whole = _padded(sequences)
    x = {"gimozen": _exact_gimozen, "ketolix": _exact_ketolix, "goletar": _exact_goletar}[name](raw, w, whole)
    rows = torch.stack([x[i, len(s) - 1] for i, s in enumerate(sequences)])
    return {"logits": rows @ w["embed" if name == "ketolix" else "head"].T}


def _padded(sequences):
    """[sequences, longest], zeros behind the shorter ones: nothing looks ahead, so they change nothing."""
    out = torch.zeros(len(sequences), max(len(s) for s in sequences), dtype=torch.long)
    for i, s in enumerate(sequences):
        out[i, : len(s)] = torch.from_numpy(s.astype(np.int64))
    return out.to(DEVICE)


def _layernorm(x, g, b, eps):
    c = x - x.mean(-1, keepdim=True)
    return c / torch.sqrt((c * c).mean(-1, keepdim=True) + eps) * g + b


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _attend(q, k, v, scale, first, window=None, cap=None, sink=None):
    """q [B, T, H, a], k [B, S, G, a], v [B, S, G, c] -> [B, T, H, c]; the query at row t of sequence b stands at position first[b] + t."""
    B, T, H, _ = q.shape
    S, G = k.shape[1], k.shape[2]
    at = first[:, None] + torch.arange(T, device=q.device)[None, :]
    keys = torch.arange(S, device=q.device)
    hidden = keys[None, None, :] > at[:, :, None]
    if window is not None:
        hidden = hidden | (keys[None, None, :] <= at[:, :, None] - window)
    out = []
    for h in range(H):
        g = h // (H // G)
        s = torch.matmul(q[:, :, h].contiguous(), k[:, :, g].transpose(1, 2).contiguous()) * scale
        if cap is not None:
            s = cap * torch.tanh(s / cap)
        s = s.masked_fill(hidden, -math.inf)
        if sink is not None:   # a key without a value
            s = torch.cat([s, sink[h].expand(B, T, 1)], dim=2)
        p = torch.softmax(s, dim=2)[:, :, :S].contiguous()
        out.append(torch.matmul(p, v[:, :, g].contiguous()))
    return torch.stack(out, dim=2)


def _start(tokens):
    return torch.zeros(tokens.shape[0], dtype=torch.long, device=tokens.device)


def _exact_gpt2(raw, w, sequences, steps):
    """Greedy from the prompts, keys and values kept; the logits behind the last token that each sequence is fed."""
    H, eps = raw["n_head"], raw["layer_norm_epsilon"]
    lengths = torch.tensor([len(s) for s in sequences], device=DEVICE)
    B, rows = len(sequences), torch.arange(len(sequences), device=DEVICE)
    kept = [[torch.zeros(B, int(lengths.max()) + max(steps), H, raw["n_embd"] // H, dtype=torch.float64, device=DEVICE) for _ in range(2)] for _ in range(raw["n_layer"])]

    def forward(tokens, first):
        T = tokens.shape[1]
        at = first[:, None] + torch.arange(T, device=DEVICE)[None, :]
        x = w["wte.weight"][tokens] + w["wpe.weight"][at.clamp(max=raw["n_positions"] - 1)]
        for i in range(raw["n_layer"]):
            p = f"h.{i}."
            h = _layernorm(x, w[p + "ln_1.weight"], w[p + "ln_1.bias"], eps)
            q, k, v = (t.reshape(B, T, H, -1) for t in (h @ w[p + "attn.c_attn.weight"] + w[p + "attn.c_attn.bias"]).chunk(3, dim=2))
            kept[i][0][rows[:, None], at], kept[i][1][rows[:, None], at] = k, v
            reach = int(at.max()) + 1
            if T > 1:
                o = _attend(q, kept[i][0][:, :reach], kept[i][1][:, :reach], q.shape[3] ** -0.5, first)
            else:   # one token a sequence: all heads at once
                s = (q * kept[i][0][:, :reach]).sum(3) * q.shape[3] ** -0.5
                s = s.masked_fill((torch.arange(reach, device=DEVICE)[None, :] > first[:, None])[:, :, None], -math.inf)
                o = (torch.softmax(s, dim=1)[..., None] * kept[i][1][:, :reach]).sum(1, keepdim=True)
            x = x + o.reshape(B, T, -1) @ w[p + "attn.c_proj.weight"] + w[p + "attn.c_proj.bias"]
            h = _layernorm(x, w[p + "ln_2.weight"], w[p + "ln_2.bias"], eps)
            u = h @ w[p + "mlp.c_fc.weight"] + w[p + "mlp.c_fc.bias"]
            u = 0.5 * u * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (u + 0.044715 * u ** 3)))
            x = x + u @ w[p + "mlp.c_proj.weight"] + w[p + "mlp.c_proj.bias"]
        return x

    def logits_of(x):
        return _layernorm(x, w["ln_f.weight"], w["ln_f.bias"], eps) @ w["wte.weight"].T

    logits = logits_of(forward(_padded(sequences), _start(rows[:, None]))[rows, lengths - 1])
    out = logits.clone()
    wanted = torch.tensor(steps, device=DEVICE)
    for n in range(1, max(steps) + 1):
        logits = logits_of(forward(logits.argmax(1)[:, None], lengths + n - 1)[:, 0])
        out = torch.where((wanted == n)[:, None], logits, out)
    return out


def _turn(x, freq, magnitude=1.0, halves=False):
    """x [B, T, heads, size]: pairs of the first 2 len(freq) elements turn by position * freq; neighbours, or element i with the one half further."""
    n = len(freq)
    angle = torch.arange(x.shape[1], dtype=torch.float64, device=x.device)[:, None] * freq[None, :]
    c, s = torch.cos(angle)[None, :, None, :] * magnitude, torch.sin(angle)[None, :, None, :] * magnitude
    if halves:
        u, v = x[..., :n], x[..., n : 2 * n]
        return torch.cat([u * c - v * s, v * c + u * s, x[..., 2 * n :]], dim=3)
    out = x.clone()
    u, v = x[..., 0 : 2 * n : 2], x[..., 1 : 2 * n : 2]
    out[..., 0 : 2 * n : 2], out[..., 1 : 2 * n : 2] = u * c - v * s, v * c + u * s
    return out


def _frequencies(dims, base):
    return float(base) ** (-2.0 * torch.arange(dims // 2, dtype=torch.float64, device=DEVICE) / dims)


def _latent(h, x, w, m, eps, freq, magnitude, halves, kept):
    """Attention over a latent: (the heads' outputs, what the layer keeps of its rows)."""
    B, T, _ = h.shape
    H, dim, r, rot = m["heads"], m["dim"], m["kv_rank"], m["rot_dim"]
    if kept is None:
        both = h @ w["dkv"].T
        kept = _rms(both[..., :r], eps) * w["dkv.norm"], _turn(both[..., None, r:], freq, magnitude, halves)
    c, k_rot = kept
    q = (h @ w["q"].T).reshape(B, T, H, dim + rot)
    q = torch.cat([q[..., :dim], _turn(q[..., dim:], freq, magnitude, halves)], dim=3)
    k = torch.cat([(c @ w["uk"].T).reshape(B, T, H, dim), k_rot.expand(B, T, H, rot)], dim=3)
    return _attend(q, k, (c @ w["uv"].T).reshape(B, T, H, -1), m["scale"], _start(x), sink=w["sink"]), kept


def _under(w, prefix):
    return {k[len(prefix):]: v for k, v in w.items() if k.startswith(prefix)}


def _gated(h, w):
    g = h @ w["gate"].T
    return (g * torch.sigmoid(g) * (h @ w["up"].T)) @ w["down"].T


def _exact_gimozen(raw, w, tokens):
    eps, alpha, kept = raw["norm"]["eps"], raw["postln_alpha"], {}
    B, T = tokens.shape
    x = w["embed"][tokens] * raw["embedding"]["scale"]
    for index, layer in enumerate(raw["layers"]):
        m, mix, p = layer["mixer"], _under(w, f"l{index}.mix."), f"l{index}."
        if layer["type"] == "attention":
            q, k, v = ((x @ mix[n].T).reshape(B, T, -1, 64) for n in "qkv")
            position = torch.arange(T, dtype=torch.float64, device=DEVICE)
            temperature = 1.0 + m["q_temp"]["coef"] * torch.log(torch.floor((position + 1) / m["q_temp"]["every"]) + 1.0)
            q = _rms(q, eps) * mix["q.norm"] * temperature[None, :, None, None]
            mixed = _attend(q, _rms(k, eps) * mix["k.norm"], v, m["scale"], _start(tokens)).reshape(B, T, -1)
        else:
            dims, base, scaling = m["rot"]["dims"], m["rot"]["base"], m["rot"]["scaling"]
            pair = lambda turns: dims * math.log(scaling["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(base))
            lo, hi = max(math.floor(pair(scaling["fast"])), 0), min(math.ceil(pair(scaling["slow"])), dims - 1)
            ramp = ((torch.arange(dims // 2, dtype=torch.float64, device=DEVICE) - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
            freq = _frequencies(dims, base)
            freq = freq / scaling["factor"] * ramp + freq * (1.0 - ramp)
            mixed, rows = _latent(x, tokens, mix, m, eps, freq, 0.1 * math.log(scaling["factor"]) + 1.0, True, kept.get(m.get("kv_from")))
            kept[index] = rows
            mixed = mixed.reshape(B, T, -1) * torch.sigmoid(x @ mix["g"].T)
        x = _rms(alpha * x + mixed @ mix["o"].T, eps) * (1.0 + w[p + "norm1"])
        x = _rms(alpha * x + _gated(x, _under(w, p + "mlp.")), eps) * (1.0 + w[p + "norm2"])
    return _rms(x, eps) * (1.0 + w["final.norm"])


def _exact_ketolix(raw, w, tokens):
    eps, v_first = raw["norm"]["eps"], None
    B, T = tokens.shape
    x = w["embed"][tokens]

    def frequencies(rot):
        f, scaling = _frequencies(rot["dims"], rot["base"]), rot.get("scaling")
        if not scaling:
            return f
        turns = scaling["original"] * f / (2.0 * math.pi)
        share = ((turns - scaling["low"]) / (scaling["high"] - scaling["low"])).clamp(0.0, 1.0)
        return (1.0 - share) * f / scaling["factor"] + share * f

    for index, layer in enumerate(raw["layers"]):
        m, mix, p = layer["mixer"], _under(w, f"l{index}.mix."), f"l{index}."
        if layer["type"] == "mlstm":
            H, dim = m["heads"], m["dim"]
            q, k, v = ((x @ mix[n].T).reshape(B, T, H, -1) for n in "qkv")
            q, cap = q * dim ** -0.5, m["gate_cap"]
            log_in = cap * torch.tanh((x @ mix["i"].T + mix["i.b"]) / cap)
            log_keep = torch.nn.functional.logsigmoid(cap * torch.tanh((x @ mix["f"].T + mix["f.b"]) / cap))
            S, n, top = x.new_zeros(B, H, dim, v.shape[3]), x.new_zeros(B, H, dim), x.new_zeros(B, H)
            out = []
            for t in range(T):
                new = torch.maximum(log_keep[:, t] + top, log_in[:, t])
                keep, take = torch.exp(log_keep[:, t] + top - new), torch.exp(log_in[:, t] - new)
                S = keep[..., None, None] * S + (take[..., None] * k[:, t])[..., None] * v[:, t][..., None, :]
                n, top = keep[..., None] * n + take[..., None] * k[:, t], new
                weight = torch.maximum((n * q[:, t]).sum(2).abs(), torch.exp(-top)) + 1e-6
                out.append((S * q[:, t][..., None]).sum(2) / weight[..., None])
            o = _rms(torch.stack(out, dim=1), eps).reshape(B, T, -1) * mix["norm"] * torch.sigmoid(x @ mix["g"].T)
            branch = o @ mix["o"].T
        elif layer["type"] == "attention":
            H, G = m["heads"], m["kv_heads"]
            q, k = _rms(x @ mix["q"].T, eps) * mix["q.norm"], _rms(x @ mix["k"].T, eps) * mix["k.norm"]
            v = x @ mix["v"].T
            v = v if v_first is None else (1.0 - mix["vmix"]) * v + mix["vmix"] * v_first
            v_first = v if v_first is None else v_first
            f = frequencies(m["rot"])
            o = _attend(_turn(q.reshape(B, T, H, -1), f), _turn(k.reshape(B, T, G, -1), f), v.reshape(B, T, G, -1), m["scale"], _start(tokens), m["mask"]["size"], m["softcap"], mix["sink"])
            branch = o.reshape(B, T, -1) @ mix["o"].T
        else:
            left, right = m["left"], m["right"]
            H, G = left["heads"], left["kv_heads"]

            def convolved(u, taps):
                past = torch.cat([u.new_zeros(B, taps.shape[1] - 1, u.shape[2]), u], dim=1)
                return sum(past[:, j : j + T] * taps[:, j] for j in range(taps.shape[1]))

            q = convolved(x @ mix["left.q"].T + mix["left.q.b"], mix["left.q.conv"])
            k = convolved(x @ mix["left.k"].T + mix["left.k.b"], mix["left.k.conv"])
            f = frequencies(left["rot"])
            qn = _turn((_rms(q, eps) * mix["left.q.norm"]).reshape(B, T, H, -1), f)
            kn = _turn((_rms(k, eps) * mix["left.k.norm"]).reshape(B, T, G, -1), f)
            o = _attend(qn, kn, k.reshape(B, T, G, -1), left["scale"], _start(tokens), left["mask"]["size"]) * torch.sigmoid(x @ mix["left.g"].T)[..., None]
            branch = m["left_scale"] * (o.reshape(B, T, -1) @ mix["left.o"].T + mix["left.o.b"])
            silu = lambda z: z * torch.sigmoid(z)
            qr, kr, vr = (silu(x @ mix["right." + n].T).reshape(B, T, right["heads"], -1) for n in "qkv")
            decay = torch.tensor(right["decay"], dtype=torch.float64, device=DEVICE)[None, :, None, None]
            S, out = x.new_zeros(B, right["heads"], right["dim"], right["vdim"]), []
            for t in range(T):
                S = decay * S + kr[:, t][..., None] * vr[:, t][..., None, :]
                out.append((S * qr[:, t][..., None]).sum(2))
            o = _rms(torch.stack(out, dim=1).reshape(B, T, -1), eps) * mix["right.norm"] * torch.sigmoid(x @ mix["right.g"].T)
            branch = branch + m["right_scale"] * (o @ mix["right.o"].T)
        x = x + _rms(branch, eps) * w[p + "norm1"]
        x = x + _rms(_gated(x, _under(w, p + "mlp.")), eps) * w[p + "norm2"]
    return _rms(x, eps) * w["final.norm"]


def _exact_goletar(raw, w, tokens):
    eps, pairs = raw["norm"]["eps"], raw["embedding"]["bigram"]
    B, T = tokens.shape
    row = torch.full_like(tokens, pairs["buckets"])
    row[:, 1:] = (tokens[:, :-1] * pairs["mul_prev"] + tokens[:, 1:] * pairs["mul_cur"]) % pairs["buckets"]
    x = w["embed"][tokens] + w["bigram"][row]
    for index, layer in enumerate(raw["layers"]):
        m, mix, p = layer["mixer"], _under(w, f"l{index}.mix."), f"l{index}."
        h = _rms(x, eps) * w[p + "norm1"]
        if layer["type"] == "latent_attention":
            o, _ = _latent(h, tokens, mix, m, eps, _frequencies(m["rot"]["dims"], m["rot"]["base"]), 1.0, False, None)
            mixed = (o * torch.sigmoid(h @ mix["g"].T)[..., None]).reshape(B, T, -1)
        else:
            z, u = torch.sigmoid(h @ mix["z"].T + mix["z.b"]), h @ mix["x"].T + mix["x.b"]
            candidate = torch.where(u >= 0, u + 0.5, torch.sigmoid(u))
            state, out = torch.zeros_like(z[:, 0]), []
            for t in range(T):
                state = (1.0 - z[:, t]) * state + z[:, t] * candidate[:, t]
                out.append(state)
            g = h @ mix["g"].T
            mixed = torch.stack(out, dim=1) * g * torch.sigmoid(g)
        x = x + _rms(mixed @ mix["o"].T, eps) * w[p + "norm1b"]
        h, mlp = _rms(x, eps) * w[p + "norm2"], layer["mlp"]
        scores = torch.sigmoid(h @ w[p + "mlp.router"].T)
        best, which = scores.topk(mlp["router"]["top"], dim=2)
        weights, limit, out = torch.zeros_like(scores).scatter(2, which, best), mlp["expert"]["limit"], torch.zeros_like(h)
        for e in range(mlp["router"]["experts"]):
            at = (weights[..., e] > 0).nonzero(as_tuple=True)
            one, rows = _under(w, f"{p}mlp.e{e}."), h[at] * weights[..., e][at][:, None]
            g = (rows @ one["gate"].T).clamp(max=limit)
            out[at] += (g * torch.sigmoid(1.702 * g) * ((rows @ one["up"].T).clamp(-limit, limit) + 1.0)) @ one["down"].T
        x = x + _rms(out, eps) * w[p + "norm2b"]
    return _rms(x, eps) * w["final.norm"]
