"""What a user of this engine has it do, as cases that can be timed and checked.

A case is one step of the engine (``LLM.core.run``, the call that serving, trace replay and scoring go through) on a
bound model: ``running`` requests that decode one more token against about ``context`` cached tokens each, beside
``prompts`` fresh prompts of ``tokens`` tokens in all.  Either may be 0.  The step returns float logits: one row per
decoding request, then the row behind each prompt's last token.

Models (random weights; layer sizes of this repository's benchmark):

* ``qwen3_8b``: the headline configuration, all 36 layers;
* ``qwen3_2k``: 8 dense layers of width 2,048, the small model, also in float32;
* ``lomozen_2k``: lightning and latent attention, routed experts, 8 layers of width 2,048;
* ``kuditar_2k``: attention variants beside the gated delta rule and gated linear attention, routed experts, 8 layers.

Weights are drawn as initialised networks have them (1 / sqrt(inputs), sublayer outputs scaled down with the depth, the
scores of attention spread enough that some keys matter); routers and embeddings agree on which experts a token prefers,
as trained ones do, so that the choice of experts does not hang on the last bit.
"""
from __future__ import annotations

import math
import zlib

import numpy as np
import torch

_QWEN3 = dict(architectures=["Qwen3ForCausalLM"], head_dim=128, rope_theta=1000000.0, rms_norm_eps=1e-6,
              tie_word_embeddings=False, max_position_embeddings=40960)


def _lomozen():
    heads = 16
    latent = {"type": "latent_attention", "mixer": {
        "heads": heads, "dim": 64, "rot_dim": 32, "vdim": 64, "kv_rank": 224, "q_rank": 768, "scale": 96 ** -0.5, "mask": {"size": 1024},
        "rot": {"base": 500000.0, "dims": 32, "scaling": {"factor": 4.0, "original": 4096, "fast": 32.0, "slow": 1.0}}}}
    lightning = {"type": "lightning", "mixer": {"heads": heads, "dim": 128, "vdim": 128,
                                                "decay": [1.0 - 2.0 ** (-5 - 3 * h / heads) for h in range(heads)]}}
    mlp = {"kind": "moe", "router": {"experts": 32, "top": 4}, "expert": {"ff": 512}, "shared": {"ff": 1024}}
    return {"architecture": "Lomozen", "vocab": 32000, "width": 2048, "norm": {"eps": 1e-5},
            "layers": [dict(latent if i % 4 else lightning, mlp=mlp) for i in range(8)]}


def _kuditar():
    own = {"heads": 16, "kv_heads": 4, "dim": 128, "vdim": 128, "scale": 128 ** -0.5}
    att = {"type": "attention", "mixer": dict(own, rot={"base": 1e6, "dims": 64, "scaling": {"factor": 4.0}}, softcap=50.0, v_mix=True)}
    par = {"type": "parallel", "mixer": {
        "left": dict(own, rot={"base": 1e4, "dims": 128}, softcap=50.0, mask={"size": 1024, "keep_first": 16}),
        "right": {"heads": 16, "kv_heads": 16, "dim": 128, "vdim": 128, "conv": 4}}}
    par2 = {"type": "parallel_2", "mixer": {"left": dict(own, mask={"size": 2048}),
                                            "right": {"heads": 16, "dim": 128, "vdim": 128, "tau": 16.0, "decay_rank": 16}}}
    order = (att, par, par2, par)
    dense = {"kind": "dense", "ff": 3072, "limit": 7.0}
    moe = {"kind": "moe", "router": {"experts": 32, "top": 4, "scale": 2.0}, "expert": {"ff": 768, "limit": 7.0}}
    return {"architecture": "Kuditar", "vocab": 32000, "width": 2048, "norm": {"eps": 1e-5}, "embedding": {"scale": 2.0},
            "layers": [dict(order[i % 4], mlp=moe if i % 4 else dense) for i in range(8)]}


_CONFIGS = {
    "qwen3_8b": dict(_QWEN3, num_hidden_layers=36, hidden_size=4096, num_attention_heads=32, num_key_value_heads=8,
                     intermediate_size=12288, vocab_size=151936),
    "qwen3_2k": dict(_QWEN3, num_hidden_layers=8, hidden_size=2048, num_attention_heads=16, num_key_value_heads=4,
                     intermediate_size=3072, vocab_size=32000),
    "lomozen_2k": _lomozen(),
    "kuditar_2k": _kuditar(),
}
_PAGE = 16
_HEADROOM = 768       # decode passes on one state before its requests end and begin again


def _vocab(cfg):
    return cfg.get("vocab") or cfg["vocab_size"]


# --------------------------------------------------------------------------- the cases
def _case(name, model, running=0, context=0, prompts=0, tokens=0, ragged=False, dtype="bf16"):
    return {"name": name, "model": model, "dtype": dtype, "running": running, "context": context, "ragged": ragged,
            "prompts": prompts, "tokens": tokens}


def listed():
    return [
        # one user's chat: latency of a token
        _case("decode_1", "qwen3_8b", running=1, context=1024),
        # the headline: eight users behind prompts of 1,024 tokens
        _case("decode_8", "qwen3_8b", running=8, context=1024),
        # a busy server: users at all stages of their answers
        _case("decode_64_ragged", "qwen3_8b", running=64, context=1024, ragged=True),
        # questions about long documents, near the benchmark's longest context
        _case("decode_8_long", "qwen3_8b", running=8, context=7900),
        # the first token behind a prompt of the benchmark's length
        _case("prefill_2048", "qwen3_8b", prompts=1, tokens=2048),
        # the first token behind a short question
        _case("prefill_short", "qwen3_8b", prompts=1, tokens=37),
        # continuous batching: portions of new prompts ride with running decodes
        _case("mixed", "qwen3_8b", running=24, context=900, ragged=True, prompts=3, tokens=1501),
        # the small model decoding for one user: the smallest call
        _case("small_decode_1", "qwen3_2k", running=1, context=300),
        # the 32-bit path (parity runs, trace replay): prompts of uneven lengths, and decoding
        _case("fp32_prefill", "qwen3_2k", prompts=3, tokens=1003, ragged=True, dtype="fp32"),
        _case("fp32_decode", "qwen3_2k", running=5, context=410, ragged=True, dtype="fp32"),
        # the other designs: a prompt of one, a batch of users of another
        _case("lomozen_prefill", "lomozen_2k", prompts=1, tokens=2048),
        _case("kuditar_decode_16", "kuditar_2k", running=16, context=1100, ragged=True),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    model = rng.choice(["qwen3_8b", "qwen3_8b", "qwen3_8b", "qwen3_2k", "qwen3_2k", "lomozen_2k", "kuditar_2k"])
    dtype = rng.choice(["bf16", "fp32"]) if model == "qwen3_2k" else "bf16"
    kind = rng.choice(["decode", "prefill", "mixed"])
    c = _case("", model, ragged=rng.random() < 0.7, dtype=dtype)
    del c["name"]
    small = dtype == "fp32"
    if kind != "prefill":
        c["running"] = _log_int(rng, 1, 16 if small else 64) if kind == "decode" else rng.randint(2, 8 if small else 24)
        c["context"] = _log_int(rng, 64, min(1024 if small else 7900, 65536 // c["running"]) if kind == "decode" else 1000)
    if kind != "decode":
        c["tokens"] = _log_int(rng, 16, 1003 if small else 2048 if kind == "prefill" else 1501)
        c["prompts"] = rng.randint(1, max(1, min(5, c["tokens"] // 12)))
    return c


def _contexts(case):
    """Cached tokens of each running request: all alike, or spread over half to one and a half of it."""
    n = case["running"]
    if not case["ragged"]:
        return [case["context"]] * n
    return [max(1, int(case["context"] * (0.5 + (i + 1) * 0.6180339887 % 1.0))) for i in range(n)]


def _prompt_lengths(case):
    n, total = case["prompts"], case["tokens"]
    if not n:
        return []
    share = [1.0 + 3.0 * ((i + 1) * 0.6180339887 % 1.0) if case["ragged"] else 1.0 for i in range(n)]
    out = [max(1, int(total * s / sum(share))) for s in share]
    out[0] += total - sum(out)
    return out


# --------------------------------------------------------------------------- weights
_OUT = ("o_proj.weight", "down_proj.weight", ".o", ".down")              # matrices whose product joins the stream
_SHARP = ("q_norm.weight", "k_norm.weight", "q.norm", "k.norm")          # head norms: they set the spread of the scores


def _generator(name, device):
    return torch.Generator(device=device).manual_seed(zlib.crc32(name.encode()) + 17)


def _experts(cfg):
    return next((x["mlp"]["router"] for x in cfg.get("layers", ()) if (x.get("mlp") or {}).get("kind") == "moe"), None)


def _skills(cfg, device):
    """One direction of the stream per expert that routers and embeddings share."""
    return torch.randn((_experts(cfg)["experts"], cfg["width"]), generator=_generator("skills", device), device=device)


def _draw_weight(name, shape, cfg, device):
    """One tensor of a model by its checkpoint name, in float32 (bfloat16 values), the same at every call."""
    g = _generator(name, device)
    layers = len(cfg["layers"]) if "layers" in cfg else cfg["num_hidden_layers"]
    x = torch.randn(shape, generator=g, device=device)
    if name in ("model.embed_tokens.weight", "embed"):
        if _experts(cfg):
            pref = torch.rand((shape[0], _experts(cfg)["experts"]), generator=g, device=device).topk(_experts(cfg)["top"], -1).indices
            x += 0.5 * _skills(cfg, device)[pref].sum(1)
        if cfg.get("architecture") == "Kuditar":
            x *= 0.5                                                        # the configuration doubles it
    elif name.endswith(".router"):
        order = torch.randperm(shape[0], generator=g, device=device)
        x = 8.0 / shape[1] * _skills(cfg, device)[order]
    elif name.endswith(".conv"):
        x = 0.3 * x
        x[:, -1] += 1.0
    elif name.endswith("A_log"):
        x -= 3.0
    elif name.endswith("a2.b"):
        x += 2.0
    elif name.endswith("vmix"):
        x = torch.rand(shape, generator=g, device=device)
    elif name.endswith((".b", "dt_bias", "sink", "correction")) and x.dim() == 1:
        x *= 0.02
    elif name.endswith(_SHARP):
        x = 1.5 * (1.0 + 0.02 * x)
    elif name.endswith((".norm1b", ".norm2b", "left.out", "right.out")):   # norms of sublayer outputs
        x = (1.0 + 0.02 * x) / math.sqrt(2 * layers)
    elif x.dim() == 1:
        x = 1.0 + 0.02 * x
    else:
        x *= 1.0 / math.sqrt(shape[-1])
        if name.endswith(_OUT):
            x *= 1.0 / math.sqrt(2 * layers)
    return x.to(torch.bfloat16).float()


_MODELS: dict = {}


def _model(case):
    """The bound model of a case: a program binds it once and keeps it."""
    from jax_vllm_amd.config.registry import resolve
    from jax_vllm_amd.parts.model import DecoderModel

    key = (case["model"], case["dtype"])
    if key not in _MODELS:
        cfg = _CONFIGS[case["model"]]
        arch, typed, _ = resolve(cfg)
        model = DecoderModel(arch.build_spec(typed))
        compute = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
        tensors = {name: _draw_weight(name, tuple(t.shape), cfg, "cuda").to(compute if t.role == "matrix" else torch.float32)
                   for name, t in model.tensor_specs().items()}
        model.bind(tensors, compute)
        _MODELS[key] = model
    return _MODELS[key]


# --------------------------------------------------------------------------- one case
def _tokens(case, seed):
    """(cached tokens of each running request, its next tokens, the prompts), all token ids on the host."""
    rng = np.random.default_rng([seed, case["running"], case["context"], case["tokens"]])
    vocab = _vocab(_CONFIGS[case["model"]])
    cached = [rng.integers(0, vocab, size=n).tolist() for n in _contexts(case)]
    coming = [rng.integers(0, vocab, size=_HEADROOM).tolist() for _ in cached]
    prompts = [rng.integers(0, vocab, size=n).tolist() for n in _prompt_lengths(case)]
    return cached, coming, prompts


def _begin(state):
    """Start the running requests: their cached tokens go through the engine in portions."""
    from jax_vllm_amd.engine.entries import StepEntry

    core, batch, room = state["core"], [], 4096
    for i, tokens in enumerate(state["cached"]):
        core.start_request(i)
        at = 0
        while at < len(tokens):
            n = min(room, len(tokens) - at)
            batch.append(StepEntry(i, tokens[at:at + n], []))
            at, room = at + n, room - n
            if room == 0:
                core.run(batch)
                batch, room = [], 4096
    if batch:
        core.run(batch)
    state["step"] = 0


def prepare(case, seed):
    from jax_vllm_amd import LLM

    cached, coming, prompts = _tokens(case, seed)
    lengths = [len(t) + _HEADROOM for t in cached] + [len(t) for t in prompts]
    pages = sum(-(-n // _PAGE) for n in lengths)
    llm = LLM(_model(case), dtype=case["dtype"], block_size=_PAGE, num_blocks=1 + pages, max_num_seqs=len(lengths),
              max_model_len=max(lengths), max_num_batched_tokens=4096, enable_prefix_cache=False)
    state = {"llm": llm, "core": llm.core, "cached": cached, "coming": coming, "prompts": prompts, "step": 0}
    if cached:
        _begin(state)
        if not prompts:
            run(state)      # a server has recorded its decode steps before users come
    return state


def run(state):
    from jax_vllm_amd.engine.entries import StepEntry

    core, at = state["core"], state["step"]
    running = range(len(state["cached"]))
    if running and at == _HEADROOM:
        for i in running:
            core.finish_request(i)
        _begin(state)
        at = 0
    entries = [StepEntry(i, [state["coming"][i][at]], [0]) for i in running]
    for k, prompt in enumerate(state["prompts"]):
        core.start_request(("prompt", k))
        entries.append(StepEntry(("prompt", k), prompt, [len(prompt) - 1]))
    logits = core.run(entries, borrow=True)
    for k in range(len(state["prompts"])):
        core.finish_request(("prompt", k))
    state["step"] = at + 1
    return logits


def _layer_sizes(cfg, tokens):
    """(weights that a step of so many tokens reads, weights that one token meets) in all layers, the head apart."""
    if "hidden_size" in cfg:
        h, d = cfg["hidden_size"], cfg["head_dim"]
        one = (2 * cfg["num_attention_heads"] + 2 * cfg["num_key_value_heads"]) * d * h + 3 * cfg["intermediate_size"] * h
        return one * cfg["num_hidden_layers"], one * cfg["num_hidden_layers"]
    w, read, met = cfg["width"], 0, 0
    for layer in cfg["layers"]:
        m, f = layer["mixer"], layer["mlp"]
        if layer["type"] == "lightning":
            mix = 5 * w * m["heads"] * m["dim"]
        elif layer["type"] == "latent_attention":
            mix = w * (m["q_rank"] + m["kv_rank"] + m["rot_dim"] + 2 * m["heads"] * m["vdim"]) + m["heads"] * (
                m["q_rank"] * (m["dim"] + m["rot_dim"]) + m["kv_rank"] * (m["dim"] + m["vdim"]))
        else:
            a = m.get("left", m)
            mix = w * a["dim"] * (2 * a["heads"] + 2 * a["kv_heads"]) + (w * a["heads"] * a["dim"] if layer["type"] == "attention" else 0)
            if "right" in m:
                mix += 5 * w * m["right"]["heads"] * m["right"]["dim"]
        read, met = read + mix, met + mix
        if f["kind"] == "dense":
            read, met = read + 3 * w * f["ff"], met + 3 * w * f["ff"]
        else:
            e, top, one, shared = f["router"]["experts"], f["router"]["top"], 3 * w * f["expert"]["ff"], 3 * w * (f.get("shared") or {"ff": 0})["ff"]
            touched = e * (1.0 - (1.0 - top / e) ** tokens)
            read, met = read + touched * one + shared, met + top * one + shared
    return read, met


def work(case):
    cfg, item = _CONFIGS[case["model"]], 2 if case["dtype"] == "bf16" else 4
    steps = [(n + 1, 1) for n in _contexts(case)] + [(n, n) for n in _prompt_lengths(case)]     # (context behind it, tokens)
    tokens, rows = sum(n for _, n in steps), len(steps)
    width = cfg.get("width") or cfg["hidden_size"]
    read, met = _layer_sizes(cfg, tokens)
    head = _vocab(cfg) * width
    nbytes, flops = (read + head + tokens * width) * item + 4.0 * rows * _vocab(cfg), 2.0 * met * tokens + 2.0 * head * rows
    layers = cfg.get("layers") or [{"type": "attention", "mixer": {
        "heads": cfg["num_attention_heads"], "kv_heads": cfg["num_key_value_heads"], "dim": 128, "vdim": 128}}] * cfg["num_hidden_layers"]
    for layer in layers:
        m = layer["mixer"].get("left", layer["mixer"])
        state = layer["mixer"].get("right") or (m if layer["type"] == "lightning" else None)
        for total, n in steps:
            if layer["type"] != "lightning":
                size = (m.get("mask") or {}).get("size") or total
                pairs = sum(min(size, p) for p in range(total - n + 1, total + 1))
                cached = m["kv_rank"] + m["rot_dim"] if "kv_rank" in m else m["kv_heads"] * (m["dim"] + m["vdim"])
                q, v = m["dim"] + m.get("rot_dim", 0), m["vdim"]
                nbytes += (min(total - n, size) + n) * cached * item        # keys and values read, the step's own written
                flops += 2.0 * pairs * m["heads"] * (q + v)
            if state:
                s = state["heads"] * state["dim"] * state["vdim"]
                nbytes += 2.0 * 4 * s
                flops += 6.0 * s * n
    return {"bytes": float(nbytes), "flops": float(flops)}


def tolerance(case):
    # about four times the error against 64 bits that was measured over listed and drawn cases: 1.4e-6..1.7e-6 in float32
    # (8 layers), 1.3e-3..3.4e-3 in bfloat16 (8 and 36 layers); single logits lie up to 6 deviations off
    if case["dtype"] == "fp32":
        return {"rel": 8e-6, "max": 8e-5}
    return {"rel": 1.2e-2, "max": 0.1}


# --------------------------------------------------------------------------- the same in 64 bits
class _Weights:
    """A model's tensors by name in float64, drawn when they are asked for."""

    def __init__(self, cfg):
        self.cfg = cfg

    def __call__(self, name, *shape):
        return _draw_weight(name, shape, self.cfg, "cuda").double()


def _by_rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(z):
    return z * torch.sigmoid(z)


def _turn(x, freqs, amp=1.0):
    """x [heads, n, size]: elements i and i + len(freqs) turn by position; angles in 32 bits, as the models define them."""
    k = freqs.numel()
    ang = (torch.arange(x.shape[1], device="cuda", dtype=torch.float32)[:, None] * freqs.float()[None, :]).double()
    cos, sin = torch.cos(ang) * amp, torch.sin(ang) * amp
    u, v = x[..., :k], x[..., k:2 * k]
    return torch.cat([u * cos - v * sin, v * cos + u * sin, x[..., 2 * k:]], -1)


def _freqs(base, dims):
    return base ** (-2.0 * torch.arange(dims // 2, dtype=torch.float64, device="cuda") / dims)


def _attend(q, k, v, scale, seen=None, cap=None, sink=None):
    """q [H, n, d] over k, v [G, n, .] with a causal mask and what ``seen`` leaves; [n, H * dv]."""
    h, n, per = q.shape[0], q.shape[1], q.shape[0] // k.shape[0]
    i, j = torch.arange(n, device="cuda")[:, None], torch.arange(n, device="cuda")[None, :]
    mask = (j <= i) if seen is None else (j <= i) & seen(i, j)
    out = []
    for a in range(h):                                  # a head at a time: the scores of long prompts are large
        s = q[a] @ k[a // per].T * scale
        if cap:
            s = cap * torch.tanh(s / cap)
        s = s.masked_fill(~mask, float("-inf"))
        if sink is not None:
            s = torch.cat([s, sink[a].expand(n, 1)], -1)
        out.append(torch.softmax(s, -1)[:, :n] @ v[a // per])
    return torch.stack(out, 1).reshape(n, -1)


def _heads(y, n):
    return y.view(y.shape[0], n, -1).transpose(0, 1)


def _qwen3_layers(w, cfg, xs):
    h, d, nq, nkv, eps, f = (cfg[k] for k in ("hidden_size", "head_dim", "num_attention_heads", "num_key_value_heads", "rms_norm_eps",
                                              "intermediate_size"))
    freqs = 1.0 / (cfg["rope_theta"] ** (torch.arange(0, d, 2, dtype=torch.float32, device="cuda") / d))
    for i in range(cfg["num_hidden_layers"]):
        p = f"model.layers.{i}."
        wq, wk, wv, wo = (w(f"{p}self_attn.{s}_proj.weight", *shape) for s, shape in (
            ("q", (nq * d, h)), ("k", (nkv * d, h)), ("v", (nkv * d, h)), ("o", (h, nq * d))))
        gate, up, down = (w(f"{p}mlp.{s}_proj.weight", *shape) for s, shape in (("gate", (f, h)), ("up", (f, h)), ("down", (h, f))))
        n1, n2 = w(p + "input_layernorm.weight", h), w(p + "post_attention_layernorm.weight", h)
        qn, kn = w(p + "self_attn.q_norm.weight", d), w(p + "self_attn.k_norm.weight", d)
        for x in xs:
            u = _by_rms(x, eps) * n1
            q, k = _by_rms(_heads(u @ wq.T, nq), eps) * qn, _by_rms(_heads(u @ wk.T, nkv), eps) * kn
            x += _attend(_turn(q, freqs), _turn(k, freqs), _heads(u @ wv.T, nkv), d ** -0.5) @ wo.T
            u = _by_rms(x, eps) * n2
            x += (_silu(u @ gate.T) * (u @ up.T)) @ down.T


def _routed(w, p, f, u, width, correction, on_input, act):
    """Routed experts on rows u; ``act(gate, up)``; the score multiplies the expert's input or its output."""
    r, ff, shared = f["router"], f["expert"]["ff"], f.get("shared")
    s = torch.sigmoid(u @ w(p + "router", r["experts"], width).T)
    chosen = (s + w(p + "correction", r["experts"]) if correction else s).topk(r["top"], -1).indices
    out = torch.zeros_like(u)

    def expert(q, x, size):
        return act(x @ w(q + "gate", size, width).T, x @ w(q + "up", size, width).T) @ w(q + "down", width, size).T

    for e in range(r["experts"]):
        rows, _ = (chosen == e).nonzero(as_tuple=True)
        if rows.numel():
            g = s[rows, e, None] * float(r.get("scale", 1.0))
            out[rows] += expert(f"{p}e{e}.", g * u[rows], ff) if on_input else g * expert(f"{p}e{e}.", u[rows], ff)
    return out + expert(p + "shared.", u, shared["ff"]) if shared else out


def _latent(w, p, m, u, width, eps):
    n, nh, d, r, dv, kr, qr = u.shape[0], *(m[k] for k in ("heads", "dim", "rot_dim", "vdim", "kv_rank", "q_rank"))
    dims, base, sc = m["rot"]["dims"], m["rot"]["base"], m["rot"]["scaling"]
    f = _freqs(base, dims)
    lo, hi = (dims * math.log(sc["original"] / (2 * math.pi * t)) / (2 * math.log(base)) for t in (sc["fast"], sc["slow"]))
    lo, hi = max(math.floor(lo), 0), min(math.ceil(hi), dims - 1)
    ramp = ((torch.arange(dims // 2, dtype=torch.float64, device="cuda") - lo) / max(hi - lo, 0.001)).clamp(0, 1)
    f, amp = f / sc["factor"] * ramp + f * (1 - ramp), 0.1 * math.log(sc["factor"]) + 1.0
    q = _heads(_by_rms(u @ w(p + "dq", qr, width).T, eps) * w(p + "dq.norm", qr) @ w(p + "uq", nh * (d + r), qr).T, nh)
    c = u @ w(p + "dkv", kr + r, width).T
    key = _turn(c[None, :, kr:], f, amp)
    c = _by_rms(c[:, :kr], eps) * w(p + "dkv.norm", kr)
    k, v = _heads(c @ w(p + "uk", nh * d, kr).T, nh), _heads(c @ w(p + "uv", nh * dv, kr).T, nh)
    q, k = torch.cat([q[..., :d], _turn(q[..., d:], f, amp)], -1), torch.cat([k, key.expand(nh, n, r)], -1)
    o = _attend(q, k, v, m["scale"], lambda i, j: i - j < m["mask"]["size"])
    return o * torch.sigmoid(u @ w(p + "g", nh * dv, width).T) @ w(p + "o", width, nh * dv).T


def _lightning(w, p, m, u, width, eps):
    n, nh, d, dv = u.shape[0], m["heads"], m["dim"], m["vdim"]
    q, k, v = (_heads(_silu(u @ w(p + s, nh * e, width).T), nh) for s, e in (("q", d), ("k", d), ("v", dv)))
    back = torch.arange(n, device="cuda")[:, None] - torch.arange(n, device="cuda")[None, :]
    o = []
    for a in range(nh):
        fade = torch.where(back >= 0, float(m["decay"][a]) ** back.clamp(min=0).double(), 0.0)
        o.append((q[a] @ k[a].T * fade) @ v[a])
    o = _by_rms(torch.stack(o, 1).reshape(n, nh * dv), eps) * w(p + "norm", nh * dv)
    return o * torch.sigmoid(u @ w(p + "g", nh * dv, width).T) @ w(p + "o", width, nh * dv).T


def _lomozen_layers(w, cfg, xs):
    width, eps = cfg["width"], cfg["norm"]["eps"]
    for i, layer in enumerate(cfg["layers"]):
        p, mixer = f"l{i}.", _latent if layer["type"] == "latent_attention" else _lightning
        for x in xs:
            a = mixer(w, p + "mix.", layer["mixer"], _by_rms(x, eps) * w(p + "norm1", width), width, eps)
            x += _by_rms(a, eps) * w(p + "norm1b", width)
            f = _routed(w, p + "mlp.", layer["mlp"], _by_rms(x, eps) * w(p + "norm2", width), width, False, True,
                        lambda g, v: _silu(g) * v)
            x += _by_rms(f, eps) * w(p + "norm2b", width)


def _layer_norm(x, a, b, eps):
    y = x - x.mean(-1, keepdim=True)
    return _by_rms(y, eps) * a + b


def _kuditar_attention(w, p, m, u, width, eps, kind, shared):
    nh, g, d = m["heads"], m["kv_heads"], m["dim"]
    q, k, v = (u @ w(p + s, c * d, width).T for s, c in (("q", nh), ("k", g), ("v", g)))
    if kind != "attention":
        q, k, v = (y + w(p + s + ".b", y.shape[1]) for s, y in (("q", q), ("k", k), ("v", v)))
    q, k, v = _heads(q, nh), _heads(k, g), _heads(v, g)
    if kind != "attention":
        q, k = _by_rms(q, eps) * w(p + "q.norm", d), _by_rms(k, eps) * w(p + "k.norm", d)
    if m.get("rot"):
        f = _freqs(m["rot"]["base"], m["rot"]["dims"]) / float((m["rot"].get("scaling") or {"factor": 1.0})["factor"])
        q, k = _turn(q, f), _turn(k, f)
    if kind == "attention":
        q, k = _by_rms(q, eps), _by_rms(k, eps)
        if shared:
            lam = w(p + "vmix").reshape(())
            v = (1 - lam) * v + lam * shared[0]
        else:
            shared.append(v)
        o = _attend(q, k, v, m["scale"], None, m["softcap"]) * torch.sigmoid(u @ w(p + "g", nh * d, width).T)
    elif kind == "parallel":
        size, keep = m["mask"]["size"], m["mask"]["keep_first"]
        o = _attend(q, k, v, m["scale"], lambda i, j: (i - j < size) | (j < keep), m["softcap"], w(p + "sink", nh))
    else:
        size = m["mask"]["size"]
        o = _attend(q, k, v, m["scale"], lambda i, j: i // size == j // size)
    return o @ w(p + "o", width, nh * d).T


def _delta(w, p, m, u, width, eps):
    n, nh, d = u.shape[0], m["heads"], m["dim"]

    def conv(s):
        y, taps = u @ w(p + s, nh * d, width).T, w(p + s + ".conv", nh * d, m["conv"])
        y = torch.cat([y.new_zeros(m["conv"] - 1, nh * d), y])
        return _silu(sum(y[j:j + n] * taps[:, j] for j in range(m["conv"]))).view(n, nh, d)

    q, k, v = (conv(s) for s in "qkv")
    q, k = (y / torch.sqrt((y * y).sum(-1, keepdim=True) + 1e-6) for y in (q, k))
    beta = torch.sigmoid(u @ w(p + "b", nh, width).T)
    rate = torch.nn.functional.softplus(u @ w(p + "a", nh, width).T + w(p + "dt_bias", nh), threshold=1e9)
    fade, q = torch.exp(-torch.exp(w(p + "A_log", nh)) * rate), q * d ** -0.5
    s, o = u.new_zeros(nh, d, d), []
    for t in range(n):
        s = s * fade[t][:, None, None]
        s = s + k[t][:, :, None] * (beta[t][:, None] * (v[t] - torch.bmm(k[t][:, None, :], s)[:, 0]))[:, None, :]
        o.append(torch.bmm(q[t][:, None, :], s)[:, 0])
    o = (_by_rms(torch.stack(o), eps) * w(p + "norm", d)).reshape(n, nh * d)
    return o * _silu(u @ w(p + "g", nh * d, width).T) @ w(p + "o", width, nh * d).T


def _gated_linear(w, p, m, u, width, eps):
    n, nh, d, r = u.shape[0], m["heads"], m["dim"], m["decay_rank"]
    q, k, v = ((u @ w(p + s, nh * d, width).T).view(n, nh, d) for s in "qkv")
    z = u @ w(p + "a1", r, width).T @ w(p + "a2", nh * d, r).T + w(p + "a2.b", nh * d)
    fade = (torch.sigmoid(z) ** (1.0 / m["tau"])).view(n, nh, d)
    s, o = u.new_zeros(nh, d, d), []
    for t in range(n):
        s = s * fade[t][:, :, None] + k[t][:, :, None] * v[t][:, None, :]
        o.append(torch.bmm(q[t][:, None, :] * d ** -0.5, s)[:, 0])
    o = (_by_rms(torch.stack(o), eps) * w(p + "norm", d)).reshape(n, nh * d)
    return o * _silu(u @ w(p + "g", nh * d, width).T) @ w(p + "o", width, nh * d).T


def _kuditar_layers(w, cfg, xs):
    width, eps, shared = cfg["width"], cfg["norm"]["eps"], [[] for _ in xs]
    for i, layer in enumerate(cfg["layers"]):
        p, m, f = f"l{i}.", layer["mixer"], layer["mlp"]
        limit = float(f.get("limit") or f["expert"]["limit"])

        def act(g, v, limit=limit):
            g = g.clamp(max=limit)
            return g * torch.sigmoid(1.702 * g) * (v.clamp(-limit, limit) + 1)

        for x, first in zip(xs, shared):
            u = _layer_norm(x, w(p + "norm1", width), w(p + "norm1.b", width), eps)
            if layer["type"] == "attention":
                x += _kuditar_attention(w, p + "mix.", m, u, width, eps, "attention", first)
            else:
                a = _kuditar_attention(w, p + "mix.left.", m["left"], u, width, eps, layer["type"], None)
                b = (_delta if layer["type"] == "parallel" else _gated_linear)(w, p + "mix.right.", m["right"], u, width, eps)
                x += (_by_rms(a, eps) * w(p + "mix.left.out", width) + _by_rms(b, eps) * w(p + "mix.right.out", width)) / 2
            u = _layer_norm(x, w(p + "norm2", width), w(p + "norm2.b", width), eps)
            if f["kind"] == "dense":
                g = act(u @ w(p + "mlp.gate", f["ff"], width).T, u @ w(p + "mlp.up", f["ff"], width).T)
                x += g @ w(p + "mlp.down", width, f["ff"]).T
            else:
                x += _routed(w, p + "mlp.", f, u, width, True, False, act)


@torch.no_grad()
def exact(case, seed):
    """The logits of the first pass, every sequence as a whole in float64; None where that takes too long."""
    cfg = _CONFIGS[case["model"]]
    cached, coming, prompts = _tokens(case, seed)
    warm = 2 if not prompts else 1                              # prepare() has already run one decode step
    rows = [t + c[:warm] for t, c in zip(cached, coming)] + prompts
    if sum(len(r) for r in rows) > (10000 if case["model"] == "qwen3_8b" else 20000):
        return None
    w = _Weights(cfg)
    if case["model"].startswith("qwen3"):
        v, h = cfg["vocab_size"], cfg["hidden_size"]
        embed = _draw_weight("model.embed_tokens.weight", (v, h), cfg, "cuda")
        xs = [embed[torch.tensor(r, device="cuda")].double() for r in rows]
        _qwen3_layers(w, cfg, xs)
        x = _by_rms(torch.stack([x[-1] for x in xs]), cfg["rms_norm_eps"]) * w("model.norm.weight", h)
        return x @ w("lm_head.weight", v, h).T
    v, h, eps = cfg["vocab"], cfg["width"], cfg["norm"]["eps"]
    embed = w("embed", v, h) * float((cfg.get("embedding") or {}).get("scale", 1.0))
    xs = [embed[torch.tensor(r, device="cuda")] for r in rows]
    if case["model"] == "lomozen_2k":
        _lomozen_layers(w, cfg, xs)
        return _by_rms(torch.stack([x[-1] for x in xs]), eps) * w("final.norm", h) @ w("head", v, h).T
    _kuditar_layers(w, cfg, xs)
    x = _layer_norm(torch.stack([x[-1] for x in xs]), w("final.norm", h), w("final.norm.b", h), eps)
    return x @ w("embed", v, h).T
