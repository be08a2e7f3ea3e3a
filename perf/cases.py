"""What the performance of this framework is measured on: calls a serving program makes through the model classes, from one token of one
conversation to a full batch of prompts, over the decoders, precisions and cache forms the framework offers.

A case is a dict of plain values:
  model     one of MODELS
  call      "score":   one step_score over whole prompts, the logits of each one's last token back on the host (prefill; the program samples)
            "extend":  step_score over one more token of cached sequences, logits back (decode; the program samples)
            "greedy":  `steps` decode steps over cached sequences, every step's greedy ids and the last one's logits back
            "request": prompts and then `steps` decode steps, as "score" with greedy ids followed by "greedy"
  batch, shortest, longest   sequences and their range of lengths; lengths are spread evenly over it and odd ones among them
  steps     decode steps
The tokens of decode steps are given (not the sampled ones), so that every implementation sees the same inputs whatever its rounding.
"""
import math

import numpy as np
import torch

import nano_vllm_candle_amd as pkg
from nano_vllm_candle_amd.gopunex import BiasAttentionConfig, ChannelDeltaConfig, LightningConfig
from nano_vllm_candle_amd.tafopel import GeluMlpConfig, LatentMixerConfig, ScanMixerConfig, Yarn

CHUNK = 4096  # rows of one forward pass (the scheduler's max_num_batched_tokens)
VOCAB = 32768  # of the decoders without a published vocabulary

# name -> (design, dtype, bits of a cached key / value element)
MODELS = {
    "qwen3-0.6b": ("qwen3", "bfloat16", 16),
    "qwen3-0.6b-kv24": ("qwen3", "bfloat16", 24),
    "qwen3-8b-4-layers": ("qwen3", "bfloat16", 16),
    "gopunex-2k": ("gopunex", "bfloat16", 16),
    "gopunex-1k-f32": ("gopunex", "float32", 32),
    "tafopel-1k": ("tafopel", "bfloat16", 16),
}


def listed():
    return [
        # one conversation: the next token, sampled by the program
        dict(name="one token", model="qwen3-0.6b", call="extend", batch=1, shortest=137, longest=137, steps=1),
        # time to first token of a short question, and of a document
        dict(name="short prompt", model="qwen3-0.6b", call="score", batch=1, shortest=117, longest=117, steps=0),
        dict(name="document", model="qwen3-0.6b", call="score", batch=1, shortest=2391, longest=2391, steps=0),
        # a small server: the headline benchmark's state, decode and prefill
        dict(name="64 decode", model="qwen3-0.6b", call="greedy", batch=64, shortest=64, longest=512, steps=16),
        dict(name="64 prompts", model="qwen3-0.6b", call="score", batch=64, shortest=64, longest=512, steps=0),
        # a busy one: more sequences than one decode chunk's fused path takes
        dict(name="200 decode", model="qwen3-0.6b", call="greedy", batch=200, shortest=64, longest=1024, steps=6),
        # a careful one: 24-bit keys and values
        dict(name="24-bit cache", model="qwen3-0.6b-kv24", call="request", batch=24, shortest=48, longest=400, steps=8),
        # layers of a big model: decode of a middling batch, and prompts
        dict(name="big decode", model="qwen3-8b-4-layers", call="greedy", batch=24, shortest=256, longest=2048, steps=8),
        dict(name="big prompts", model="qwen3-8b-4-layers", call="score", batch=3, shortest=700, longest=2000, steps=0),
        # the layered decoders: whole requests of a middling batch, and the 32-bit mode
        dict(name="gopunex", model="gopunex-2k", call="request", batch=24, shortest=64, longest=512, steps=8),
        dict(name="tafopel", model="tafopel-1k", call="request", batch=24, shortest=64, longest=512, steps=8),
        dict(name="gopunex 32-bit", model="gopunex-1k-f32", call="request", batch=16, shortest=24, longest=160, steps=12),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """one more case of these ranges"""
    kind = rng.choice(["extend", "prompt", "prompts", "decode", "decode", "kv24", "big decode", "big prompts", "gopunex", "tafopel", "f32"])
    if kind == "extend":
        n = _log_int(rng, 16, 2048)
        return dict(model="qwen3-0.6b", call="extend", batch=rng.randint(1, 8), shortest=n, longest=n + rng.randint(0, 100), steps=1)
    if kind == "prompt":
        n = _log_int(rng, 16, 3000)
        return dict(model="qwen3-0.6b", call="score", batch=1, shortest=n, longest=n, steps=0)
    if kind in ("prompts", "big prompts"):
        big = kind == "big prompts"
        lo = _log_int(rng, 48, 700 if big else 200)
        hi = lo + rng.randint(1, 600)
        most = (4000 if big else 16000) * 2 // (lo + hi)
        return dict(model="qwen3-8b-4-layers" if big else "qwen3-0.6b", call="score", batch=rng.randint(2, max(2, min(64, most))), shortest=lo, longest=hi, steps=0)
    if kind in ("decode", "big decode"):
        big = kind == "big decode"
        batch = _log_int(rng, 16, 48 if big else 200)
        lo = _log_int(rng, 32, 256)
        hi = min(lo + _log_int(rng, 16, 1500), 2 * 100000 // batch)
        return dict(model="qwen3-8b-4-layers" if big else "qwen3-0.6b", call="greedy", batch=batch, shortest=lo, longest=max(lo, hi), steps=max(6, min(12, 400 // batch)))
    lo = _log_int(rng, 16, 100)
    if kind == "f32":
        return dict(model="gopunex-1k-f32", call="request", batch=rng.randint(10, 16), shortest=lo, longest=lo + rng.randint(1, 60), steps=rng.randint(10, 12))
    model = {"kv24": "qwen3-0.6b-kv24", "gopunex": "gopunex-2k", "tafopel": "tafopel-1k"}[kind]
    return dict(model=model, call="request", batch=rng.randint(16, 24), shortest=lo, longest=lo + rng.randint(1, 300), steps=rng.randint(6, 8))


# ---- configurations -----------------------------------------------------------------------------------------------------------
def _config(name):
    if name.startswith("qwen3-0.6b"):
        return pkg.Qwen3Config.qwen3_0_6b()
    if name.startswith("qwen3-8b"):  # four of its layers
        c = pkg.Qwen3Config.qwen3_8b()
        c.num_hidden_layers = 4
        return c
    if name.startswith("gopunex"):  # one layer of each mixer
        w = 2048 if "2k" in name else 1024
        layers = [(BiasAttentionConfig(16, 8, 128, 128, 128 ** -0.5, 32, 512.0, True), 9 * w // 2), (ChannelDeltaConfig(16, 16, 128, 128, 4, 128, 128), 9 * w // 2),
                  (LightningConfig(16, 128, 128, tuple(math.exp(-(i + 1) / 32) for i in range(16))), 9 * w // 2)]
        return pkg.GopunexConfig(VOCAB, w, layers, 1e-6, 1.0, 0.5)
    attn = LatentMixerConfig(16, 64, 64, 128, 256, 512, 1e6, 128 ** -0.5, Yarn(8.0, 4096.0, 32.0, 1.0))
    scan = ScanMixerConfig(2048, 16, 4, 64)
    return pkg.TafopelConfig(VOCAB, 1024, [(m, GeluMlpConfig(3072)) for m in (scan, attn, scan, attn)], 1e-6)


def _lengths(case):
    n = np.linspace(case["shortest"], case["longest"], case["batch"]).astype(int)
    return [int(x) for x in np.random.default_rng(7).permutation(n)]


def _tokens(case, seed):
    rng = np.random.default_rng([seed, 1])
    vocab = _config(case["model"]).vocab_size
    return [rng.integers(0, vocab, n + case["steps"]).astype(np.uint32) for n in _lengths(case)]


# ---- weights ------------------------------------------------------------------------------------------------------------------
def _wrap(x):
    """a 64-bit pattern as a signed number"""
    return (x & (2 ** 64 - 1)) - (2 ** 64 if x & 2 ** 63 else 0)


def _shift(x, n):
    return (x >> n) & ((1 << (64 - n)) - 1)


def _mix(z):
    z = (z ^ _shift(z, 30)) * _wrap(0xBF58476D1CE4E5B9)
    z = (z ^ _shift(z, 27)) * _wrap(0x94D049BB133111EB)
    return z ^ _shift(z, 31)


def _synthetic(name, shape, seed, dev):
    """tensor of the deterministic checkpoint generator (nvllm_model_fill_synthetic), in 64 bits"""
    h = 0xCBF29CE484222325
    for c in name.encode():
        h = ((h ^ c) * 0x100000001B3) & (2 ** 64 - 1)
    h ^= (seed * 0x9E3779B97F4A7C15) & (2 ** 64 - 1)
    out = torch.empty(math.prod(shape), dtype=torch.float64, device=dev)
    for a in range(0, out.numel(), 1 << 26):
        i = torch.arange(a, min(out.numel(), a + (1 << 26)), device=dev)
        z = _mix((i + 1) * _wrap(0x9E3779B97F4A7C15) + _wrap(h))
        out[a:a + len(i)] = (_shift(z, 56) - 128).double() / 4096 if len(shape) == 2 else 1 + (_shift(z, 40) % 33 - 16).double() / 128
    return out.view(shape)


def _random(name, shape, rng, dev):
    """bf16 tensor of a layered decoder: unit-variance products, norms near their neutral value, decays from slow to fast"""
    def normal(mean, dev_):
        return mean + dev_ * torch.randn(shape, generator=rng, device=dev)

    def uniform(lo, hi):
        return lo + (hi - lo) * torch.rand(shape, generator=rng, device=dev)

    if name.endswith("A_log"):
        a = uniform(-3.0, 0.5) if len(shape) == 1 else uniform(-2.0, 2.5)
    elif name.endswith("dt.b"):
        a = uniform(-4.0, 0.5)
    elif name.endswith("dt_bias"):
        a = normal(-1.0, 0.2)
    elif name.endswith(("mix.D", "conv.b")):
        a = uniform(-0.5, 1.0)
    elif name.endswith("sink"):
        a = uniform(-1.0, 2.0)
    elif name.endswith("vmix"):
        a = uniform(0.2, 0.7)
    elif name == "embed" or name.endswith("rel"):
        a = normal(0.0, 1.0)
    elif len(shape) == 2:
        a = normal(0.0, shape[1] ** -0.5)
    else:
        a = normal(1.0 if name.endswith(("q.norm", "k.norm", "mix.norm", "dq.norm", "dkv.norm")) else 0.0, 0.2)
    return a.bfloat16()


def _state_dict(cfg, seed, dev):
    rng = torch.Generator(dev).manual_seed(seed)
    w = {n: _random(n, s, rng, dev) for n, s in cfg.tensor_shapes().items()}
    if isinstance(cfg, pkg.TafopelConfig):  # its layer norms' weights are stored whole
        w = {n: a + 1 if n == "final.norm" or n.endswith("norm1") else a for n, a in w.items()}
    return w


# ---- one pass -----------------------------------------------------------------------------------------------------------------
def prepare(case, seed):
    design, dtype, kv_bits = MODELS[case["model"]]
    cfg = _config(case["model"])
    if design == "qwen3":
        model = pkg.Qwen3ForCausalLM.from_synthetic(cfg, seed)
        if kv_bits == 24:
            model.set_option("kv_v_bits", 24)
            model.set_option("kv_k_bits", 24)
    else:
        cls = {"gopunex": pkg.GopunexForCausalLM, "tafopel": pkg.TafopelForCausalLM}[design]
        weights = {n: a.view(torch.int16).cpu().numpy().view(np.uint16) for n, a in _state_dict(cfg, seed, "cuda").items()}
        model = cls.from_state_dict(cfg, weights, dtype=dtype)
    lengths, tokens = _lengths(case), _tokens(case, seed)
    model.kv_alloc(sum(-(-len(t) // 256) for t in tokens), case["batch"], CHUNK)
    ids = list(range(case["batch"]))
    prompts = [t[:n] for t, n in zip(tokens, lengths)]
    grown = [[t[:n + k] for t, n in zip(tokens, lengths)] for k in range(1, case["steps"] + 1)]
    last = [[len(t) - 1] for t in (grown[0] if case["call"] == "extend" else prompts)]
    if case["call"] in ("extend", "greedy"):
        model.step(ids, prompts, True)
    return dict(model=model, call=case["call"], ids=ids, prompts=prompts, grown=grown, last=last)


def run(state):
    m, ids = state["model"], state["ids"]
    if state["call"] == "score":
        return {"logits": m.step_score(ids, state["prompts"], True, state["last"])}
    if state["call"] == "extend":
        return {"logits": m.step_score(ids, state["grown"][0], False, state["last"])}
    tokens = [m.step(ids, state["prompts"], True)[0]] if state["call"] == "request" else []
    for k, sequences in enumerate(state["grown"], 1):
        out, logits = m.step(ids, sequences, False, want_logits=k == len(state["grown"]))
        tokens.append(out)
    return {"tokens": np.stack(tokens), "logits": logits}


# ---- what a pass cannot do without --------------------------------------------------------------------------------------------
def work(case):
    design, dtype, kv_bits = MODELS[case["model"]]
    cfg = _config(case["model"])
    shapes = cfg.hf_tensor_shapes() if design == "qwen3" else cfg.tensor_shapes()
    head = "lm_head.weight" if design == "qwen3" else "head"
    embed = "model.embed_tokens.weight" if design == "qwen3" else "embed"
    layer_params = sum(math.prod(s) for n, s in shapes.items() if n not in (head, embed))
    head_params = math.prod(shapes[head])
    width = shapes[head][1]
    # per layer: (key size, value size, query heads, cached elements a token, bytes of state a sequence, flops a token of the recurrence)
    if design == "qwen3":
        mixers = [(cfg.head_dim, cfg.head_dim, cfg.num_attention_heads, 2 * cfg.num_key_value_heads * cfg.head_dim, 0, 0)] * cfg.num_hidden_layers
    else:
        mixers = []
        for m, _ in cfg.layers:
            if isinstance(m, BiasAttentionConfig):
                mixers.append((m.dim, m.vdim, m.heads, m.kv_heads * (m.dim + m.vdim), 0, 0))
            elif isinstance(m, LatentMixerConfig):
                mixers.append((m.dim + m.rot_dim, m.vdim, m.heads, m.kv_rank + m.rot_dim, 0, 0))
            elif isinstance(m, ScanMixerConfig):
                mixers.append((0, 0, 0, 0, 4 * m.inner * m.state, 6 * m.inner * m.state))
            else:
                elems = m.heads * m.dim * m.vdim
                mixers.append((0, 0, 0, 0, 4 * elems, (7 if isinstance(m, ChannelDeltaConfig) else 5) * elems))
    lengths = _lengths(case)
    passes = []  # (rows, keys seen by all rows, cached tokens read, rows of the head)
    if case["call"] in ("score", "request"):
        passes.append((sum(lengths), sum(n * (n + 1) / 2 for n in lengths), 0))
    for k in range(1, case["steps"] + 1):
        seen = sum(n + k for n in lengths)
        passes.append((case["batch"], seen, seen))
    total = {"bytes": 0.0, "flops": 0.0}
    for rows, seen, cached in passes:
        total["bytes"] += 2 * (layer_params + head_params) + rows * width * 2
        total["flops"] += 2 * rows * layer_params + 2 * case["batch"] * head_params
        for key, value, heads, elems, state, recur in mixers:
            total["bytes"] += kv_bits / 8 * elems * (cached + rows) + state * case["batch"] * (2 if cached else 1)
            total["flops"] += 2 * heads * (key + value) * seen + recur * rows
    total["bytes"] += 4 * case["batch"] * cfg.vocab_size
    return total


def tolerance(case):
    """about four times the error measured against `exact`: an f16 cache leaves 3.5e-4 (0.6B) to 6.2e-4 (8B layers), a 24-bit one 2.3e-5, the
    layered decoders 9e-5 and, in 32 bits, 1.3e-6; a rounded near-tie may flip a greedy id"""
    rel = {"qwen3-0.6b": 1.5e-3, "qwen3-0.6b-kv24": 1e-4, "qwen3-8b-4-layers": 2.5e-3, "gopunex-2k": 4e-4, "gopunex-1k-f32": 6e-6, "tafopel-1k": 4e-4}
    return {"rel": rel[case["model"]], "max": 20 * rel[case["model"]], "differ": 0.01}


# ---- the same in 64 bits, plain torch -------------------------------------------------------------------------------------------
def _rms(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _softmax(s, sink=None):
    """causal softmax of [..., T, T] scores, with one more term exp(sink) below"""
    n = s.shape[-1]
    s = s.masked_fill(torch.ones(n, n, dtype=torch.bool, device=s.device).triu(1), -math.inf)
    if sink is None:
        return s.softmax(-1)
    top = torch.maximum(s.amax(-1, keepdim=True), sink)
    e = (s - top).exp()
    return e / (e.sum(-1, keepdim=True) + (sink - top).exp())


def _each(x, sequences, f):
    """f on the rows of every sequence"""
    return torch.cat([f(a) for a in x.split(sequences)])


def _exact_qwen3(cfg, w, ids, sequences):
    H, G, D = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim
    pos = torch.cat([torch.arange(n, device=ids.device) for n in sequences]).double()
    ang = pos[:, None] * cfg.rope_theta ** (-2.0 * torch.arange(D // 2, device=ids.device).double() / D)
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]

    def rope(x):
        u, v = x[..., :D // 2], x[..., D // 2:]
        return torch.cat([u * cos - v * sin, v * cos + u * sin], -1)

    x = w("model.embed_tokens.weight")[ids]
    for l in range(cfg.num_hidden_layers):
        p = f"model.layers.{l}."
        h = _rms(x, w(p + "input_layernorm.weight"), cfg.rms_norm_eps)
        q, k, v = ((h @ w(p + f"self_attn.{n}_proj.weight").T).unflatten(-1, (-1, D)) for n in "qkv")
        q = rope(_rms(q, w(p + "self_attn.q_norm.weight"), cfg.rms_norm_eps))
        k = rope(_rms(k, w(p + "self_attn.k_norm.weight"), cfg.rms_norm_eps))

        def attend(a):
            q, k, v = (b.transpose(0, 1) for b in a.split((H, G, G), 1))
            k, v = k.repeat_interleave(H // G, 0), v.repeat_interleave(H // G, 0)
            return (_softmax(q @ k.transpose(1, 2).contiguous() * D ** -0.5) @ v).transpose(0, 1).flatten(1)

        x = x + _each(torch.cat([q, k, v], 1), sequences, attend) @ w(p + "self_attn.o_proj.weight").T
        h = _rms(x, w(p + "post_attention_layernorm.weight"), cfg.rms_norm_eps)
        a = torch.nn.functional.silu(h @ w(p + "mlp.gate_proj.weight").T) * (h @ w(p + "mlp.up_proj.weight").T)
        x = x + a @ w(p + "mlp.down_proj.weight").T
    return lambda rows: _rms(x[rows], w("model.norm.weight"), cfg.rms_norm_eps) @ w("lm_head.weight").T


def _conv(x, sequences, taps):
    """causal convolution of every channel, last tap on the current row"""
    def one(a):
        a = torch.cat([a.new_zeros(taps.shape[1] - 1, a.shape[1]), a])
        return sum(a[i:len(a) - taps.shape[1] + 1 + i] * taps[:, i] for i in range(taps.shape[1]))
    return _each(x, sequences, one)


def _over_time(sequences, rows, state, step):
    """step(state, rows of one position of every sequence) -> (state, output rows), position by position; rows: tensors [rows, ...]"""
    pad = [torch.nn.utils.rnn.pad_sequence(r.split(sequences)) for r in rows]
    out = []
    for t in range(max(sequences)):
        state, y = step(state, [p[t] for p in pad])
        out.append(y)
    out = torch.stack(out, 1)
    return torch.cat([out[i, :n] for i, n in enumerate(sequences)])


def _exact_gopunex(cfg, w, ids, sequences):
    eps, silu, B, dev = cfg.norm_eps, torch.nn.functional.silu, len(sequences), ids.device
    x = w("embed")[ids] * cfg.embed_scale
    first = None
    for l, (m, ff) in enumerate(cfg.layers):
        p = f"l{l}.mix."
        if isinstance(m, BiasAttentionConfig):
            q, k, v = (x @ w(p + n).T + w(p + n + ".b") for n in "qkv")
            q, k = _rms(q, w(p + "q.norm"), eps), _rms(k, w(p + "k.norm"), eps)
            if m.v_mix:
                own = v
                v = v if first is None else (1 - w(p + "vmix")) * v + w(p + "vmix") * first
                first = own if first is None else first
            half = m.bias_rows // 2
            row = [n if n < half else min(m.bias_rows - 1, half + int(math.floor(math.log(n / half) / math.log(m.bias_max / half) * (m.bias_rows - half) + 1e-9)))
                   for n in range(max(sequences))]
            by_distance = w(p + "rel")[torch.tensor(row, device=dev)].T

            def attend(a):
                q, k, v = (b.unflatten(1, (-1, m.dim)).transpose(0, 1) for b in a.split((m.heads * m.dim, m.kv_heads * m.dim, m.kv_heads * m.vdim), 1))
                k, v = (b.repeat_interleave(m.heads // m.kv_heads, 0) for b in (k, v))
                n = torch.arange(len(a), device=dev)
                bias = by_distance[:, (n[:, None] - n).clamp(min=0)]
                return (_softmax(q @ k.transpose(1, 2).contiguous() * m.scale + bias, torch.zeros(1, device=dev).double()) @ v).transpose(0, 1).flatten(1)

            y = _each(torch.cat([q, k, v], 1), sequences, attend)
        elif isinstance(m, LightningConfig):
            q, k, v = (silu(x @ w(p + n).T).unflatten(1, (m.heads, -1)) for n in "qkv")
            decay = torch.tensor(m.decay, device=dev).double()[:, None, None]

            def step(S, r):
                q, k, v = r
                S = decay * S + k[..., None] * v[..., None, :]
                return S, (q[..., None, :] @ S).squeeze(-2)

            y = _over_time(sequences, (q, k, v), torch.zeros(B, m.heads, m.dim, m.vdim, device=dev).double(), step).flatten(1)
            y = _rms(y, w(p + "norm"), eps) * torch.sigmoid(x @ w(p + "g").T)
        else:
            q, k, v = (silu(_conv(x @ w(p + n).T, sequences, w(p + n + ".conv"))) for n in "qkv")
            q, k = (a.unflatten(1, (m.kv_heads, -1)) for a in (q, k))
            q, k = ((a / (a.square().sum(-1, keepdim=True) + 1e-6).sqrt()).repeat_interleave(m.heads // m.kv_heads, 1) for a in (q, k))
            z = (x @ w(p + "a1").T) @ w(p + "a2").T + w(p + "dt_bias")
            g = (-w(p + "A_log").exp()[:, None] * torch.nn.functional.softplus(z).unflatten(1, (m.heads, -1))).exp()

            def step(S, r):
                q, k, v, g, beta = r
                S = g[..., None] * S
                u = beta[..., None] * (v - (k[..., None, :] @ S).squeeze(-2))
                S = S + k[..., None] * u[..., None, :]
                return S, (q[..., None, :] @ S).squeeze(-2)

            rows = (q * m.dim ** -0.5, k, v.unflatten(1, (m.heads, -1)), g, torch.sigmoid(x @ w(p + "b").T))
            y = _over_time(sequences, rows, torch.zeros(B, m.heads, m.dim, m.vdim, device=dev).double(), step)
            y = (_rms(y, w(p + "norm"), eps) * torch.sigmoid((x @ w(p + "g1").T) @ w(p + "g2").T).view_as(y)).flatten(1)
        x = x + cfg.residual_mult * _rms(y @ w(p + "o").T, 1 + w(f"l{l}.norm1"), eps)
        y = (x @ w(f"l{l}.mlp.up").T).clamp(min=0).square() @ w(f"l{l}.mlp.down").T
        x = x + cfg.residual_mult * _rms(y, 1 + w(f"l{l}.norm2"), eps)
    return lambda rows: _rms(x[rows], 1 + w("final.norm"), eps) @ w("head").T


def _exact_tafopel(cfg, w, ids, sequences):
    eps, silu, B, dev = cfg.norm_eps, torch.nn.functional.silu, len(sequences), ids.device

    def norm(x, weight):
        return torch.nn.functional.layer_norm(x, x.shape[-1:], eps=eps) * weight

    def rotation(m):
        n, y = m.rot_dim, m.yarn
        lo, hi = (n * math.log(y.original / (2 * math.pi * t)) / (2 * math.log(m.rot_base)) for t in (y.fast, y.slow))
        lo, hi = max(math.floor(lo), 0), min(math.ceil(hi), n - 1)
        i = torch.arange(n // 2, device=dev).double()
        f = m.rot_base ** (-2.0 * i / n)
        ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0, 1)
        pos = torch.cat([torch.arange(k, device=dev) for k in sequences]).double()
        return pos[:, None] * (f / y.factor * ramp + f * (1 - ramp)), 0.1 * math.log(y.factor) + 1

    def rope(x, ang, mult):
        cos, sin = ang.cos() * mult, ang.sin() * mult
        u, v = x[..., 0::2], x[..., 1::2]
        return torch.stack([u * cos - v * sin, v * cos + u * sin], -1).flatten(-2)

    x = w("embed")[ids]
    for l, (m, mlp) in enumerate(cfg.layers):
        p = f"l{l}.mix."
        h = norm(x, w(f"l{l}.norm1"))
        if isinstance(m, ScanMixerConfig):
            xz = h @ w(p + "in").T
            u, z = silu(_conv(xz[:, :m.inner], sequences, w(p + "conv")) + w(p + "conv.b")), xz[:, m.inner:]
            d = u @ w(p + "x").T
            dt = torch.nn.functional.softplus(d[:, :m.dt_rank] @ w(p + "dt").T + w(p + "dt.b"))
            A = -w(p + "A_log").exp()

            def step(S, r):
                u, dt, b, c = r
                S = (dt[..., None] * A).exp() * S + (dt * u)[..., None] * b[:, None]
                return S, (S @ c[..., None]).squeeze(-1)

            y = _over_time(sequences, (u, dt, d[:, m.dt_rank:m.dt_rank + m.state], d[:, m.dt_rank + m.state:]), torch.zeros(B, m.inner, m.state, device=dev).double(), step)
            y = (y + w(p + "D") * u) * silu(z)
        else:
            ang, mult = rotation(m)
            d = h @ w(p + "dkv").T
            c, r = _rms(d[:, :m.kv_rank], w(p + "dkv.norm"), eps), rope(d[:, m.kv_rank:], ang, mult)
            q = (_rms(h @ w(p + "dq").T, w(p + "dq.norm"), eps) @ w(p + "uq").T).unflatten(1, (m.heads, -1))
            q = torch.cat([q[..., :m.dim], rope(q[..., m.dim:], ang[:, None], mult)], -1)
            k = torch.cat([(c @ w(p + "uk").T).unflatten(1, (m.heads, -1)), r[:, None].expand(-1, m.heads, -1)], -1)
            v = (c @ w(p + "uv").T).unflatten(1, (m.heads, -1))
            sink = w(p + "sink")[:, None, None]

            def attend(a):
                q, k, v = (b.transpose(0, 1) for b in a.split((m.dim + m.rot_dim, m.dim + m.rot_dim, m.vdim), 2))
                return (_softmax(q @ k.transpose(1, 2).contiguous() * m.scale, sink) @ v).transpose(0, 1).flatten(1)

            y = _each(torch.cat([q, k, v], 2), sequences, attend)
        p = f"l{l}.mlp."
        a = torch.nn.functional.gelu(h @ w(p + "gate").T, approximate="tanh") * (h @ w(p + "up").T)
        x = x + y @ w(f"l{l}.mix.o").T + a @ w(p + "down").T
    return lambda rows: norm(x[rows], w("final.norm")) @ w("head").T


def exact(case, seed):
    design = MODELS[case["model"]][0]
    cfg, dev = _config(case["model"]), "cuda" if torch.cuda.is_available() else "cpu"
    if design == "qwen3":
        shapes = cfg.hf_tensor_shapes()
        weight = lambda n: _synthetic(n, shapes[n], seed, dev)  # noqa: E731
    else:
        tensors = _state_dict(cfg, seed, dev)
        weight = lambda n: tensors[n].double()  # noqa: E731
    tokens = _tokens(case, seed)
    sequences = [len(t) for t in tokens]
    ids = torch.from_numpy(np.concatenate(tokens).astype(np.int64)).to(dev)
    head = {"qwen3": _exact_qwen3, "gopunex": _exact_gopunex, "tafopel": _exact_tafopel}[design](cfg, weight, ids, sequences)
    last = torch.tensor(np.cumsum(sequences) - 1, device=dev)
    logits = head(last).cpu().numpy()
    return {"logits": logits} if case["call"] in ("score", "extend") else {"tokens": None, "logits": logits}
