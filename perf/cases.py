"""The steps whose time counts, as a serving program takes them.

A case is one call of the engine's step function (``ModelRunner.step``) on a model that is in place: the next token of
requests whose earlier tokens are cached (``decoding`` > 0), whole prompts (``prompts`` > 0), or both in one step, as
the scheduler plans them.  The sizes are those of ``bench.py``: the layer sizes of Llama 3.2 3B and Llama 3.1 8B, and
the larger of its two sizes of Buderax (parallel layers, routed experts) and Gisodra (windowed attention with sinks,
gated linear attention, latent attention).  ``layers`` says how many of a model's layers are there; where it is less
than the whole model, the layers left out do what the others do.

A request that decodes is one token longer after every pass, as in a program; prompts are let go behind their step.
"""

from __future__ import annotations

import math
import zlib

import torch

from fastgen_amd.engine import Model, ModelRunner, StepEntry

PAGE = 64
FEED = 8192  # tokens of a step that brings the requests' earlier tokens into the cache

_LLAMA = dict(architectures=["LlamaForCausalLM"], rms_norm_eps=1e-5, vocab_size=128256, rope_theta=500000.0,
              max_position_embeddings=131072)


def _scaling(factor):
    return dict(rope_type="llama3", factor=factor, low_freq_factor=1.0, high_freq_factor=4.0,
                original_max_position_embeddings=8192)


def config_of(case):
    """The model's ``config.json`` as a dict."""
    n = case["layers"]
    if case["model"] == "llama-3b":
        return dict(_LLAMA, hidden_size=3072, intermediate_size=8192, num_hidden_layers=n, num_attention_heads=24,
                    num_key_value_heads=8, rope_scaling=_scaling(32.0), tie_word_embeddings=True)
    if case["model"] == "llama-8b":
        return dict(_LLAMA, hidden_size=4096, intermediate_size=14336, num_hidden_layers=n, num_attention_heads=32,
                    num_key_value_heads=8, rope_scaling=_scaling(8.0), tie_word_embeddings=False)
    if case["model"] == "buderax":
        mixer = dict(heads=16, kv_heads=4, dim=128, vdim=128, scale=128**-0.5,
                     rot=dict(base=1000000.0, dims=64, scaling=dict(factor=8.0)))
        mlp = dict(kind="moe", router=dict(experts=32, top=4), expert=dict(ff=768))
        return dict(architecture="Buderax", width=2048, vocab=32000, embedding=dict(scale=2.0), norm=dict(eps=1e-6),
                    layers=[dict(type="attention", mixer=mixer, mlp=mlp) for _ in range(n)])
    if case["model"] == "gisodra":
        ff = dict(kind="dense", ff=5632)
        mask = dict(size=4096)

        def attention(**more):
            return dict(type="attention", mlp=ff, mixer=dict(heads=16, kv_heads=4, dim=128, vdim=128,
                                                             scale=128**-0.5, mask=mask, **more))

        gla = dict(type="gla", mlp=None, mixer=dict(heads=16, dim=128, vdim=128, tau=16.0))
        latent = dict(type="latent_attention", mlp=ff, mixer=dict(
            heads=16, dim=128, rot_dim=64, vdim=128, kv_rank=192, q_rank=768, scale=192**-0.5, mask=mask,
            rot=dict(base=1000000.0, dims=64)))
        layers = []
        for i in range(0, n, 4):
            layers += [attention(), gla, attention(kv_from=i), latent]
        return dict(architecture="Gisodra", width=2048, vocab=32000, norm=dict(eps=1e-6), logit_softcap=30.0,
                    layers=layers[:n])
    raise ValueError(case["model"])


def _case(model, dtype, layers, decoding=0, context=(0, 0), prompts=0, prompt=(0, 0), **name):
    return dict(name, model=model, dtype=dtype, layers=layers, decoding=decoding, context_low=context[0],
                context_high=context[1], prompts=prompts, prompt_low=prompt[0], prompt_high=prompt[1])


def listed():
    return [
        # somebody types to a small model and waits for the next word: latency and launches
        _case("llama-3b", "bf16", 28, 1, (150, 150), name="3b one reply"),
        # the decode step that bench.py quotes: eight requests of about 2,048 tokens
        _case("llama-8b", "bf16", 32, 8, (1900, 2200), name="8b decode 8"),
        # a busy server: many requests of all lengths
        _case("llama-8b", "bf16", 16, 64, (100, 2400), name="8b decode 64"),
        # two people in long documents: the cache is most of what a step reads
        _case("llama-8b", "bf16", 8, 2, (12000, 20000), name="8b long documents"),
        # the prompt that bench.py quotes
        _case("llama-8b", "bf16", 32, prompts=1, prompt=(2048, 2048), name="8b prompt 2048"),
        # continuous batching: new prompts beside the requests that decode
        _case("llama-3b", "bf16", 28, 24, (100, 1500), 2, (300, 1100), name="3b prompts beside decode"),
        # the 32-bit path: a prompt, and the next token of a few requests
        _case("llama-3b", "fp32", 7, prompts=1, prompt=(400, 400), name="3b fp32 prompt 400"),
        _case("llama-3b", "fp32", 7, 4, (200, 500), name="3b fp32 decode 4"),
        # routed experts: two prompts of odd lengths, and a batch that decodes
        _case("buderax", "bf16", 8, prompts=2, prompt=(611, 1437), name="buderax two prompts"),
        _case("buderax", "bf16", 8, 12, (300, 1400), name="buderax decode 12"),
        # recurrent, windowed and latent layers: one prompt, and a batch that decodes
        _case("gisodra", "bf16", 8, prompts=1, prompt=(2000, 2000), name="gisodra prompt 2000"),
        _case("gisodra", "bf16", 8, 8, (900, 1200), name="gisodra decode 8"),
    ]


def draw(rng):
    def spread(low, high):
        return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))

    model, dtype, layers = rng.choice([("llama-3b", "bf16", 28), ("llama-8b", "bf16", 16), ("llama-3b", "fp32", 7),
                                       ("buderax", "bf16", 8), ("gisodra", "bf16", 8)])
    kind = rng.choice(["decode", "decode", "prompt", "prompt", "both"])
    decoding = prompts = 0
    context = prompt = (0, 0)
    if kind != "prompt":
        decoding = spread(1, 8 if dtype == "fp32" else 64)
        # (the tokens that requests bring along are fed for every state: 60,000 at most)
        context = sorted((spread(30, 3000), spread(30, min(12000, 60000 // decoding))))
        if dtype == "fp32":
            context = [min(c, 600) for c in context]
    if kind != "decode":
        prompts = rng.randint(1, 3)
        longest = (500 if dtype == "fp32" else 2048) // prompts
        prompt = sorted((spread(16, longest), spread(16, longest)))
    return _case(model, dtype, layers, decoding, tuple(context), prompts, tuple(prompt))


# ---------------------------------------------------------------- inputs
def _lengths(n, low, high, phase):
    """``n`` lengths spread over ``low .. high``, the same for every seed."""
    if n == 1:
        return [high]
    return [low + int((high - low) * ((i * 0.6180339887 + phase) % 1.0)) for i in range(n)]


class Weights:
    """A checkpoint: tensors by name, drawn from the seed when they are asked for."""

    def __init__(self, config, seed, dtype):
        self.seed, self.dtype = seed, dtype
        self.shapes = _llama_shapes(config) if "architectures" in config else (
            _buderax_shapes(config) if config["architecture"] == "Buderax" else _gisodra_shapes(config))
        self.llama = "architectures" in config
        self.layers = config.get("num_hidden_layers") or len(config["layers"])
        self.zero_centred = config.get("architecture") == "Buderax"

    def names(self):
        return list(self.shapes)

    def shape(self, name):
        return self.shapes[name]

    def get(self, name):
        shape = self.shapes[name]
        g = torch.Generator(device="cuda").manual_seed(zlib.crc32(f"{self.seed}:{name}".encode()))
        t = torch.randn(shape, generator=g, device="cuda", dtype=self.dtype)
        # what goes into the stream is scaled down by depth, as such models are initialised
        depth = (2 * self.layers) ** -0.5
        if name.endswith(("norm1b", "norm2b")):
            return t.mul_(0.2).add_(1.0).mul_(depth)
        if "norm" in name:
            return t.mul_(0.1 if self.llama else 0.2).add_(0.0 if self.zero_centred else 1.0)
        if self.llama:
            if "embed" in name or "head" in name:
                return t.mul_(0.02)
            behind = name.endswith(("o_proj.weight", "down_proj.weight"))
            return t.mul_(shape[-1] ** -0.5 * (depth if behind else 1.0))
        if name.endswith(".a2.b"):
            return t.add_(2.0)  # decays near one
        if len(shape) == 1:
            return t if name.endswith("sink") else t.mul_(0.3)
        if name == "embed":
            return t.mul_(0.5) if self.zero_centred else t.mul_(1.0)
        if name.endswith("router"):
            return t.mul_(2.0 * shape[-1] ** -0.5)
        behind = self.zero_centred and name.endswith((".mix.o", ".down"))
        return t.mul_(shape[-1] ** -0.5 * (depth if behind else 1.0))


def _llama_shapes(c):
    D, F, V = c["hidden_size"], c["intermediate_size"], c["vocab_size"]
    kv = c["num_key_value_heads"] * (D // c["num_attention_heads"])
    s = {"model.embed_tokens.weight": (V, D), "model.norm.weight": (D,)}
    if not c["tie_word_embeddings"]:
        s["lm_head.weight"] = (V, D)
    for i in range(c["num_hidden_layers"]):
        p = f"model.layers.{i}."
        s.update({p + "self_attn.q_proj.weight": (D, D), p + "self_attn.k_proj.weight": (kv, D),
                  p + "self_attn.v_proj.weight": (kv, D), p + "self_attn.o_proj.weight": (D, D),
                  p + "mlp.gate_proj.weight": (F, D), p + "mlp.up_proj.weight": (F, D),
                  p + "mlp.down_proj.weight": (D, F), p + "input_layernorm.weight": (D,),
                  p + "post_attention_layernorm.weight": (D,)})
    return s


def _buderax_shapes(c):
    D, V = c["width"], c["vocab"]
    s = {"embed": (V, D), "final.norm": (D,), "head": (V, D)}
    for i, layer in enumerate(c["layers"]):
        m, r, ff, p = layer["mixer"], layer["mlp"]["router"], layer["mlp"]["expert"]["ff"], f"l{i}"
        H, G, d = m["heads"], m["kv_heads"], m["dim"]
        s.update({f"{p}.norm1": (D,), f"{p}.mix.q": (H * d, D), f"{p}.mix.k": (G * d, D), f"{p}.mix.g": (H * d, D),
                  f"{p}.mix.o": (D, H * d), f"{p}.mlp.router": (r["experts"], D), f"{p}.mlp.router.b": (r["experts"],)})
        for e in range(r["experts"]):
            s.update({f"{p}.mlp.e{e}.gate": (ff, D), f"{p}.mlp.e{e}.up": (ff, D), f"{p}.mlp.e{e}.down": (D, ff)})
    return s


def _gisodra_shapes(c):
    D, V = c["width"], c["vocab"]
    s = {"embed": (V, D), "final.norm": (D,)}
    for i, layer in enumerate(c["layers"]):
        m, p = layer["mixer"], f"l{i}.mix"
        s.update({f"l{i}.norm1": (D,), f"l{i}.norm1b": (D,)})
        H, d, e = m["heads"], m["dim"], m["vdim"]
        if layer["type"] == "attention":
            G = m["kv_heads"]
            s.update({f"{p}.q": (H * d, D), f"{p}.q.b": (H * d,), f"{p}.q.norm": (d,), f"{p}.sink": (H,),
                      f"{p}.o": (D, H * e)})
            if "kv_from" not in m:
                s.update({f"{p}.k": (G * d, D), f"{p}.k.b": (G * d,), f"{p}.v": (G * e, D), f"{p}.v.b": (G * e,),
                          f"{p}.k.norm": (d,)})
        elif layer["type"] == "gla":
            s.update({f"{p}.q": (H * d, D), f"{p}.k": (H * d, D), f"{p}.v": (H * e, D), f"{p}.g": (H * e, D),
                      f"{p}.o": (D, H * e), f"{p}.norm": (e,), f"{p}.a1": (16, D), f"{p}.a2": (H * d, 16),
                      f"{p}.a2.b": (H * d,)})
        else:
            r, R, Q = m["rot_dim"], m["kv_rank"], m["q_rank"]
            s.update({f"{p}.dq": (Q, D), f"{p}.dq.norm": (Q,), f"{p}.uq": (H * (d + r), Q), f"{p}.dkv": (R + r, D),
                      f"{p}.dkv.norm": (R,), f"{p}.uk": (H * d, R), f"{p}.uv": (H * e, R), f"{p}.sink": (H,),
                      f"{p}.g": (H, D), f"{p}.o": (D, H * e)})
        if layer["mlp"] is not None:
            F = layer["mlp"]["ff"]
            s.update({f"l{i}.norm2": (D,), f"l{i}.norm2b": (D,), f"l{i}.mlp.gate": (F, D), f"l{i}.mlp.up": (F, D),
                      f"l{i}.mlp.down": (D, F)})
    return s


def _tokens(case, seed):
    """(earlier tokens of the requests that decode, their next tokens pass by pass, prompts)."""
    vocab = config_of(case).get("vocab") or config_of(case)["vocab_size"]
    g = torch.Generator().manual_seed(seed)

    def some(n):
        return torch.randint(0, vocab, (n,), generator=g).tolist()

    earlier = [some(n) for n in _lengths(case["decoding"], case["context_low"], case["context_high"], 0.3)]
    prompts = [some(n) for n in _lengths(case["prompts"], case["prompt_low"], case["prompt_high"], 0.1)]
    return earlier, [some(256) for _ in earlier], prompts


def _dtype(case):
    return torch.float32 if case["dtype"] == "fp32" else torch.bfloat16


class State:
    def __init__(self, runner, following, prompts):
        self.runner, self.following, self.prompts, self.passes = runner, following, prompts, 0


def prepare(case, seed):
    """A model with its cache, the earlier tokens of the requests that decode in place, one decode step taken."""
    dtype = _dtype(case)
    config = config_of(case)
    model = Model.from_config(config, dtype, "cuda:0")
    model.load(Weights(config, seed, dtype))
    earlier, following, prompts = _tokens(case, seed)
    room = 8192 if case["decoding"] <= 16 else 3072  # tokens that a request may still get
    held = sum(len(t) + room + PAGE for t in earlier) + sum(len(t) + PAGE for t in prompts)
    runner = ModelRunner(model, page_size=PAGE, max_tokens=held, max_requests=max(1, len(earlier) + len(prompts)))
    entries, n = [], 0
    for i, t in enumerate(earlier):
        at = 0
        while at < len(t):
            take = min(FEED - n, len(t) - at)
            entries.append(StepEntry(i, t[at:at + take]))
            at, n = at + take, n + take
            if n == FEED:
                runner.step(entries)
                entries, n = [], 0
    if entries:
        runner.step(entries)
    state = State(runner, following, prompts)
    if earlier:
        runner.step([StepEntry(i, [t[0]], [0]) for i, t in enumerate(following)])
        state.passes = 1
    return state


def run(state):
    runner, at = state.runner, state.passes
    state.passes = at + 1
    entries = [StepEntry(i, [t[at % len(t)]], [0]) for i, t in enumerate(state.following)]
    entries += [StepEntry(("prompt", i), t, [len(t) - 1]) for i, t in enumerate(state.prompts)]
    logits = runner.step(entries)
    for i in range(len(state.prompts)):
        runner.release(("prompt", i))
    # the recurrent layers' states of the requests that go on
    n = len(state.following)
    return {"logits": logits, "states": [t[:n] for _, t in sorted(runner.storage.state.items())] if n else []}


# ---------------------------------------------------------------- what a pass needs
def _sizes(case):
    """(weights of one token's products, weights of all products, cached values a token, state values a request,
    heads x head width of the attention summed over layers, head's weights)."""
    c = config_of(case)
    if "architectures" in c:
        D, F, n = c["hidden_size"], c["intermediate_size"], c["num_hidden_layers"]
        hd = D // c["num_attention_heads"]
        per = 2 * D * D + 2 * D * c["num_key_value_heads"] * hd + 3 * D * F
        return n * per, n * per, n * 2 * c["num_key_value_heads"] * hd, 0, n * D, c["vocab_size"] * D
    D, each, every, cached, state, wide = c["width"], 0, 0, 0, 0, 0
    for i, layer in enumerate(c["layers"]):
        m, mlp = layer["mixer"], layer["mlp"]
        H, d, e = m["heads"], m["dim"], m["vdim"]
        if c["architecture"] == "Buderax":
            mix = D * (3 * H * d + m["kv_heads"] * d)
            cached += 2 * m["kv_heads"] * d
            wide += H * d
        elif layer["type"] == "attention":
            own = 0 if "kv_from" in m else m["kv_heads"] * (d + e)
            mix = D * (H * d + H * e + own)
            cached += m["kv_heads"] * (d + e)  # (a layer that reads another's cache reads as much)
            wide += H * d
        elif layer["type"] == "gla":
            mix = D * (2 * H * d + 3 * H * e)
            state += H * d * e
        else:
            R, r, Q = m["kv_rank"], m["rot_dim"], m["q_rank"]
            mix = D * (Q + R + r + H * e) + Q * H * (d + r) + R * H * (d + e)
            cached += R + r
            wide += H * d
        each, every = each + mix, every + mix
        if mlp is not None and mlp["kind"] == "moe":
            r, ff = mlp["router"], mlp["expert"]["ff"]
            tokens = case["decoding"] + sum(_lengths(case["prompts"], case["prompt_low"], case["prompt_high"], 0.1))
            each += r["experts"] * D + r["top"] * 3 * D * ff
            every += r["experts"] * D + min(r["experts"], tokens * r["top"]) * 3 * D * ff
        elif mlp is not None:
            each, every = each + 3 * D * mlp["ff"], every + 3 * D * mlp["ff"]
    return each, every, cached, state, wide, c["vocab"] * D


def work(case):
    each, every, cached, state, wide, head = _sizes(case)
    size = 4 if case["dtype"] == "fp32" else 2
    contexts = _lengths(case["decoding"], case["context_low"], case["context_high"], 0.3)
    prompts = _lengths(case["prompts"], case["prompt_low"], case["prompt_high"], 0.1)
    rows, tokens = len(contexts) + len(prompts), len(contexts) + sum(prompts)
    pairs = sum(contexts) + sum(n * (n + 1) // 2 for n in prompts)
    nbytes = (every + head + cached * (sum(contexts) + tokens)) * size + 2 * 4 * state * rows
    nbytes += rows * 4 * (config_of(case).get("vocab") or config_of(case)["vocab_size"])
    return {"bytes": nbytes, "flops": 2 * tokens * each + 2 * rows * head + 4 * pairs * wide + 4 * tokens * state}


def tolerance(case):
    """Four times what the same step shows when its tokens come in other portions, so that other kernels sum in
    another order: bfloat16 0.002 to 0.013 (largest difference 0.006 to 0.06; what 64 bits give is as far away; an
    expert chosen otherwise at a tie moves more), 32-bit within 4e-6 and 2e-5 of what 64 bits give (and the same
    bits under every cut)."""
    if case["dtype"] == "fp32":
        return {"rel": 1.5e-5, "max": 1e-4}
    return {"rel": 0.03, "max": 0.3}


# ---------------------------------------------------------------- the same in 64 bits
def _norm(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _turn(x, pos, freqs, pairs):
    """``x [T, heads, n]``; ``pairs``: (2i, 2i+1), else (i, i + n/2) of the first ``2 len(freqs)`` elements."""
    n = 2 * freqs.numel()
    angle = pos[:, None].double() * freqs[None, :]
    c, s = torch.cos(angle)[:, None, :], torch.sin(angle)[:, None, :]
    a, b = (slice(0, n, 2), slice(1, n, 2)) if pairs else (slice(0, n // 2), slice(n // 2, n))
    out = x.clone()
    out[..., a] = x[..., a] * c - x[..., b] * s
    out[..., b] = x[..., b] * c + x[..., a] * s
    return out


def _attend(q, k, v, starts, scale, window=None, sink=None):
    """Causal attention of every sequence (``starts``: its first row) over itself; kv heads shared by groups."""
    heads, groups = q.shape[1], k.shape[1]
    out = torch.empty(q.shape[0], heads, v.shape[2], dtype=q.dtype, device=q.device)
    for a, b in zip(starts, starts[1:]):
        for i in range(a, b, 2048):
            j = min(i + 2048, b)
            row, col = torch.arange(i, j, device=q.device)[:, None], torch.arange(a, j, device=q.device)[None, :]
            hidden = col > row if window is None else (col > row) | (row - col >= window)
            for h in range(heads):
                g = h // (heads // groups)
                s = ((q[i:j, h] @ k[a:j, g].T) * scale).masked_fill_(hidden, -math.inf)
                if sink is not None:  # one more term of the denominator, without a value
                    s = torch.cat([s, sink[h].expand(j - i, 1)], 1)
                p = torch.softmax(s, -1)
                out[i:j, h] = p[:, :j - a] @ v[a:j, g]
    return out


def _exact_llama(c, W, tok, pos, starts, want):
    D, H, KV, eps = c["hidden_size"], c["num_attention_heads"], c["num_key_value_heads"], c["rms_norm_eps"]
    hd, T, s = D // H, tok.numel(), c["rope_scaling"]
    freqs = c["rope_theta"] ** (-torch.arange(0, hd, 2, dtype=torch.float64, device="cuda") / hd)
    turns = s["original_max_position_embeddings"] * freqs / (2 * math.pi)
    blend = ((turns - s["low_freq_factor"]) / (s["high_freq_factor"] - s["low_freq_factor"])).clamp(0, 1)
    freqs = blend * freqs + (1 - blend) * freqs / s["factor"]
    x = W("model.embed_tokens.weight", tok)
    for i in range(c["num_hidden_layers"]):
        p = f"model.layers.{i}."
        n = _norm(x, W(p + "input_layernorm.weight"), eps)
        q = _turn((n @ W(p + "self_attn.q_proj.weight").T).view(T, H, hd), pos, freqs, False)
        k = _turn((n @ W(p + "self_attn.k_proj.weight").T).view(T, KV, hd), pos, freqs, False)
        v = (n @ W(p + "self_attn.v_proj.weight").T).view(T, KV, hd)
        x = x + _attend(q, k, v, starts, hd**-0.5).view(T, D) @ W(p + "self_attn.o_proj.weight").T
        n = _norm(x, W(p + "post_attention_layernorm.weight"), eps)
        a = torch.nn.functional.silu(n @ W(p + "mlp.gate_proj.weight").T)
        a *= n @ W(p + "mlp.up_proj.weight").T
        x = x + a @ W(p + "mlp.down_proj.weight").T
    head = "model.embed_tokens.weight" if c["tie_word_embeddings"] else "lm_head.weight"
    return _norm(x[want], W("model.norm.weight"), eps) @ W(head).T, []


def _exact_buderax(c, W, tok, pos, starts, want):
    eps, T = c["norm"]["eps"], tok.numel()
    x = W("embed", tok) * c["embedding"]["scale"]
    for i, layer in enumerate(c["layers"]):
        m, p, router = layer["mixer"], f"l{i}", layer["mlp"]["router"]
        H, G, d, dims = m["heads"], m["kv_heads"], m["dim"], m["rot"]["dims"]
        n = _norm(x, 1 + W(p + ".norm1"), eps)
        i2 = torch.arange(0, dims, 2, dtype=torch.float64, device="cuda")
        freqs = m["rot"]["base"] ** (-i2 / dims) / m["rot"]["scaling"]["factor"]
        q, k = (n @ W(p + ".mix.q").T).view(T, H, d), (n @ W(p + ".mix.k").T).view(T, G, d)
        o = _attend(_turn(q, pos, freqs, True), _turn(k, pos, freqs, True), k, starts, m["scale"]).view(T, H * d)
        y = (o * torch.sigmoid(n @ W(p + ".mix.g").T)) @ W(p + ".mix.o").T
        value, chosen = torch.topk(n @ W(p + ".mlp.router").T + W(p + ".mlp.router.b"), router["top"], -1)
        weight = torch.softmax(value, -1)
        for e in range(router["experts"]):
            row, place = (chosen == e).nonzero(as_tuple=True)
            ne = n[row]
            a = torch.nn.functional.silu(ne @ W(f"{p}.mlp.e{e}.gate").T) * (ne @ W(f"{p}.mlp.e{e}.up").T)
            y.index_add_(0, row, weight[row, place][:, None] * (a @ W(f"{p}.mlp.e{e}.down").T))
        x = x + y
    return _norm(x[want], 1 + W("final.norm"), eps) @ W("head").T, []


def _exact_gla(q, k, v, decay, starts):
    """``S <- decay_t S + k_t v_t^T``, ``o_t = S^T q_t``: the outputs, and every sequence's last state."""
    n = len(starts) - 1
    out = torch.empty_like(v)
    first = torch.tensor(starts[:-1], device=q.device)
    length = torch.tensor([b - a for a, b in zip(starts, starts[1:])], device=q.device)
    S = torch.zeros(n, q.shape[1], q.shape[2], v.shape[2], dtype=q.dtype, device=q.device)
    for t in range(int(length.max())):
        live = (length > t).nonzero()[:, 0] if n > 1 else slice(None)
        row = (first + t)[live]
        S[live] = decay[row][..., None] * S[live] + k[row][..., None] * v[row][:, :, None, :]
        out[row] = (S[live] * q[row][..., None]).sum(2)
    return out, S


def _exact_gisodra(c, W, tok, pos, starts, want):
    eps, T, cap = c["norm"]["eps"], tok.numel(), c["logit_softcap"]
    x, kept, states = W("embed", tok), {}, []
    for i, layer in enumerate(c["layers"]):
        m, p = layer["mixer"], f"l{i}.mix"
        H, d, e = m["heads"], m["dim"], m["vdim"]
        n = _norm(x, W(f"l{i}.norm1"), eps)
        if layer["type"] == "attention":
            if "kv_from" not in m:
                k = (n @ W(p + ".k").T + W(p + ".k.b")).view(T, -1, d)
                v = (n @ W(p + ".v").T + W(p + ".v.b")).view(T, -1, e)
                kept[i] = _norm(k, W(p + ".k.norm"), eps), v
            q = _norm((n @ W(p + ".q").T + W(p + ".q.b")).view(T, H, d), W(p + ".q.norm"), eps)
            o = _attend(q, *kept[m.get("kv_from", i)], starts, m["scale"], m["mask"]["size"], W(p + ".sink"))
        elif layer["type"] == "gla":
            q, k = ((n @ W(p + w).T).view(T, H, d) for w in (".q", ".k"))
            z = (n @ W(p + ".a1").T) @ W(p + ".a2").T + W(p + ".a2.b")
            decay = torch.exp(torch.nn.functional.logsigmoid(z) / m["tau"]).view(T, H, d)
            o, S = _exact_gla(q * d**-0.5, k, (n @ W(p + ".v").T).view(T, H, e), decay, starts)
            states.append(S)
            o = _norm(o, W(p + ".norm"), eps) * torch.nn.functional.silu(n @ W(p + ".g").T).view(T, H, e)
        else:
            r, R, base, dims = m["rot_dim"], m["kv_rank"], m["rot"]["base"], m["rot"]["dims"]
            freqs = base ** (-torch.arange(0, dims, 2, dtype=torch.float64, device="cuda") / dims)
            q = (_norm(n @ W(p + ".dq").T, W(p + ".dq.norm"), eps) @ W(p + ".uq").T).view(T, H, d + r)
            both = n @ W(p + ".dkv").T
            low = _norm(both[:, :R], W(p + ".dkv.norm"), eps)
            shared = _turn(both[:, None, R:], pos, freqs, False)
            q = torch.cat([q[..., :d], _turn(q[..., d:], pos, freqs, False)], -1)
            k = torch.cat([(low @ W(p + ".uk").T).view(T, H, d), shared.expand(T, H, r)], -1)
            v = (low @ W(p + ".uv").T).view(T, H, e)
            o = _attend(q, k, v, starts, m["scale"], m["mask"]["size"], W(p + ".sink"))
            o = o * torch.sigmoid(n @ W(p + ".g").T)[:, :, None]
        x = x + _norm(o.reshape(T, -1) @ W(p + ".o").T, W(f"l{i}.norm1b"), eps)
        if layer["mlp"] is not None:
            n = _norm(x, W(f"l{i}.norm2"), eps)
            a = torch.nn.functional.gelu(n @ W(f"l{i}.mlp.gate").T, approximate="tanh") * (n @ W(f"l{i}.mlp.up").T)
            x = x + _norm(a @ W(f"l{i}.mlp.down").T, W(f"l{i}.norm2b"), eps)
    return cap * torch.tanh(_norm(x[want], W("final.norm"), eps) @ W("embed").T / cap), states


def exact(case, seed):
    """The logits of the first pass (and the states behind it) from whole sequences, in 64 bits."""
    if work(dict(case, prompts=case["prompts"] + case["decoding"], decoding=0, prompt_low=max(1, case["context_low"]),
                 prompt_high=max(case["prompt_high"], case["context_high"])))["flops"] > 8e14:
        return None
    config = config_of(case)
    source = Weights(config, seed, _dtype(case))

    def W(name, rows=None):
        t = source.get(name)
        return (t if rows is None else t[rows]).double()

    earlier, following, prompts = _tokens(case, seed)
    sequences = [e + f[:2] for e, f in zip(earlier, following)] + prompts
    starts = [0]
    for s in sequences:
        starts.append(starts[-1] + len(s))
    tok = torch.tensor([t for s in sequences for t in s], device="cuda")
    pos = torch.cat([torch.arange(len(s), device="cuda") for s in sequences])
    want = torch.tensor(starts[1:], device="cuda") - 1
    forward = _exact_llama if "architectures" in config else (
        _exact_buderax if config["architecture"] == "Buderax" else _exact_gisodra)
    logits, states = forward(config, W, tok, pos, starts, want)
    n = len(earlier)
    return {"logits": logits, "states": [S[:n] for S in states] if n else []}
