"""What this engine is measured on: single passes of `ModelRunner.step`, the one way by which tokens reach a
model (the scheduler, the trace replay and the benchmark all call it), over the sizes that a server meets.

A case is one batch: `decoding` requests that hold up to `context` tokens each and decode one more, and
`prompts` new prompts of `tokens` tokens in all, which a pass admits, runs (whole, or in steps of `portion`
tokens beside the decoding requests) and closes again.  Models are the named layer shapes of
`wllm_amd/config/shapes` with all their layers; weights are random, from generators keyed by a tensor's
name, token ids are uniform and come from the seed.  A pass returns the logits of its last step: a row
for every decoding request and for the last token of every prompt.
"""
from __future__ import annotations

import hashlib
import json
import math
import os
import random

import torch

import wllm_amd
from wllm_amd.engine import ModelRunner, StepEntry
from wllm_amd.parts import build_model

PAGE = 16                # tokens a page
ROOM = 1024              # tokens that a decoding request may add before it is closed and its prompt runs again
DTYPES = {"bfloat16": torch.bfloat16, "float32": torch.float32}


def listed():
    def case(name, shape="gemma-2b", dtype="bfloat16", decoding=0, context=0, prompts=0, tokens=0, portion=0):
        return {"name": name, "shape": shape, "dtype": dtype, "decoding": decoding, "context": context,
                "prompts": prompts, "tokens": tokens, "portion": portion}

    return [
        # one user watching an answer grow: the weights are read for a single row, launches and latency count
        case("decode 1", decoding=1, context=1900),
        # the benchmark's batch: a few users at once, prompts of up to 2,048 tokens
        case("decode 8", decoding=8, context=2048),
        # a busy server: the caches read are as large as a third of the weights, contexts far apart
        case("decode 64", decoding=64, context=3000),
        # a short chat turn: nothing but launches and one pass over the weights
        case("prompt 37", prompts=1, tokens=37),
        # the benchmark's prompt, and about the longest that the configuration's 8,192 positions hold
        case("prompt 2048", prompts=1, tokens=2048),
        case("prompt 7777", prompts=1, tokens=7777),
        # chunked prefill: a prompt in portions beside everyone who is decoding meanwhile
        case("portions beside 60", decoding=60, context=1500, prompts=1, tokens=1000, portion=448),
        # the true 32-bit path, which people run to check another implementation against: two middling prompts
        case("float32 prompts 333", dtype="float32", prompts=2, tokens=333),
        # layers of attention, latent attention and a state-space recurrence: each direction
        case("tokuvik prompt 1500", shape="tokuvik-2b", prompts=1, tokens=1500),
        case("tokuvik decode 8", shape="tokuvik-2b", decoding=8, context=1500),
        # experts, latent attention with a turned key part, a forget-gate recurrence, short convolutions: a
        # batch of prompts admitted together, and a middling batch decoding
        case("duvozen prompts 3001", shape="duvozen-2b", prompts=3, tokens=3001),
        case("duvozen decode 24", shape="duvozen-2b", decoding=24, context=800),
    ]


def draw(rng: random.Random):
    def spread(low, high):
        return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))

    u = rng.random()
    shape = "gemma-2b" if u < 0.55 else "tokuvik-2b" if u < 0.73 else "duvozen-2b" if u < 0.91 else "gemma-7b"
    dtype = "float32" if shape == "gemma-2b" and rng.random() < 0.2 else "bfloat16"
    case = {"shape": shape, "dtype": dtype, "decoding": 0, "context": 0, "prompts": 0, "tokens": 0, "portion": 0}
    kind = rng.choice(("decode", "prompt", "prompt", "portions"))
    if kind != "prompt":
        case["decoding"] = spread(1, 16 if shape == "gemma-7b" else 64)
        most = 12_000 if shape == "gemma-7b" else 96_000
        case["context"] = spread(64, min(4000, most // case["decoding"]))
    if kind != "decode":
        most = {"gemma-2b": 6000, "tokuvik-2b": 3000, "duvozen-2b": 3500, "gemma-7b": 1500}[shape]
        case["tokens"] = spread(5, 450 if dtype == "float32" else most)
        case["prompts"] = min(rng.choice((1, 1, 1, 2, 5)), case["tokens"])
    if kind == "portions":
        case["prompts"] = 1
        case["tokens"] = min(case["tokens"], 1800)
        case["portion"] = rng.choice((256, 448, 512))
    return case


# ---- lengths and token ids ---------------------------------------------------------------------------

def contexts(case):
    """Tokens that each decoding request holds before the pass: from a quarter of `context` up to all of it."""
    b, c = case["decoding"], case["context"]
    return [c - (3 * c // 4) * i // max(1, b - 1) for i in range(b)]


def prompt_lengths(case):
    """`tokens` shared out over the prompts as 1 : 2 : 3 : ..."""
    n, k = case["tokens"], case["prompts"]
    if k == 0:
        return []
    cuts = [n * i * (i + 1) // (k * (k + 1)) for i in range(k + 1)]
    return [max(1, b - a) for a, b in zip(cuts, cuts[1:])]


def steps_of(case):
    """Per step of a pass, the (prompt, first token, end) of each portion in it."""
    lengths = prompt_lengths(case)
    if not case["portion"]:
        return [[(i, 0, n) for i, n in enumerate(lengths)]]
    return [[(0, a, min(a + case["portion"], lengths[0]))] for a in range(0, lengths[0], case["portion"])]


def token_ids(case, seed):
    """Ids of the decoding requests (what they hold and what they decode next) and of the prompts."""
    vocab = vocabulary(shape_config(case["shape"]))
    g = torch.Generator().manual_seed(int(seed))

    def ids(n):
        return torch.randint(0, vocab, (n,), generator=g).tolist()

    return [ids(n + ROOM) for n in contexts(case)], [ids(n) for n in prompt_lengths(case)]


# ---- weights ---------------------------------------------------------------------------------------------

def shape_config(shape):
    with open(os.path.join(os.path.dirname(wllm_amd.__file__), "config", "shapes", shape + ".json")) as f:
        return json.load(f)


def is_gemma(config):
    return "architectures" in config


def family(config):
    return "Gemma" if is_gemma(config) else config["architecture"]


def vocabulary(config):
    return config["vocab_size"] if is_gemma(config) else config["vocab"]


def weight(name, size, family):
    """The bfloat16 numbers of a tensor, keyed by its name: matrices normal with deviation 0.02, and the small
    vectors where trained models have them."""
    g = torch.Generator(device="cuda")
    g.manual_seed(int.from_bytes(hashlib.sha256(name.encode()).digest()[:7], "little"))
    t = torch.empty(tuple(size), dtype=torch.float32, device="cuda")
    last = name.rsplit(".", 1)[-1]
    if len(size) > 1:
        # taps of a short convolution sum few terms, so their weights are larger
        # (and Duvozen takes its token vectors unscaled, so they are of the stream's own size)
        wide = 0.3 if last in ("conv", "canon1", "canon2") else 1.0 if (family, last) == ("Duvozen", "embed") else 0.02
        t.normal_(0.0, wide, generator=g)
    elif last == "A_log":                                   # decay rates 1 .. 16
        t.uniform_(1.0, 16.0, generator=g).log_()
    elif last == "dt_bias":                                 # step sizes 0.001 .. 0.1 behind the softplus
        t.uniform_(math.log(1e-3), math.log(1e-1), generator=g).exp_().expm1_().log_()
    elif last == "lower":                                   # lower bounds of forget gates
        t.uniform_(0.0, 0.95, generator=g)
    elif last == "sink" or name.endswith(".b"):
        t.normal_(0.0, 0.1, generator=g)
    elif family == "Duvozen" and last in ("norm1", "norm2"):
        # the norms behind sublayers, whose sum the next sublayer reads with no norm before it: it stays near one
        t.normal_(0.05, 0.005, generator=g)
    else:                                                   # norms, skips: around one (Gemma stores the offset)
        t.normal_(0.0 if family == "Gemma" else 1.0, 0.1, generator=g)
    return t.to(torch.bfloat16)


class Weights:
    """What `CausalLM.load_from` asks for its tensors."""

    def __init__(self, expected, dtype, family):
        self.expected, self.dtype, self.family = expected, dtype, family
        self.device, self.tiled_copies = torch.device("cuda:0"), True

    def has(self, name):
        return name in self.expected and not self.expected[name].optional

    def matrix(self, name):
        return weight(name, self.expected[name].shape, self.family).to(self.dtype)

    def vector(self, name):
        return weight(name, self.expected[name].shape, self.family).float()

    def to_device(self, t):
        return t.contiguous().to(self.device)


_loaded = {}             # the model that was asked for last: a server loads one and keeps it for every request


def loaded_model(shape, dtype):
    if (shape, dtype) not in _loaded:
        _loaded.clear()
        torch.cuda.empty_cache()
        config = shape_config(shape)
        model = build_model(config)
        model.load_from(Weights(model.expected_tensors(), DTYPES[dtype], family(config)))
        _loaded[shape, dtype] = model
    return _loaded[shape, dtype]


# ---- a pass ----------------------------------------------------------------------------------------------

def fill(state):
    """Runs the decoding requests' prompts, several in a step, and one decode step (a server's graphs of the
    batch size exist by then)."""
    runner, held = state["runner"], state["held"]
    for i in range(len(held)):
        if runner.cache.is_open(i):
            runner.close(i)
        runner.open(i)
    entries, room = [], 4096
    for i, n in enumerate(held):
        if n > room and entries:
            runner.step(entries)
            entries, room = [], 4096
        entries.append(StepEntry(i, state["decoding"][i][:n], []))
        room -= n
    if entries:
        runner.step(entries)
        runner.step([StepEntry(i, [state["decoding"][i][n]], [0]) for i, n in enumerate(held)])
    state["decoded"] = 1


@torch.inference_mode()
def prepare(case, seed):
    decoding, prompts = token_ids(case, seed)
    held, b = contexts(case), case["decoding"]
    pages = sum(-(-(n + ROOM) // PAGE) for n in held) + sum(-(-len(p) // PAGE) for p in prompts) + 2
    runner = ModelRunner.create(loaded_model(case["shape"], case["dtype"]), num_pages=pages, page_size=PAGE,
                                max_requests=b + len(prompts))
    state = {"runner": runner, "held": held, "decoding": decoding, "prompts": prompts, "steps": steps_of(case)}
    if b:
        runner.enable_graphs()
        fill(state)
    return state


@torch.inference_mode()
def run(state):
    runner, decoding, prompts = state["runner"], state["decoding"], state["prompts"]
    if decoding and state["decoded"] + len(state["steps"]) >= ROOM:
        fill(state)
    for i in range(len(prompts)):
        runner.open(("prompt", i))
    logits = None
    for portions in state["steps"]:
        entries = []
        if decoding:
            k = state["decoded"]
            entries = [StepEntry(i, [ids[n + k]], [0]) for i, (ids, n) in enumerate(zip(decoding, state["held"]))]
            state["decoded"] = k + 1
        for i, a, e in portions:
            entries.append(StepEntry(("prompt", i), prompts[i][a:e], [e - a - 1] if e == len(prompts[i]) else []))
        logits = runner.step(entries)
    for i in range(len(prompts)):
        runner.close(("prompt", i))
    return logits


# ---- what a pass cannot do without -----------------------------------------------------------------------

def layer_sizes(config):
    """Per layer: elements of its matrices that every token uses, elements of one expert, experts, experts a
    token uses, cached elements a token (and whether the layer reads another's), heads * (key + value
    elements) of a score and its weighted sum, the span of keys seen, elements of a request's state."""
    out = []
    if is_gemma(config):
        h, d = config["hidden_size"], config["head_dim"]
        q, kv = config["num_attention_heads"] * d, config["num_key_value_heads"] * d
        dense = 2 * h * q + 2 * h * kv + 3 * h * config["intermediate_size"]
        return [dict(dense=dense, expert=0, experts=0, top=0, cached=2 * kv, owns=True, heads=2 * q, span=None, state=0)
                for _ in range(config["num_hidden_layers"])]
    w = config["width"]
    for layer in config["layers"]:
        m, f = layer["mixer"], layer["mlp"]
        dim, vdim, heads = m.get("dim", 0), m["vdim"], m["heads"]
        s = dict(expert=0, experts=0, top=0, cached=0, owns="kv_from" not in m, heads=heads * (dim + vdim),
                 span=(m.get("mask") or {}).get("size"), state=0)
        if layer["type"] == "attention":
            gate = heads if config["architecture"] == "Tokuvik" else heads * vdim
            s["cached"] = m["kv_heads"] * (dim + vdim)
            s["dense"] = w * (heads * (dim + vdim) + gate + (s["cached"] if s["owns"] else 0))
        elif layer["type"] == "latent_attention":
            rot, rank = m.get("rot_dim", 0), m["kv_rank"]
            s["cached"] = rank + rot
            s["heads"] += heads * rot
            s["dense"] = w * (rank + rot + heads * vdim) + heads * (dim + vdim) * rank
            if "q_rank" in m:
                s["dense"] += m["q_rank"] * (w + heads * dim) + w * heads * vdim
            else:
                s["dense"] += w * heads * (dim + rot)
        elif layer["type"] == "mamba2":
            s["dense"] = w * (3 * heads * vdim + 2 * m["groups"] * m["state"] + heads)
            s["heads"], s["state"] = 0, heads * vdim * m["state"]
        else:
            s["dense"] = w * heads * 2 * (dim + vdim)
            s["heads"], s["state"] = 0, heads * dim * vdim
        if f["kind"] == "dense":
            s["dense"] += 3 * w * f["ff"]
        else:
            s["dense"] += 3 * w * f["shared"]["ff"] + w * f["router"]["experts"]
            s.update(expert=3 * w * f["expert"]["ff"], experts=f["router"]["experts"], top=f["router"]["top"])
        if "token_side" in config:
            s["dense"] += 2 * w * config["token_side"]["dim"]
        out.append(s)
    return out


def work(case):
    config, size = shape_config(case["shape"]), DTYPES[case["dtype"]].itemsize
    width = config["hidden_size"] if is_gemma(config) else config["width"]
    vocab, layers = vocabulary(config), layer_sizes(config)
    held, nbytes, flops = contexts(case), 0.0, 0.0
    lengths = prompt_lengths(case)
    for portions in steps_of(case):
        spans = [(n + 1, n + 2) for n in held] + [(a, e) for _, a, e in portions]      # tokens before, and with, the step's
        rows = sum(e - a for a, e in spans)
        logit_rows = len(held) + sum(e == lengths[i] for i, _, e in portions)
        nbytes += vocab * width * size * (logit_rows > 0) + logit_rows * vocab * 4 + rows * width * size
        flops += 2.0 * logit_rows * vocab * width
        for s in layers:
            reached = s["experts"] * (1.0 - (1.0 - s["top"] / s["experts"]) ** rows) if s["experts"] else 0.0
            nbytes += (s["dense"] + reached * s["expert"]) * size
            flops += 2.0 * rows * (s["dense"] + s["top"] * s["expert"])
            for a, e in spans:
                seen = a if s["span"] is None else min(a, s["span"])
                nbytes += s["cached"] * size * (seen + (e - a) * s["owns"])
                flops += 2.0 * s["heads"] * ((e - a) * seen + (e - a) * (e - a + 1) / 2.0) + 6.0 * (e - a) * s["state"]
                nbytes += 8.0 * s["state"]
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case["dtype"] == "float32":
        return {"rel": 1.2e-5, "max": 2e-4}                   # 2.9e-6 off the result in 64 bits
    if case["shape"] == "duvozen-2b":
        # 0.2% from rounding; a token whose third and fourth expert score alike may use the other: 2 to 5% of its row
        return {"rel": 0.02, "max": 0.5}
    # 18 layers of bfloat16 activations: 1.1 to 1.6% off the result in 64 bits, and the same prompt whole and in two
    # portions differs by 0.8 to 1.7%
    return {"rel": 0.03, "max": 0.3}


# ---- the same in 64 bits -----------------------------------------------------------------------------------

class Plain64:
    """A model's layers over one whole sequence at a time in float64, no cache; weights are drawn when a
    layer needs them.  `x`: a list of streams [tokens, width], one a sequence."""

    def __init__(self, config, dtype):
        self.config, self.dtype, self.gemma, self.family = config, dtype, is_gemma(config), family(config)
        self.eps = config["rms_norm_eps"] if self.gemma else config["norm"]["eps"]
        self.width = config["hidden_size"] if self.gemma else config["width"]
        self.kept = {}

    def w(self, name, *size):
        return weight(name, size, self.family).double()

    def rms(self, x, w):
        return x / torch.sqrt(x.square().mean(-1, keepdim=True) + self.eps) * w

    def layer_norm(self, x, name):
        d = x - x.mean(-1, keepdim=True)
        return d / torch.sqrt(d.square().mean(-1, keepdim=True) + self.eps) * self.w(name, x.shape[-1])

    def attend(self, q, k, v, scale, sink=None, span=None):
        """q [t, heads, d], k and v [t, key heads, d]: causal, inside chunks of `span` positions."""
        t, heads, rep = q.shape[0], q.shape[1], q.shape[1] // k.shape[1]
        out = torch.empty(t, heads, v.shape[2], dtype=q.dtype, device=q.device)
        at = torch.arange(t, device=q.device)
        for h in range(heads):
            kh, vh = k[:, h // rep].T.contiguous(), v[:, h // rep].contiguous()
            for a in range(0, t, 2048):
                rows = at[a:a + 2048, None]
                seen = at[None, :] <= rows
                if span:
                    seen &= (at[None, :] // span) == (rows // span)
                s = (q[a:a + 2048, h].contiguous() @ kh * scale).masked_fill(~seen, float("-inf"))
                if sink is not None:
                    s = torch.cat([s, sink[h].expand(s.shape[0], 1)], 1)
                out[a:a + 2048, h] = torch.softmax(s, -1)[:, :t] @ vh
        return out.reshape(t, -1)

    def turn(self, x, dims, freq, pairs, magnitude=1.0):
        """x [t, heads, d]: the first `dims` elements turned by position * freq."""
        angle = torch.arange(x.shape[0], device=x.device, dtype=x.dtype)[:, None] * freq[None, :]
        cos, sin = (angle.cos() * magnitude)[:, None], (angle.sin() * magnitude)[:, None]
        y, half = x.clone(), dims // 2
        a, b = (slice(0, half), slice(half, dims)) if pairs == "half" else (slice(0, dims, 2), slice(1, dims, 2))
        y[..., a], y[..., b] = x[..., a] * cos - x[..., b] * sin, x[..., b] * cos + x[..., a] * sin
        return y

    def freq(self, dims, base):
        return float(base) ** (-torch.arange(0, dims, 2, device="cuda", dtype=torch.float64) / dims)

    def gated(self, h, gate, up, down, act):
        out = torch.empty(h.shape[0], down.shape[0], dtype=h.dtype, device=h.device)
        for a in range(0, h.shape[0], 8192):
            r = h[a:a + 8192]
            out[a:a + 8192] = (act(r @ gate.T) * (r @ up.T)) @ down.T
        return out

    def dense(self, p, ff, act, names=("gate", "up", "down")):
        w = [self.w(p + n, *((self.width, ff) if n.startswith("down") else (ff, self.width))) for n in names]
        return lambda h: self.gated(h, *w, act)

    def logits(self, sequences):
        """The last position's logits of each sequence."""
        c, table = self.config, "model.embed_tokens.weight" if self.gemma else "embed"
        vocab = vocabulary(c)
        scale = c["hidden_size"] ** 0.5 if self.gemma else (c.get("embedding") or {}).get("scale", 1.0)
        if self.gemma:
            scale = float(torch.tensor(scale).to(self.dtype))            # the factor is one of the model's dtype
        emb = weight(table, (vocab, self.width), self.family)
        ids = [torch.tensor(s, device="cuda") for s in sequences]
        x = [emb[i].double() * scale for i in ids]
        del emb
        run = self.gemma_layer if self.gemma else getattr(self, c["architecture"].lower() + "_layer")
        for layer in range(c["num_hidden_layers"] if self.gemma else len(c["layers"])):
            run(layer, x, ids)
        last = torch.stack([s[-1] for s in x])
        if self.gemma:
            last = self.rms(last, 1.0 + self.w("model.norm.weight", self.width))
        else:
            last = self.layer_norm(last, "final.norm")
        head = weight("head" if c.get("architecture") == "Duvozen" else table, (vocab, self.width), self.family)
        return torch.cat([last @ head[a:a + 32768].double().T for a in range(0, vocab, 32768)], 1)

    def gemma_layer(self, i, x, ids):
        c, w, p = self.config, self.width, f"model.layers.{i}."
        heads, kv, d = c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"]
        q, k, v = (self.w(p + f"self_attn.{n}_proj.weight", m * d, w) for n, m in (("q", heads), ("k", kv), ("v", kv)))
        o = self.w(p + "self_attn.o_proj.weight", w, heads * d)
        n1, n2 = (1.0 + self.w(p + n + ".weight", w) for n in ("input_layernorm", "post_attention_layernorm"))
        mlp = self.dense(p + "mlp.", c["intermediate_size"], lambda z: torch.nn.functional.gelu(z, approximate="tanh"),
                         ("gate_proj.weight", "up_proj.weight", "down_proj.weight"))
        freq = self.freq(d, c["rope_theta"])
        for j, s in enumerate(x):
            h, t = self.rms(s, n1), s.shape[0]
            qs, ks = (self.turn((h @ m.T).view(t, -1, d), d, freq, "half") for m in (q, k))
            s = s + self.attend(qs, ks, (h @ v.T).view(t, kv, d), d ** -0.5) @ o.T
            x[j] = s + mlp(self.rms(s, n2))

    def tokuvik_layer(self, i, x, ids):
        layer, w, p = self.config["layers"][i], self.width, f"l{i}."
        m, dim = layer["mixer"], self.config["token_side"]["dim"]
        mixer = getattr(self, "tokuvik_" + layer["type"])(i, p + "mix.", m)
        mlp = self.dense(p + "mlp.", layer["mlp"]["ff"], torch.nn.functional.silu)
        gate, proj, norm = self.w(p + "side.gate", dim, w), self.w(p + "side.proj", w, dim), self.w(p + "side.norm", w)
        layers = len(self.config["layers"])
        side = weight("side.embed", (self.config["vocab"], layers * dim), self.family)[:, i * dim:(i + 1) * dim]
        for j, s in enumerate(x):
            s = s + self.layer_norm(mixer(self.layer_norm(s, p + "norm1"), j), p + "norm1b")
            s = s + self.layer_norm(mlp(self.layer_norm(s, p + "norm2")), p + "norm2b")
            g = torch.nn.functional.gelu(s @ gate.T, approximate="tanh") * side[ids[j]].double()
            x[j] = s + self.rms(g @ proj.T, norm)

    def tokuvik_attention(self, i, p, m):
        w, heads, kv, d = self.width, m["heads"], m["kv_heads"], m["dim"]
        q, qn, g = self.w(p + "q", heads * d, w), self.w(p + "q.norm", heads * d), self.w(p + "g", heads, w)
        o, own = self.w(p + "o", w, heads * d), "kv_from" not in m
        if own:
            k, kn, v = self.w(p + "k", kv * d, w), self.w(p + "k.norm", kv * d), self.w(p + "v", kv * d, w)

        def mixer(h, j):
            t = h.shape[0]
            if own:
                self.kept[i, j] = (self.rms(h @ k.T, kn).view(t, kv, d), (h @ v.T).view(t, kv, d))
            ks, vs = self.kept[m.get("kv_from", i), j]
            y = self.attend(self.rms(h @ q.T, qn).view(t, heads, d), ks, vs, m["scale"], span=m["mask"]["size"])
            return (y.view(t, heads, d) * torch.sigmoid(h @ g.T)[:, :, None]).reshape(t, -1) @ o.T
        return mixer

    def tokuvik_latent_attention(self, i, p, m):
        w, heads, d, qr, r = self.width, m["heads"], m["dim"], m["q_rank"], m["kv_rank"]
        dq, dqn, uq = self.w(p + "dq", qr, w), self.w(p + "dq.norm", qr), self.w(p + "uq", heads * d, qr)
        dkv, dkvn = self.w(p + "dkv", r, w), self.w(p + "dkv.norm", r)
        uk, uv = self.w(p + "uk", heads * d, r), self.w(p + "uv", heads * d, r)
        o, g, sink = self.w(p + "o", w, heads * d), self.w(p + "g", heads * d, w), self.w(p + "sink", heads)

        def mixer(h, j):
            t = h.shape[0]
            q, c = self.rms(h @ dq.T, dqn) @ uq.T, self.rms(h @ dkv.T, dkvn)
            y = self.attend(*(z.view(t, heads, d) for z in (q, c @ uk.T, c @ uv.T)), m["scale"], sink)
            return (y * torch.sigmoid(h @ g.T)) @ o.T
        return mixer

    def tokuvik_mamba2(self, i, p, m):
        w, heads, d, n, groups = self.width, m["heads"], m["vdim"], m["state"], m["groups"]
        inner, rep = heads * d, heads // groups
        rows = self.w(p + "in", 2 * inner + 2 * groups * n + heads, w)
        conv, bias = self.w(p + "conv", inner + 2 * groups * n, m["conv"]), self.w(p + "conv.b", inner + 2 * groups * n)
        dtb, rate = self.w(p + "dt_bias", heads), self.w(p + "A_log", heads).exp()
        skip, norm, o = self.w(p + "D", heads), self.w(p + "norm", inner), self.w(p + "o", w, inner)

        def mixer(h, j):
            t = h.shape[0]
            z, u, dt = (h @ rows.T).split([inner, inner + 2 * groups * n, heads], 1)
            u = torch.nn.functional.pad(u, (0, 0, m["conv"] - 1, 0))
            u = torch.nn.functional.silu(bias + sum(u[k:k + t] * conv[:, k] for k in range(m["conv"])))
            v, b, c = u.split([inner, groups * n, groups * n], 1)
            v = v.reshape(t, heads, d)
            b, c = (y.reshape(t, groups, n).repeat_interleave(rep, 1) for y in (b, c))
            dt = torch.nn.functional.softplus(dt + dtb)
            y = self.recurrence(torch.exp(-rate * dt)[:, :, None], b * dt[:, :, None], v, c) + skip[:, None] * v
            y = (y.reshape(t, inner) * torch.nn.functional.silu(z)).view(t, m["norm_groups"], -1)
            return (self.rms(y, 1.0).reshape(t, inner) * norm) @ o.T
        return mixer

    @staticmethod
    def recurrence(decay, k, v, q):
        """S = decay S + k v^T, y = S^T q, token by token; decay and k, q [t, heads, n] (or 1), v [t, heads, d]."""
        s = torch.zeros(k.shape[1], k.shape[2], v.shape[2], dtype=k.dtype, device=k.device)
        out = torch.empty_like(v)
        for i in range(k.shape[0]):
            s.mul_(decay[i][:, :, None]).baddbmm_(k[i][:, :, None], v[i][:, None])
            out[i] = torch.bmm(q[i][:, None], s)[:, 0]
        return out

    def convolved(self, x, taps):
        t, k = x.shape[0], taps.shape[1]
        u = torch.nn.functional.pad(x, (0, 0, k - 1, 0))
        return x + sum(u[j:j + t] * taps[:, j] for j in range(k))

    def duvozen_layer(self, i, x, ids):
        layer, w, p, taps = self.config["layers"][i], self.width, f"l{i}.", self.config["canon"]["taps"]
        mixer = getattr(self, "duvozen_" + layer["type"])(p + "mix.", layer["mixer"])
        f = layer["mlp"]
        mlp = self.experts(p + "mlp.", f) if f["kind"] == "moe" else self.dense(
            p + "mlp.", f["ff"], lambda z: torch.nn.functional.gelu(z, approximate="tanh"))
        c1, c2 = self.w(p + "canon1", w, taps), self.w(p + "canon2", w, taps)
        for j, s in enumerate(x):
            s = s + self.layer_norm(mixer(self.convolved(s, c1)), p + "norm1")
            x[j] = s + self.layer_norm(mlp(self.convolved(s, c2)), p + "norm2")

    def experts(self, p, f):
        silu, count = torch.nn.functional.silu, f["router"]["experts"]
        router, shared = self.w(p + "router", count, self.width), self.dense(p + "shared.", f["shared"]["ff"], silu)
        each = [self.dense(p + f"e{e}.", f["expert"]["ff"], silu) for e in range(count)]

        def mlp(h):
            top = torch.sigmoid(h @ router.T).topk(f["router"]["top"], -1)
            out = shared(h)
            for e in range(count):
                row, at = (top.indices == e).nonzero(as_tuple=True)
                out.index_add_(0, row, each[e](h[row] * top.values[row, at][:, None]))
            return out
        return mlp

    def duvozen_attention(self, p, m):
        w, heads, kv, d = self.width, m["heads"], m["kv_heads"], m["dim"]
        q, k, v = (self.w(p + n, c * d, w) for n, c in (("q", heads), ("k", kv), ("v", kv)))
        g, o, sink = self.w(p + "g", heads * d, w), self.w(p + "o", w, heads * d), self.w(p + "sink", heads)
        qn, kn, freq = self.w(p + "q.norm", d), self.w(p + "k.norm", d), self.freq(m["rot"]["dims"], m["rot"]["base"])

        def mixer(h):
            t = h.shape[0]
            qs, ks = (self.turn(self.rms((h @ a.T).view(t, -1, d), n), m["rot"]["dims"], freq, "half")
                      for a, n in ((q, qn), (k, kn)))
            return (self.attend(qs, ks, (h @ v.T).view(t, kv, d), m["scale"], sink) * torch.sigmoid(h @ g.T)) @ o.T
        return mixer

    def duvozen_latent_attention(self, p, m):
        w, heads, d, r, rot, turned = self.width, m["heads"], m["dim"], m["kv_rank"], m["rot_dim"], m["rot"]
        q, dkv, o = self.w(p + "q", heads * (d + rot), w), self.w(p + "dkv", r + rot, w), self.w(p + "o", w, heads * d)
        dkvn, uk, uv = self.w(p + "dkv.norm", r), self.w(p + "uk", heads * d, r), self.w(p + "uv", heads * d, r)
        s, dims = turned["scaling"], turned["dims"]
        # frequencies between the plain ones and the ones divided by the factor, by the turns made in `original`
        lo, hi = (dims * math.log(s["original"] / (2.0 * math.pi * n)) / (2.0 * math.log(turned["base"]))
                  for n in (s["fast"], s["slow"]))
        lo, hi = max(math.floor(lo), 0), min(math.ceil(hi), dims - 1)
        ramp = ((torch.arange(dims // 2, device="cuda", dtype=torch.float64) - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
        freq, magnitude = self.freq(dims, turned["base"]), 0.1 * math.log(s["factor"]) + 1.0
        freq = freq / s["factor"] * ramp + freq * (1.0 - ramp)

        def mixer(h):
            t = h.shape[0]
            qs, down = (h @ q.T).view(t, heads, d + rot), h @ dkv.T
            c = self.rms(down[:, :r], dkvn)
            qt, kt = (self.turn(z, dims, freq, "neighbours", magnitude) for z in (qs[..., d:], down[:, None, r:]))
            ks = torch.cat([(c @ uk.T).view(t, heads, d), kt.expand(t, heads, rot)], 2)
            y = self.attend(torch.cat([qs[..., :d], qt], 2), ks, (c @ uv.T).view(t, heads, d), m["scale"])
            return y @ o.T
        return mixer

    def duvozen_hgrn2(self, p, m):
        w, heads, d, v = self.width, m["heads"], m["dim"], m["vdim"]
        q, f, values, o = self.w(p + "q", heads * d, w), self.w(p + "f", heads * d, w), self.w(p + "v", heads * v, w), \
            self.w(p + "o", w, heads * v)
        bias, lower, norm = self.w(p + "f.b", heads * d), self.w(p + "lower", heads * d), self.w(p + "norm", v)

        def mixer(h):
            t = h.shape[0]
            forget = (lower + (1.0 - lower) * torch.sigmoid(h @ f.T + bias)).view(t, heads, d)
            y = self.recurrence(forget, 1.0 - forget, (h @ values.T).view(t, heads, v),
                                torch.nn.functional.silu(h @ q.T).view(t, heads, d))
            return self.rms(y, norm).reshape(t, -1) @ o.T
        return mixer


@torch.inference_mode()
def exact(case, seed):
    decoding, prompts = token_ids(case, seed)
    held, steps = contexts(case), len(steps_of(case))
    sequences = [ids[:n + 1 + steps] for ids, n in zip(decoding, held)] + prompts     # one more: the step of `fill`
    total, config = sum(len(s) for s in sequences), shape_config(case["shape"])
    layers = layer_sizes(config)
    per_token = 2.0 * sum(s["dense"] + s["top"] * s["expert"] for s in layers)
    # float64 products at some 30 TFLOP/s, and five launches a token and recurrent layer
    if total * per_token / 3e13 + 6e-5 * total * sum(s["state"] > 0 for s in layers) > 12.0:
        return None
    return Plain64(config, DTYPES[case["dtype"]]).logits(sequences)
