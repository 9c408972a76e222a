"""The work that programs using this library have it do, as cases that can be timed and checked.

A case is one model (a preset, whole or its first layers), a precision, a batch of sequences and what is done
with them through `Engine.step`:

* `prompt`: new requests; their prompts in one step, the logits of every prompt's last token (`want` "last") or of
  the second half of its tokens (`want` "half": continuations scored under the model); the slots are given back.
* `decode`: requests under way; `steps` single-token steps of the whole batch, the logits of all of them.  The
  contexts grow from pass to pass as a served request's do; where the engine's room ends the requests end and others
  of the first lengths take their place.
* `turn`: whole short requests: slots, prompts, `steps` single-token steps, slots given back.

Sequences of a batch have lengths spread evenly from `lo` to `hi`, the longest first (the order of the generation
loop).  Weights are the library's random ones (matrices N(0, 0.02), norm weights around 1), token ids uniform.
"""
import math

import numpy as np
import torch

import braidinfer_amd as B
from braidinfer_amd.config import spec_of
from braidinfer_amd.engine import DecoderModel
from braidinfer_amd.weights import random_tensor

STD, JITTER = 0.02, 0.2
GROWTH = 1024                 # tokens a decode case's sequences may grow by before they are replaced


def _case(name, model, layers, task, batch, lo, hi, steps=0, want="last", dtype="bfloat16"):
    return {"name": name, "model": model, "layers": layers, "task": task, "batch": batch, "lo": lo, "hi": hi,
            "steps": steps, "want": want, "dtype": dtype}


def listed():
    return [
        # one user in a chat, the answer being written: the smallest step, launches and latency count
        _case("mistral decode 1", "mistral-7b-v0.3", 8, "decode", 1, 701, 701, steps=4),
        # the headline workload of bench.py: a small batch of unequal contexts
        _case("mistral decode 8", "mistral-7b-v0.3", 8, "decode", 8, 128, 2048, steps=4),
        # a server's full batch: weights and caches weigh about the same
        _case("mistral decode 64", "mistral-7b-v0.3", 8, "decode", 64, 128, 2048, steps=4),
        # a chat message of a few lines: the time to the first token of a short prompt
        _case("mistral prompt short", "mistral-7b-v0.3", 8, "prompt", 1, 67, 67),
        # several requests of unequal length taken in together
        _case("mistral prompts ragged", "mistral-7b-v0.3", 8, "prompt", 5, 93, 1357),
        # a document: a long prompt through window attention, the largest case
        _case("mistral prompt long", "mistral-7b-v0.1", 8, "prompt", 1, 7001, 7001),
        # the 32-bit path, as used to check a checkpoint: short requests from start to end
        _case("mistral float32 turn", "mistral-7b-v0.3", 8, "turn", 3, 29, 157, steps=6, dtype="float32"),
        # window attention with pooled blocks between gated recurrences: prompts of some thousand tokens
        _case("kesitar prompts", "kesitar-7b", 8, "prompt", 2, 1501, 3517),
        # routed experts behind every half: a text scored under the model
        _case("sidirax score", "sidirax-7b", 8, "prompt", 1, 1801, 1801, want="half"),
        # the same model answering a handful of users
        _case("sidirax decode 6", "sidirax-7b", 8, "decode", 6, 211, 1203, steps=12),
        # delta rule beside attention, lightning attention and experts: unequal texts scored
        _case("zivovik score", "zivovik-7b", 2, "prompt", 3, 301, 1307, want="half"),
        # the same model serving a batch
        _case("zivovik decode 40", "zivovik-7b", 2, "decode", 40, 65, 901, steps=4),
    ]


MODELS = [("mistral-7b-v0.3", 8, 3), ("mistral-7b-v0.1", 8, 1), ("kesitar-7b", 8, 2), ("kesitar-1b", 16, 1),
          ("sidirax-7b", 8, 2), ("sidirax-1b", 4, 1), ("zivovik-7b", 2, 2), ("zivovik-1b", 2, 1)]


def draw(rng):
    """Another case of the same ranges: a model, what is done with it, and sizes spread over their logarithms."""
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.1:
        lo, hi = sorted((log(3, 160), log(3, 160)))
        case = _case("", "mistral-7b-v0.3", 4, "turn", log(1, 4), lo, hi, steps=rng.randint(2, 6), dtype="float32")
        del case["name"]
        return case
    model, layers, _ = rng.choices(MODELS, weights=[m[2] for m in MODELS])[0]
    routed = model.startswith(("sidirax", "zivovik"))
    task = rng.choices(("prompt", "decode", "turn"), weights=(4, 4, 1))[0]
    if task == "prompt":
        batch = log(1, 8)
        total = max(24 * batch, log(64 if routed else 24, 7000))
        want = "half" if routed else "last"
        mean = total // batch
        half = 0 if batch == 1 else rng.randint(0, mean - mean // 4)
        case = _case("", model, layers, "prompt", batch, max(2, mean - half), mean + half, want=want)
    elif task == "decode":
        lo, hi = sorted((log(24, 2048), log(24, 2048)))
        batch = log(1, min(64, 65536 // hi))
        case = _case("", model, layers, "decode", batch, lo, hi, steps=max(4, -(-48 // batch)) if routed else 4)
    else:
        batch = log(1, 16)
        lo, hi = sorted((log(5, 200), log(5, 200)))
        case = _case("", model, layers, "turn", batch, lo, hi, steps=max(rng.randint(4, 12), -(-48 // batch) if routed else 0))
    del case["name"]
    return case


# ------------------------------------------------------------------ a case's inputs --
def _config(case):
    if case["model"].startswith("mistral"):
        return B.preset(case["model"], num_hidden_layers=case["layers"])
    full = B.any_preset(case["model"])
    once = {"loop": None} if getattr(full, "loop", None) else {}       # passes over a layer are the same work again
    return B.any_preset(case["model"], layers=[dict(layer) for layer in full.layers[:case["layers"]]], **once)


def _lengths(case):
    n, lo, hi = case["batch"], case["lo"], case["hi"]
    return [hi - (hi - lo) * i // max(1, n - 1) for i in range(n)]


def _vocab(config):
    return config.vocab_size if hasattr(config, "vocab_size") else config.vocab


def _tokens(case, config, seed):
    """(the prompts, the token that every sequence is fed in each of the steps that follow)."""
    rng = np.random.default_rng(seed)
    prompts = [rng.integers(0, _vocab(config), n).tolist() for n in _lengths(case)]
    fed = rng.integers(0, _vocab(config), (max(1, case["steps"]), case["batch"])).tolist()
    return prompts, fed


class _State:
    pass


def _admit(s):
    """Slots for the batch, and its prompts in steps of at most 16,384 tokens."""
    s.slots = [s.engine.alloc_slot() for _ in s.prompts]
    i = 0
    while i < len(s.slots):
        j, total = i, 0
        while j < len(s.slots) and (j == i or total + len(s.prompts[j]) <= 16384):
            total += len(s.prompts[j])
            j += 1
        s.engine.step([B.StepEntry(s.slots[b], s.prompts[b]) for b in range(i, j)])
        i = j


def prepare(case, seed):
    s = _State()
    config = _config(case)
    s.task, s.steps = case["task"], case["steps"]
    s.prompts, s.fed = _tokens(case, config, seed)
    grows = GROWTH + s.steps if s.task == "decode" else s.steps
    s.most = max(len(p) for p in s.prompts) + grows
    room = sum(-(-(len(p) + grows) // 64) * 64 for p in s.prompts)
    s.engine = B.Engine.random(config, seed=seed, dtype=case["dtype"], max_tokens=room, max_seq_len=s.most,
                               n_slots=case["batch"], std=STD, vector_jitter=JITTER)
    s.want = [list(range(len(p) // 2, len(p))) if case["want"] == "half" else [len(p) - 1] for p in s.prompts]
    if s.task == "decode":
        _admit(s)
    return s


def run(s):
    engine, out = s.engine, []
    if s.task == "decode":
        if engine.length(s.slots[0]) + s.steps > s.most:      # the room ends: the requests do, and others come
            for slot in s.slots:
                engine.free_slot(slot)
            _admit(s)
        for t in range(s.steps):
            out.append(engine.step([B.StepEntry(slot, [token], [0]) for slot, token in zip(s.slots, s.fed[t])]))
        return torch.cat(out)
    slots = [engine.alloc_slot() for _ in s.prompts]
    out.append(engine.step([B.StepEntry(slot, p, want) for slot, p, want in zip(slots, s.prompts, s.want)]))
    for t in range(s.steps):
        out.append(engine.step([B.StepEntry(slot, [token], [0]) for slot, token in zip(slots, s.fed[t])]))
    for slot in slots:
        engine.free_slot(slot)
    return torch.cat(out) if s.steps else out[0]


# ------------------------------------------------------------------ what it costs ----
def _model_layers(case, config):
    """[(layer, how often a pass runs it)] of a configuration with a list of layers."""
    order = config.run_order() if hasattr(config, "run_order") else [(i, False) for i in range(len(config.layers))]
    times = {}
    for i, _ in order:
        times[i] = times.get(i, 0) + 1
    return [(config.layers[i], i, times[i]) for i in sorted(times)]


def _sizes(case, config):
    """Per layer: (dense weights, experts, experts a token takes, weights of an expert, key and value numbers a token keeps,
    what a query reads per kept token in operations, window, numbers of recurrent state, operations on it per token, runs)."""
    out = []
    if case["model"].startswith("mistral"):
        c = config
        H, d, nq, nkv = c.hidden_size, c.head_dim, c.num_attention_heads, c.num_key_value_heads
        w = (nq + 2 * nkv) * d * H + H * nq * d + 3 * H * c.intermediate_size
        return [(w, 0, 0, 0, 2 * nkv * d, 4 * nq * d, c.sliding_window, 0, 0, 1)] * c.num_hidden_layers
    W, E = config.width, {"experts": 0, "top": 0}
    for layer, i, runs in _model_layers(case, config):
        w = sum(int(np.prod(shape)) for name, shape, _, _ in _table(config)
                if name.startswith(f"l{i}.") and ".e" not in name and not name.endswith("router"))
        m, mlp = layer["mixer"], layer.get("mlp") or {}
        r = mlp.get("router") or E
        expert = 3 * W * mlp["expert"]["ff"] if r["experts"] else 0
        kept = reads = state = ops = 0
        window = None
        kind = layer["type"]
        if kind == "parallel":
            state = m["right"]["heads"] * m["right"]["dim"] * m["right"]["vdim"]
            ops, m = 7 * state, m["left"]
        if kind in ("attention", "parallel"):
            g = m.get("kv_heads", m["heads"])
            kept, reads = g * (m["dim"] + m["vdim"]), 2 * m["heads"] * (m["dim"] + m["vdim"])
            window = (m.get("mask") or {}).get("size")
        elif kind == "latent_attention":
            kept = m["kv_rank"] + m["rot_dim"]
            reads = 2 * m["heads"] * (2 * m["kv_rank"] + m["rot_dim"])
        else:
            state = m["heads"] * m["dim"] * m.get("vdim", m["dim"])
            ops = 5 * state
        out.append((w, r["experts"], r["top"], expert, kept, reads, window, state, ops, runs))
    return out


def work(case):
    """Every weight a step needs read once, what the caches and states hold read and written once, the embedding's rows
    read, the logits written; products, attention over what a query sees and recurrences counted as operations."""
    config = _config(case)
    size = 2 if case["dtype"] == "bfloat16" else 4
    V = _vocab(config)
    H = config.hidden_size if hasattr(config, "hidden_size") else config.width
    lengths = _lengths(case)
    single = [[(n + t, 1, 1) for n in lengths] for t in range(case["steps"])]
    wants = [n - n // 2 if case["want"] == "half" else 1 for n in lengths]
    steps = single if case["task"] == "decode" else [[(0, n, k) for n, k in zip(lengths, wants)]] + single
    nbytes = flops = 0
    for step in steps:
        T, wanted = sum(new for _, new, _ in step), sum(k for _, _, k in step)
        nbytes += V * H * size + T * H * size + wanted * V * 4
        flops += 2 * V * H * wanted
        for w, experts, top, expert, kept, reads, window, state, ops, runs in _sizes(case, config):
            nbytes += w * size
            flops += 2 * T * (w + top * expert) * runs + T * ops * runs
            if experts:
                nbytes += experts * (1.0 - (1.0 - top / experts) ** T) * expert * size
            for held, new, _ in step:
                total = held + new
                seen = [min(p + 1, window or total) for p in (held, total - 1)]
                nbytes += runs * (size * kept * (new + min(held, window or held)) + 4 * state * (2 if held else 1))
                if window is None or total <= window:
                    pairs = new * (seen[0] + seen[1]) / 2
                else:
                    ramp = max(0, min(new, window - held))
                    pairs = ramp * (held + 1 + held + ramp) / 2 + (new - ramp) * window
                flops += runs * reads * pairs
    return {"bytes": float(nbytes), "flops": float(flops)}


def tolerance(case):
    # What a prompt's logits differ by when the same tokens run alone, among other prompts or one by one (other kernels, other
    # orders of the sums): float32 1e-5; bfloat16, whose activations are rounded between the kernels, 0.008 (Kesitar), 0.014
    # (Mistral) and, where a near tie sends a token to another expert, 0.01 to 0.02 with single values up to 0.4.
    if case["dtype"] == "float32":
        return {"rel": 5e-5, "max": 1e-3}
    if case["model"].startswith("kesitar"):
        return {"rel": 0.025, "max": 0.15}
    return {"rel": 0.03, "max": 0.25 if case["model"].startswith("mistral") else 0.9}


# ------------------------------------------------------------------ in 64 bits -------
_tables = {}


def _table(config):
    """[(name, shape, index, the tensor's declaration)] of a configuration's weights, in the order of their names."""
    key = repr(config.to_dict())
    if key not in _tables:
        _tables.clear()
        _tables[key] = [(t.name, t.shape, i, t) for i, t in enumerate(DecoderModel(spec_of(config)).weight_specs())]
    return _tables[key]


class _Weights:
    """The random weights of a configuration and a seed, by name, as float64 on the GPU: inputs, the same values that
    `Engine.random` takes."""

    def __init__(self, config, seed):
        self.by_name = {name: (i, spec) for name, _, i, spec in _table(config)}
        self.seed = seed

    def __contains__(self, name):
        return name in self.by_name

    def __getitem__(self, name):
        i, spec = self.by_name[name]
        return random_tensor(spec, i, self.seed, "cuda", torch.bfloat16, STD, JITTER).to(torch.float64)


def _rms(x, eps, weight=None):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    return y if weight is None else y * weight


def _layer_norm(x, weight, eps):
    return torch.nn.functional.layer_norm(x, x.shape[-1:], weight, None, eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _turn(x, freq, adjacent, magnitude=1.0):
    """Rotary positions 0, 1, .. on the first 2 len(freq) elements of x [T, heads, d]."""
    n = len(freq)
    angle = torch.arange(x.shape[0], dtype=torch.float64, device=x.device)[:, None, None] * freq
    c, s = torch.cos(angle) * magnitude, torch.sin(angle) * magnitude
    y = x.clone()
    a, b = (slice(0, 2 * n, 2), slice(1, 2 * n, 2)) if adjacent else (slice(0, n), slice(n, 2 * n))
    y[..., a] = x[..., a] * c - x[..., b] * s
    y[..., b] = x[..., b] * c + x[..., a] * s
    return y


def _frequencies(dims, base, scaling=None):
    """Frequency of each pair, and the factor on cos and sin; {factor, original, fast, slow} stretches slow pairs."""
    i = torch.arange(dims // 2, dtype=torch.float64, device="cuda")
    f = base ** (-2.0 * i / dims)
    if not scaling:
        return f, 1.0

    def pair_of(turns):
        return dims * math.log(scaling["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(base))
    lo, hi = max(math.floor(pair_of(scaling["fast"])), 0), min(math.ceil(pair_of(scaling["slow"])), dims - 1)
    ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
    return f / scaling["factor"] * ramp + f * (1.0 - ramp), 0.1 * math.log(scaling["factor"]) + 1.0


def _attend(q, k, v, scale, window=None, pool=0, sink=None):
    """q [T, H, d], k [T, G, d], v [T, G, e]: query i sees the keys of the last `window` positions and, with `pool`, the
    mean key and value of every block of `pool` positions that lies wholly before them; `sink` [H] joins the softmax."""
    T, H, _ = q.shape
    G, e = k.shape[1], v.shape[2]
    blocks = T // pool if pool else 0
    if blocks:
        k = torch.cat([k[:blocks * pool].reshape(blocks, pool, G, -1).mean(1), k])
        v = torch.cat([v[:blocks * pool].reshape(blocks, pool, G, -1).mean(1), v])
    ends = torch.arange(blocks, device=q.device) * pool + pool - 1
    j = torch.arange(T, device=q.device)
    keys, values = k.permute(1, 2, 0).contiguous(), v.permute(1, 0, 2).contiguous()
    out = torch.empty(T, H, e, dtype=q.dtype, device=q.device)
    step = max(1, (1 << 28) // (H * len(k)))
    for a in range(0, T, step):
        i = torch.arange(a, min(T, a + step), device=q.device)[:, None]
        seen = (j <= i) if window is None else (j <= i) & (i - j < window)
        if blocks:
            seen = torch.cat([ends <= i - window, seen], 1)
        qs = q[a:a + step].reshape(len(i), G, H // G, -1).permute(1, 2, 0, 3).reshape(G, -1, q.shape[2])
        s = torch.bmm(qs, keys).reshape(G, H // G, len(i), -1) * scale
        s = s.masked_fill(~seen, -math.inf)
        if sink is not None:
            s = torch.cat([sink.reshape(G, H // G, 1, 1).expand(-1, -1, len(i), 1), s], -1)
        p = torch.softmax(s, -1)
        if sink is not None:
            p = p[..., 1:].contiguous()
        o = torch.bmm(p.reshape(G, -1, p.shape[-1]), values).reshape(G, H // G, len(i), e)
        out[a:a + step] = o.permute(2, 0, 1, 3).reshape(len(i), H, e)
    return out


def _each(seqs, f, *rows):
    """f over every sequence's rows of packed tensors."""
    return torch.cat([f(*(r[a:b] for r in rows)) for a, b in seqs])


def _walk(seqs, like, state, token):
    """A recurrence walked over all sequences at once: `token(S [n, ..], rows [n])` -> (S, o) for the n sequences that are
    still going (the longest come first); returns the outputs in packed order."""
    out = torch.empty_like(like)
    starts = torch.tensor([a for a, _ in seqs], device=like.device)
    lengths = [b - a for a, b in seqs]
    n = len(seqs)
    for t in range(lengths[0]):
        while lengths[n - 1] <= t:
            n -= 1
        state, out[starts[:n] + t] = token(state[:n], starts[:n] + t)
    return out


def _experts(h, w, p, mlp, over_all):
    E, top = mlp["router"]["experts"], mlp["router"]["top"]
    z = h @ w[p + "router"].T
    if p + "router.b" in w:
        z = z + w[p + "router.b"]
    z, chosen = torch.sort(z, dim=1, descending=True, stable=True)
    share = torch.softmax(z, 1)[:, :top] if over_all else torch.softmax(z[:, :top], 1)
    share = share / (share.sum(1, keepdim=True) + (1e-20 if over_all else 0.0))
    out = torch.zeros_like(h)
    for e in range(E):
        t, k = (chosen[:, :top] == e).nonzero(as_tuple=True)
        if len(t):
            q, x = f"{p}e{e}.", h[t]
            out[t] += share[t, k, None] * ((_silu(x @ w[q + "gate"].T) * (x @ w[q + "up"].T)) @ w[q + "down"].T)
    return out


def _mistral(c, w, tokens, seqs):
    eps, d, H, G = c.rms_norm_eps, c.head_dim, c.num_attention_heads, c.num_key_value_heads
    x = w["model.embed_tokens.weight"][tokens]
    freq, _ = _frequencies(d, c.rope_theta)
    for i in range(c.num_hidden_layers):
        p = f"model.layers.{i}."
        h = _rms(x, eps, w[p + "input_layernorm.weight"])
        q, k, v = ((h @ w[f"{p}self_attn.{n}_proj.weight"].T).reshape(len(x), -1, d) for n in "qkv")
        q, k = (_each(seqs, lambda r: _turn(r, freq, False), r) for r in (q, k))
        o = _each(seqs, lambda q, k, v: _attend(q, k, v, d ** -0.5, c.sliding_window), q, k, v)
        x = x + o.reshape(len(x), H * d) @ w[p + "self_attn.o_proj.weight"].T
        h = _rms(x, eps, w[p + "post_attention_layernorm.weight"])
        h = _silu(h @ w[p + "mlp.gate_proj.weight"].T) * (h @ w[p + "mlp.up_proj.weight"].T)
        x = x + h @ w[p + "mlp.down_proj.weight"].T
    return _rms(x, eps, w["model.norm.weight"]), w["lm_head.weight"], 1.0


def _kesitar(c, w, tokens, seqs):
    eps, T, first = c.norm_eps, len(tokens), None
    x = w["embed"][tokens] * c.embedding_scale
    for i, layer in enumerate(c.layers):
        p, m = f"l{i}.", layer["mixer"]
        q, H, d, e = p + "mix.", m["heads"], m["dim"], m["vdim"]
        h = _layer_norm(x, w[p + "norm1"], eps)
        if layer["type"] == "attention":
            G = m.get("kv_heads", H)
            Q, Kk, v = ((h @ w[q + n].T + w[q + n + ".b"]).reshape(T, g, -1) for n, g in (("q", H), ("k", G), ("v", G)))
            Q, Kk = _rms(Q, eps, w[q + "q.norm"]), _rms(Kk, eps, w[q + "k.norm"])
            if m.get("rot"):
                freq, _ = _frequencies(m["rot"]["dims"], m["rot"]["base"])
                Q, Kk = (_each(seqs, lambda r: _turn(r, freq, False), r) for r in (Q, Kk))
            if m.get("v_mix"):
                if first is None:
                    first = v
                else:
                    v = v + w[q + "vmix"] * (first - v)
            sink = torch.zeros(H, dtype=x.dtype, device=x.device)
            o = _each(seqs, lambda a, b, g: _attend(a, b, g, m["scale"], m["mask"]["size"], m["mask"].get("pool") or 0, sink), Q, Kk, v)
        else:
            r = _silu(h @ w[q + "q"].T).reshape(T, H, d, 1)
            v = (h @ w[q + "v"].T).reshape(T, H, 1, e)
            low = w[q + "lower"]
            f = (low + (1.0 - low) * torch.sigmoid(h @ w[q + "f"].T + w[q + "f.b"])).reshape(T, H, d, 1)

            def token(S, at):
                S = torch.lerp(v[at].expand_as(S), S, f[at].expand_as(S))
                return S, (S * r[at]).sum(2)
            o = _walk(seqs, v[:, :, 0], torch.zeros(len(seqs), H, d, e, dtype=x.dtype, device=x.device), token)
            o = _rms(o, eps, w[q + "norm"])
        x = x + _layer_norm(o.reshape(T, H * e) @ w[q + "o"].T, w[p + "norm1b"], eps)
        h = _layer_norm(x, w[p + "norm2"], eps)
        h = (_silu(h @ w[p + "mlp.gate"].T) * (h @ w[p + "mlp.up"].T)) @ w[p + "mlp.down"].T
        x = x + _layer_norm(h, w[p + "norm2b"], eps)
    return _layer_norm(x, w["final.norm"], eps), w["embed"], c.logit_scale


def _sidirax(c, w, tokens, seqs):
    eps, T, kept = c.norm_eps, len(tokens), {}
    x = w["embed"][tokens]
    for i, layer in enumerate(c.layers):
        p, m, mlp = f"l{i}.", layer["mixer"], layer["mlp"]
        q, H, d = p + "mix.", m["heads"], m["dim"]
        h = _rms(x, eps, w[p + "norm1"])
        if layer["type"] == "latent_attention":
            rank, freq = m["kv_rank"], _frequencies(m["rot"]["dims"], m["rot"]["base"], m["rot"].get("scaling"))

            def turned(r):
                return _each(seqs, lambda s: _turn(s, freq[0], True, freq[1]), r)
            if m.get("kv_from") is None:
                rows = h @ w[q + "dkv"].T
                kept[i] = _rms(rows[:, :rank], eps, w[q + "dkv.norm"]), turned(rows[:, None, rank:].contiguous())
            latent, shared = kept[i if m.get("kv_from") is None else m["kv_from"]]
            Q = (_rms(h @ w[q + "dq"].T, eps, w[q + "dq.norm"]) @ w[q + "uq"].T).reshape(T, H, -1)
            Q = torch.cat([Q[..., :d], turned(Q[..., d:].contiguous())], -1)
            Kk = torch.cat([(latent @ w[q + "uk"].T).reshape(T, H, d), shared.expand(T, H, -1)], -1)
            v = (latent @ w[q + "uv"].T).reshape(T, H, -1)
            sink = w[q + "sink"]
            o = _each(seqs, lambda a, b, g: _attend(a, b, g, m["scale"], sink=sink), Q, Kk, v).reshape(T, -1)
        else:
            def before(s):
                return torch.cat([torch.zeros_like(s[:1]), s[:-1]])
            back = _each(seqs, before, h) - h
            r, k, v, g, decay = (h + back * w[q + "mu." + n] for n in "rkvgw")
            r, k = ((s @ w[q + n].T).reshape(T, H, d, 1) for s, n in ((r, "r"), (k, "k")))
            v, g = (v @ w[q + "v"].T).reshape(T, H, 1, d), _silu(g @ w[q + "g"].T)
            decay = torch.exp(-torch.exp(torch.tanh(decay @ w[q + "w1"].T) @ w[q + "w2"].T + w[q + "w0"])).reshape(T, H, d, 1)
            u = w[q + "u"].reshape(H, d, 1)

            def token(S, at):
                kv = k[at] * v[at]
                return decay[at] * S + kv, (r[at] * (S + u * kv)).sum(2)
            o = _walk(seqs, v[:, :, 0], torch.zeros(len(seqs), H, d, d, dtype=x.dtype, device=x.device), token)
            o = _rms(o, eps).reshape(T, H * d) * w[q + "norm"] * g
        y = o @ w[q + "o"].T
        q = p + "mlp."
        if mlp["kind"] == "dense":
            g = (h @ w[q + "gate"].T + w[q + "gate.b"]).clamp(max=mlp["limit"])
            up = (h @ w[q + "up"].T + w[q + "up.b"]).clamp(-mlp["limit"], mlp["limit"])
            y = y + (g * torch.sigmoid(1.702 * g) * (up + 1.0)) @ w[q + "down"].T + w[q + "down.b"]
        else:
            y = y + _experts(h, w, q, mlp, False)
        x = x + y
    return _rms(x, eps, w["final.norm"]), w["embed"], 1.0


def _zivovik(c, w, tokens, seqs):
    eps, mult, T = c.norm_eps, c.residual_mult, len(tokens)
    at = torch.cat([torch.arange(b - a, device="cuda") for a, b in seqs])
    x = w["embed"][tokens] * c.embedding_scale + w["pos"][at]
    start = x

    def temperature(m):
        return (1.0 + m["q_temp"]["coef"] * torch.log((at + 1) // m["q_temp"]["every"] + 1.0))[:, None, None]

    def conv(rows, taps):
        def one(r):
            n = taps.shape[1]
            r = torch.cat([torch.zeros(n - 1, r.shape[1], dtype=r.dtype, device=r.device), r])
            return sum(r[j:len(r) - n + 1 + j] * taps[:, j] for j in range(n))
        return _silu(_each(seqs, one, rows))

    for i, again in c.run_order():
        layer = c.layers[i]
        p, m = f"l{i}.", layer["mixer"]
        q = p + "mix."
        x = x + start if again else x
        h = _rms(x, eps, 1.0 + w[p + "norm1"])
        if layer["type"] == "attention":
            H, G, d = m["heads"], m["kv_heads"], m["dim"]
            Q, v = (h @ w[q + "q"].T).reshape(T, H, d), (h @ w[q + "k"].T).reshape(T, G, d)
            o = _each(seqs, lambda a, b, g: _attend(a, b, g, m["scale"]), _rms(Q, eps) * temperature(m), _rms(v, eps), v)
            y = (o.reshape(T, -1) * torch.sigmoid(h @ w[q + "g"].T)) @ w[q + "o"].T
        elif layer["type"] == "parallel":
            m, s, q, r = m["left"], m["right"], q + "left.", q + "right."
            H, G = m["heads"], m["kv_heads"]
            Q, Kk, v = ((h @ w[q + n].T).reshape(T, g, -1) for n, g in (("q", H), ("k", G), ("v", G)))
            o = _each(seqs, lambda a, b, g: _attend(a, b, g, m["scale"]), Q * temperature(m), Kk, v)
            y = _rms((o * torch.sigmoid(h @ w[q + "g"].T)[:, :, None]).reshape(T, -1) @ w[q + "o"].T, eps, w[q + "out"])
            H, G, d, e = s["heads"], s["kv_heads"], s["dim"], s["vdim"]
            Q, Kk, v = (conv(h @ w[r + n].T, w[r + n + ".conv"]).reshape(T, g, -1) for n, g in (("q", G), ("k", G), ("v", H)))
            Q, Kk = (a / torch.sqrt((a * a).sum(-1, keepdim=True) + 1e-6) for a in (Q, Kk))
            Q, Kk = (a.repeat_interleave(H // G, 1).unsqueeze(-1) for a in (Q * d ** -0.5, Kk))
            beta = torch.sigmoid(h @ w[r + "b"].T)[:, :, None]
            g = torch.exp(-torch.exp(w[r + "A_log"]) * torch.nn.functional.softplus(h @ w[r + "a"].T + w[r + "dt_bias"]))[:, :, None, None]

            def token(S, n):
                S = g[n] * S
                u = beta[n] * (v[n] - (S * Kk[n]).sum(2))
                S = S + Kk[n] * u[:, :, None]
                return S, (S * Q[n]).sum(2)
            o = _walk(seqs, v, torch.zeros(len(seqs), H, d, e, dtype=x.dtype, device=x.device), token)
            o = _rms(o, eps, w[r + "norm"]).reshape(T, -1) * _silu(h @ w[r + "g"].T)
            y = 0.5 * (y + _rms(o @ w[r + "o"].T, eps, w[r + "out"]))
        else:
            H, d, e = m["heads"], m["dim"], m["vdim"]
            Q, Kk, v = (_silu(h @ w[q + n].T).reshape(T, H, -1) for n in "qkv")
            keep = torch.tensor(m["decay"], dtype=x.dtype, device=x.device)[:, None, None]

            def token(S, n):
                S = keep * S + Kk[n][..., None] * v[n][:, :, None]
                return S, (S * Q[n][..., None]).sum(2)
            o = _walk(seqs, v, torch.zeros(len(seqs), H, d, e, dtype=x.dtype, device=x.device), token)
            y = (_rms(o.reshape(T, -1), eps, w[q + "norm"]) * torch.sigmoid(h @ w[q + "g"].T)) @ w[q + "o"].T
        x = x + mult * y
        if layer.get("mlp") is not None:
            x = x + mult * _experts(_rms(x, eps, 1.0 + w[p + "norm2"]), w, p + "mlp.", layer["mlp"], True)
    return _rms(x, eps, 1.0 + w["final.norm"]), w["head"], 1.0


_EXACT = {"mistral": _mistral, "kesitar": _kesitar, "sidirax": _sidirax, "zivovik": _zivovik}


def exact(case, seed):
    """What the first pass after `prepare` returns, every sequence run in float64 from its first token to its last."""
    config = _config(case)
    prompts, fed = _tokens(case, config, seed)
    whole = dict(case, task="turn")
    if work(whole)["flops"] > 4e14:           # about 20 seconds in float64
        return None
    steps = case["steps"]
    tokens, seqs, wanted = [], [], [[] for _ in range(steps + 1)]
    for b, p in enumerate(prompts):
        a = len(tokens)
        tokens += p + [fed[t][b] for t in range(steps)]
        seqs.append((a, len(tokens)))
        first = len(p) // 2 if case["want"] == "half" else len(p) - 1
        wanted[0] += range(a + first, a + len(p))
        for t in range(steps):
            wanted[t + 1].append(a + len(p) + t)
    if case["task"] == "decode":
        wanted = wanted[1:]
    family = case["model"].split("-")[0]
    h, head, scale = _EXACT[family](config, _Weights(config, seed), torch.tensor(tokens, device="cuda"), seqs)
    return h[torch.tensor(sum(wanted, []), device="cuda")] @ head.T * scale
