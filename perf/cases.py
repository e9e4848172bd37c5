"""Performance cases: what a program that serves models with this framework has it do.

Two calls carry that program: `Engine.prefill`, a prompt or a further turn of a conversation into a slot's cache, and the
pipelined decode (`decode_submit`, `decode_sample`, `decode_collect`) that the scheduler drives, with the next step's forward on
the GPU while the host takes the last step's tokens.  The engine, its weights and the cached contexts are what such a program
keeps: they are made by `prepare`.  One engine per model and cache type serves every state of a process, each in slots of its own.

The weights are random, in the byte layout of GGUF files (Q4_K_M: Q6_K for the output matrix and for part of attn_v and
ffn_down, Q4_K elsewhere) or bf16.  The output matrix is close to the embeddings of a permuted vocabulary, so the model is as
sure of its next token as a trained one: decoded tokens do not hang on rounding.
"""
from __future__ import annotations

import math

import torch

DEV = "cuda"
BATCH, SLOTS, POOL = 16, 64, 1 << 18     # the service's batch; slots of the states alive at a time; tokens of the cache pool
STEPS = 8                                # tokens a decode pass makes for each sequence

# what a server holds of each model: (preset, recipe, cache type, context).  The context is the loader's default, and the whole
# 32k where a long conversation is kept in the fp8 cache.
ENGINES = {
    "tinyllama-q4": ("tinyllama-1.1b", "Q4_K_M", "bf16", 2048),
    "tinyllama-bf16": ("tinyllama-1.1b", "BF16", "bf16", 2048),
    "mistral-q4": ("mistral-7b", "Q4_K_M", "bf16", 4096),
    "mistral-q4-fp8kv": ("mistral-7b", "Q4_K_M", "fp8_e4m3", 32768),
    "qwen3-q4": ("qwen3-8b", "Q4_K_M", "bf16", 4096),
    "seledra-bf16": ("seledra-1b", "BF16", "bf16", 4096),
}


def listed():
    def prefill(name, engine, tokens, start=0):
        return dict(name=name, op="prefill", engine=engine, tokens=tokens, start=start)

    def decode(name, engine, batch, context, temperature=0.0):
        return dict(name=name, op="decode", engine=engine, batch=batch, context=context, temperature=temperature)

    return [
        # a short instruction to the operational tier: the smallest prompt
        prefill("prefill-tiny-23", "tinyllama-q4", 23),
        # an agent's goal with its system prompt, to the tactical tier
        prefill("prefill-mistral-130", "mistral-q4", 130),
        # the same with tool results and memory retrieved into it
        prefill("prefill-qwen3-711", "qwen3-q4", 711),
        # a whole document, more than the engine takes in one portion
        prefill("prefill-mistral-3900", "mistral-q4", 3900),
        # a further turn of a long conversation, its prefix in the fp8 cache
        prefill("prefill-turn-300", "mistral-q4-fp8kv", 300, start=6000),
        # a prompt of a design described layer by layer: attention beside a linear recurrence, bf16 weights
        prefill("prefill-seledra-1500", "seledra-bf16", 1500),
        # one stream of the operational tier: the lightest token
        decode("decode-tiny-b1", "tinyllama-q4", 1, 128),
        # three goals at once on the unquantised operational model
        decode("decode-tinybf16-b3", "tinyllama-bf16", 3, 500, 0.7),
        # one stream of the tactical tier
        decode("decode-mistral-b1", "mistral-q4", 1, 128),
        # one stream far into a long conversation
        decode("decode-mistral-long", "mistral-q4-fp8kv", 1, 16000),
        # the service's full batch
        decode("decode-mistral-b16", "mistral-q4", 16, 1000, 0.7),
        # the same on the layered design, whose recurrent state stands after one token
        decode("decode-seledra-b16", "seledra-bf16", 16, 300),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    engine = rng.choice(sorted(ENGINES))
    ctx = ENGINES[engine][3]
    long = ctx > 4096
    if rng.random() < 0.5:
        # a prompt from the shortest to nearly the whole context, or a further turn behind a cached one
        start = _log(rng, 64, 12000 if long else ctx // 2) if engine != "seledra-bf16" and (long or rng.random() < 0.3) else 0
        tokens = _log(rng, 8, 1000 if long else min(3900, ctx - start - 8))
        return dict(op="prefill", engine=engine, tokens=tokens, start=start)
    batch = _log(rng, 1, 4 if long else BATCH)
    most = min(16000 if long else ctx - 96, 24000 // batch)
    return dict(op="decode", engine=engine, batch=batch, context=_log(rng, 1000 if long else 32, most),
                temperature=rng.choice([0.0, 0.7]))


# ---- weights ----------------------------------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(DEV).manual_seed(seed & 0x7FFFFFFFFFFFFFFF)


class Q4K:
    """256 weights: 8 groups of 32 values d s q - e m of 4-bit q, 6-bit s and m; d, e in fp16."""
    TYPE = "Q4_K"

    def __init__(self, rows, cols, std, seed):
        g, n = _gen(seed), cols // 256
        self.q = torch.randn(rows, n, 8, 32, generator=g, device=DEV).mul_(2.6).add_(7.5).round_().clamp_(0, 15).to(torch.uint8)
        self.s = torch.randint(24, 64, (rows, n, 8), generator=g, device=DEV, dtype=torch.uint8)
        d = std / (2.6 * 43.5) * (0.8 + 0.4 * torch.rand(rows, n, generator=g, device=DEV))
        self.d, self.e, self.m = d.half(), (7.5 * d).half(), self.s

    def bytes(self):
        s, m, q = self.s, self.m, self.q
        rows, n = s.shape[:2]
        sc = torch.cat([s[..., :4] & 63 | (s[..., 4:] >> 4) << 6, m[..., :4] & 63 | (m[..., 4:] >> 4) << 6,
                        s[..., 4:] & 15 | (m[..., 4:] & 15) << 4], -1)
        qs = (q[:, :, 0::2] | q[:, :, 1::2] << 4).reshape(rows, n, 128)
        de = torch.stack([self.d, self.e], -1).view(torch.uint8).reshape(rows, n, 4)
        return torch.cat([de, sc, qs], -1)

    def values(self, dt):
        w = (self.d.to(dt)[..., None] * self.s.to(dt))[..., None] * self.q.to(dt)
        w -= (self.e.to(dt)[..., None] * self.m.to(dt))[..., None]
        return w.reshape(w.shape[0], -1)


class Q6K:
    """256 weights: 16 groups of 16 values d s (q - 32) of 6-bit q, 8-bit s; d in fp16."""
    TYPE = "Q6_K"

    def __init__(self, rows, cols, std, seed):
        g, n = _gen(seed), cols // 256
        self.q = torch.randn(rows, n, 16, 16, generator=g, device=DEV).mul_(10).add_(32).round_().clamp_(0, 63).to(torch.uint8)
        self.s = torch.randint(64, 128, (rows, n, 16), generator=g, device=DEV, dtype=torch.uint8)
        self.d = (std / 960 * (0.8 + 0.4 * torch.rand(rows, n, generator=g, device=DEV))).half()

    @classmethod
    def of(cls, w):
        """The matrix w, rounded."""
        o, w = cls.__new__(cls), w.reshape(w.shape[0], -1, 16, 16)
        top = w.abs().amax(-1).clamp_(min=1e-6)
        o.d = (top.amax(-1) / (31 * 120)).half()
        o.s = (top / (31 * o.d.float()[..., None])).ceil_().clamp_(1, 127).to(torch.uint8)
        o.q = (w / (o.d.float()[..., None] * o.s.float())[..., None]).round_().add_(32).clamp_(0, 63).to(torch.uint8)
        return o

    def bytes(self):
        rows, n = self.s.shape[:2]
        q = self.q.reshape(rows, n, 2, 4, 32)
        lo, hi = q & 15, q >> 4
        ql = torch.cat([lo[:, :, :, 0] | lo[:, :, :, 2] << 4, lo[:, :, :, 1] | lo[:, :, :, 3] << 4], -1).reshape(rows, n, 128)
        qh = (hi[:, :, :, 0] | hi[:, :, :, 1] << 2 | hi[:, :, :, 2] << 4 | hi[:, :, :, 3] << 6).reshape(rows, n, 64)
        return torch.cat([ql, qh, self.s, self.d[..., None].view(torch.uint8).reshape(rows, n, 2)], -1)

    def values(self, dt):
        w = (self.d.to(dt)[..., None] * self.s.to(dt))[..., None] * (self.q.to(dt) - 32)
        return w.reshape(w.shape[0], -1)


class Plain:
    """bf16 weights, or fp32 ones."""

    def __init__(self, w, dt):
        self.w, self.TYPE = w.to(dt), "BF16" if dt == torch.bfloat16 else "F32"

    def bytes(self):
        return self.w.contiguous().view(torch.uint8)

    def values(self, dt):
        return self.w.to(dt)


def _normal(shape, std, seed, base=0.0):
    return torch.randn(shape, generator=_gen(seed), device=DEV) * std + base


def _output_of(emb, cls):
    """Row t's direction is the embedding of the token before t: (matrix, the token after each token)."""
    V, d = emb.shape
    after = torch.randperm(V, generator=_gen(11), device=DEV)
    w = torch.empty_like(emb)
    w[after] = emb * (1.5 / math.sqrt(d))
    return cls(w), after


class Llama:
    """The llama family's tensors, in the order of a GGUF file; a class per tensor, so that a layer is made when asked for."""

    def __init__(self, cfg, recipe):
        self.cfg, self.recipe = cfg, recipe

    def _matrix(self, name, layer, rows, cols, std, k):
        seed, n = 1000 * (layer + 2) + k, self.cfg.n_layers
        if self.recipe == "BF16":
            return Plain(_normal((rows, cols), std, seed), torch.bfloat16)
        more = layer < n // 8 or layer >= 7 * n // 8 or (layer - n // 8) % 3 == 2
        six = name in ("attn_v", "ffn_down") and more
        return (Q6K if six else Q4K)(rows, cols, std, seed)

    def head(self):
        """(embeddings, output matrix, output norm, the token after each token)."""
        c = self.cfg
        emb = self._matrix("token_embd", -1, c.vocab_size, c.d_model, 1.0, 0)
        cls = (lambda w: Plain(w, torch.bfloat16)) if self.recipe == "BF16" else Q6K.of
        out, after = _output_of(emb.values(torch.float32), cls)
        return emb, out, Plain(_normal((c.d_model,), 0.1, 5, 1.0), torch.float32), after

    def layer(self, i):
        c = self.cfg
        d, qd, kd, ff = c.d_model, c.n_heads * c.head_dim, c.n_kv_heads * c.head_dim, c.d_ff
        g = 1 / math.sqrt(d)
        shapes = [("attn_q", qd, d, g), ("attn_k", kd, d, g), ("attn_v", kd, d, g), ("attn_output", d, qd, 0.3 / math.sqrt(qd)),
                  ("ffn_gate", ff, d, g), ("ffn_up", ff, d, g), ("ffn_down", d, ff, 0.3 / math.sqrt(ff))]
        w = {n: self._matrix(n, i, r, k, std, j) for j, (n, r, k, std) in enumerate(shapes)}
        norms = {"attn_norm": d, "ffn_norm": d, **({"attn_q_norm": c.head_dim, "attn_k_norm": c.head_dim} if c.qk_norm else {})}
        for j, (n, k) in enumerate(norms.items()):
            w[n] = Plain(_normal((k,), 0.1, 1000 * (i + 2) + 50 + j, 1.0), torch.float32)
        return w

    def tensors(self):
        emb, out, norm, _ = self.head()
        yield from (("token_embd.weight", emb), ("output.weight", out), ("output_norm.weight", norm))
        for i in range(self.cfg.n_layers):
            for n, t in self.layer(i).items():
                yield f"blk.{i}.{n}.weight", t


class Seledra:
    def __init__(self, cfg, recipe):
        self.cfg = cfg

    def head(self):
        c = self.cfg
        emb = Plain(_normal((c.vocab_size, c.d_model), 1.0, 0), torch.bfloat16)
        out, after = _output_of(emb.values(torch.float32), lambda w: Plain(w, torch.bfloat16))
        return emb, out, Plain(_normal((c.d_model,), 0.1, 5, 1.0), torch.bfloat16), after

    def positions(self):
        return Plain(_normal((self.cfg.max_ctx, self.cfg.d_model), 0.3, 7), torch.bfloat16)

    def layer(self, i):
        c, l, d, ff = self.cfg, self.cfg.layers[i], self.cfg.d_model, self.cfg.layers[i].ff
        g, w = 1 / math.sqrt(d), {"attn_norm.weight": ((d,), 0.1, 1.0), "ffn_norm.weight": ((d,), 0.1, 1.0)}
        if l.mixer == "gqa":
            H, G = l.heads, l.kv_heads
            for n, k in (("q", H * l.dim), ("k", G * l.dim), ("v", G * l.vdim)):
                w.update({f"attn_{n}.weight": ((k, d), g, 0), f"attn_{n}.bias": ((k,), 0.3, 0)})
            w.update({"attn_q_norm.weight": ((H * l.dim,), 0.1, 1), "attn_k_norm.weight": ((G * l.dim,), 0.1, 1),
                      "attn_temp.weight": ((H,), 0.2, 1), "attn_gate.weight": ((H, d), g, 0),
                      "attn_output.weight": ((d, H * l.vdim), 0.5 / math.sqrt(H * l.vdim), 0),
                      "attn_v_mix.weight": ((1,), 0.1, 0.5)})
        else:
            H, G, nk, nv = l.lin.heads, l.lin.groups, l.lin.groups * l.lin.dim, l.lin.heads * l.lin.vdim
            for n, k in (("q", nk), ("k", nk), ("v", nv)):
                w.update({f"delta_{n}.weight": ((k, d), g, 0), f"delta_{n}_conv1d.weight": ((k, l.lin.conv), 0.5, 0)})
            w.update({"delta_b.weight": ((H, d), g, 0), "delta_a.weight": ((H, d), g, 0), "delta_a_log.bias": ((H,), 0.5, -1),
                      "delta_dt.bias": ((H,), 0.5, -1.5), "delta_norm.weight": ((l.lin.vdim,), 0.1, 1),
                      "delta_gate.weight": ((nv, d), g, 0), "delta_output.weight": ((d, nv), 0.5 / math.sqrt(nv), 0)})
        w.update({"ffn_up.weight": ((ff, d), g, 0), "ffn_down.weight": ((d, ff), 0.3 / math.sqrt(ff), 0), "ffn_act.bias": ((2,), 0.2, 0)})
        return {n: Plain(_normal(s, std, 1000 * (i + 2) + j, base), torch.bfloat16) for j, (n, (s, std, base)) in enumerate(w.items())}

    def tensors(self):
        emb, out, norm, _ = self.head()
        yield from (("token_embd.weight", emb), ("output.weight", out), ("output_norm.weight", norm),
                    ("position_embd.weight", self.positions()))
        for i in range(self.cfg.n_layers):
            w = self.layer(i)
            if self.cfg.layers[i].mixer == "gqa" and not self.cfg.layers[i].v_mix:
                del w["attn_v_mix.weight"]
            for n, t in w.items():
                yield f"blk.{i}.{n}", t


def _model(engine):
    from aios_amd.models.config import get_preset

    preset, recipe, _, _ = ENGINES[engine]
    cfg = get_preset(preset)
    return (Seledra if cfg.layers else Llama)(cfg, recipe)


# ---- the program ------------------------------------------------------------------------------------------------------
_held = {}


def _engine(engine):
    """(engine, its free slots): loaded once, as a server does."""
    if engine not in _held:
        from aios_amd.gguf.quants import GGMLType
        from aios_amd.runtime import loader, native

        model, (_, _, kv, ctx) = _model(engine), ENGINES[engine]
        eng = native.require().Engine(native.engine_config(model.cfg, max_ctx=ctx, max_slots=SLOTS, max_batch=BATCH, kv_dtype=kv,
                                                           kv_pool_tokens=POOL))
        for name, t in model.tensors():
            raw = t.bytes()
            shape = raw.shape if t.TYPE in ("Q4_K", "Q6_K") else t.w.shape
            rows = shape[0] if len(shape) > 1 else 1
            cols = shape[1] * 256 if t.TYPE in ("Q4_K", "Q6_K") else t.w.numel() // rows
            eng.set_tensor(name, int(GGMLType[t.TYPE]), rows, cols, raw.reshape(-1).cpu().numpy())
        loader.finalize(eng)
        if kv != "bf16":
            eng.set_kv_scales([1 / 32] * (2 * model.cfg.n_layers))  # keys and values are of size 1; codes reach 448
        _held[engine] = eng, list(range(SLOTS))
    return _held[engine]


class State:
    """Slots of the engine with their contexts cached; given back at its end."""

    def __init__(self, engine, n):
        self.engine, free = _engine(engine)
        self.slots = [free.pop() for _ in range(n)]
        self.free = free

    def __del__(self):
        for s in self.slots:
            self.engine.release_slot(s)
            self.free.append(s)


def _tokens(case, seed):
    """Per sequence (tokens cached before the call, tokens of the call): the last are the prompt, or the token to go on from."""
    from aios_amd.models.config import get_preset

    g = torch.Generator().manual_seed(seed)
    V, B = get_preset(ENGINES[case["engine"]][0]).vocab_size, case.get("batch", 1)
    out = []
    for b in range(B):
        if case["op"] == "prefill":
            before, now = case["start"], case["tokens"]
        else:  # contexts of unlike length, as they are in a batch
            before, now = max(1, case["context"] - case["context"] * b // (2 * B)), 1
        t = torch.randint(3, V, (before + now,), generator=g).tolist()
        out.append((t[:before], t[before:]))
    return out


def _steps(case):
    return 1 if case["engine"] == "seledra-bf16" else STEPS


def prepare(case, seed):
    seqs = _tokens(case, seed)
    st = State(case["engine"], len(seqs))
    st.case, st.now = case, [now for _, now in seqs]
    for slot, (before, _) in zip(st.slots, seqs):
        if before:
            st.engine.prefill(slot, before, 0, False)
    st.pos = [len(before) for before, _ in seqs]
    st.seeds = [seed * 100 + b for b in range(len(seqs))]
    return st


def run(st):
    eng = st.engine
    if st.case["op"] == "prefill":
        return eng.prefill(st.slots[0], st.now[0], st.pos[0], True)
    B, T = len(st.slots), st.case["temperature"]
    kw = dict(temperature=[T] * B, top_k=[40 if T else 0] * B, top_p=[0.95 if T else 1.0] * B, seeds=st.seeds)
    pos, made = list(st.pos), []
    eng.decode_submit(st.slots, [t[0] for t in st.now], pos, **kw)
    eng.decode_sample()
    for _ in range(_steps(st.case) - 1):  # the next step is on its way before the host sees this one's tokens
        pos = [p + 1 for p in pos]
        eng.decode_submit(st.slots, [], pos, **kw)
        made.append(eng.decode_collect())
        eng.decode_sample()
    made.append(eng.decode_collect())
    return {"tokens": torch.tensor(made), "logits": eng.last_logits(B)}


# ---- what a pass cannot do without --------------------------------------------------------------------------------------
def _sizes(engine):
    """(bytes of the layers' weights, of the output matrix, of a token's cache; numbers of the layers, of the output matrix;
    numbers per query and key that attention multiplies)."""
    from aios_amd.models.config import get_preset

    preset, recipe, kv, _ = ENGINES[engine]
    c = get_preset(preset)
    d, V, out = c.d_model, c.vocab_size, 0
    if c.layers:
        n = c.n_params() - (2 * V + c.max_ctx) * d
        att = [l for l in c.layers if l.mixer == "gqa"]
        return (2 * n, 2 * V * d, 2 * sum(l.kv_heads * (l.dim + l.vdim) for l in att), n, V * d,
                sum(l.heads * (l.dim + l.vdim) for l in att))
    qd, kd = c.n_heads * c.head_dim, c.n_kv_heads * c.head_dim
    nb = n = 0.0
    for i in range(c.n_layers):
        more = i < c.n_layers // 8 or i >= 7 * c.n_layers // 8 or (i - c.n_layers // 8) % 3 == 2
        for numbers, six in ((d * (2 * qd + kd + 2 * c.d_ff), False), (d * (kd + c.d_ff), more)):
            n += numbers
            nb += numbers * (2 if recipe == "BF16" else 210 / 256 if six else 144 / 256)
    return nb, V * d * (2 if recipe == "BF16" else 210 / 256), 2 * c.n_layers * kd * (1 if kv != "bf16" else 2), n, V * d, 2 * c.n_layers * qd


def work(case):
    wb, ob, kvb, wn, on, att = _sizes(case["engine"])
    if case["op"] == "prefill":
        T, s = case["tokens"], case["start"]
        keys = T * s + T * (T + 1) / 2
        return {"bytes": wb + ob + kvb * (s + T), "flops": 2.0 * (wn * T + on + att * keys)}
    B, n = case["batch"], _steps(case)
    keys = sum(max(1, case["context"] - case["context"] * b // (2 * B)) + (n + 1) / 2 for b in range(B))
    by, fl = wb + ob + kvb * keys, 2.0 * (wn * B + on * B + att * keys)
    if case["engine"] == "seledra-bf16":  # every sequence's recurrent state, read and written
        from aios_amd.models.config import get_preset

        by += B * sum(8 * l.lin.heads * l.lin.dim * l.lin.vdim for l in get_preset(ENGINES[case["engine"]][0]).layers if l.lin)
    return {"bytes": by * n, "flops": fl * n}


def tolerance(case):
    # four times the measured distance of the logits from 64 bits and of two runs from each other, no more than 0.03: bf16
    # weights and products 0.0036, max 0.02; 4-bit weights with bf16 products 0.0080, max 0.031, with the 8-bit activations
    # of up to four rows 0.013, max 0.071.  (The sums' order is not fixed in every product.)
    if case["engine"].endswith("bf16"):
        return {"rel": 0.015, "max": 0.08, "differ": 0.01}
    return {"rel": 0.03, "max": 0.28 if case.get("batch", 99) <= 4 else 0.13, "differ": 0.01}


# ---- the same in 64 bits, from the weights' numbers -----------------------------------------------------------------------
F64 = torch.float64


def _rms(x, eps, w=None):
    x = x / torch.sqrt(x.pow(2).mean(-1, keepdim=True) + eps)
    return x if w is None else x * w


def _attend(q, k, v, n_keep, scale, extra):
    """Causal attention of the last n_keep rows' queries; extra: a number added to the softmax's denominator."""
    T, H, hd = q.shape
    G, out = k.shape[1], torch.empty(n_keep, H, v.shape[2], dtype=F64, device=q.device)
    step = max(1, int(1.5e9) // (8 * T * (H // G)))
    for g in range(G):
        hs = slice(g * (H // G), (g + 1) * (H // G))
        for a in range(T - n_keep, T, step):
            b = min(T, a + step)
            s = torch.matmul(q[a:b, hs].transpose(0, 1), k[:b, g].T.contiguous()) * scale
            s.masked_fill_(torch.arange(b, device=q.device) > torch.arange(a, b, device=q.device)[:, None], -math.inf)
            if extra:
                s = torch.cat([s, torch.zeros_like(s[..., :1])], -1)
            p = torch.softmax(s, -1)[..., :b]
            out[a - (T - n_keep):b - (T - n_keep), hs] = torch.matmul(p, v[:b, g]).transpose(0, 1)
    return out.reshape(n_keep, -1)


def _llama64(model, seqs):
    """Logits of every sequence's last token."""
    c = model.cfg
    H, G, hd = c.n_heads, c.n_kv_heads, c.head_dim
    lens = [len(s) for s in seqs]
    emb, out, norm, _ = model.head()
    x = emb.values(F64)[torch.tensor([t for s in seqs for t in s], device=DEV)]
    pos = torch.cat([torch.arange(n, device=DEV) for n in lens]).to(F64)
    ang = pos[:, None] * c.rope_theta ** (-2.0 * torch.arange(hd // 2, device=DEV, dtype=F64) / hd)
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]

    def turn(y):
        if c.rope_mode == 2:
            a, b = y[..., :hd // 2], y[..., hd // 2:]
            return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)
        a, b = y[..., 0::2], y[..., 1::2]
        return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).reshape(y.shape)

    for i in range(c.n_layers):
        w = model.layer(i)
        W = lambda n: w.pop(n).values(F64)  # noqa: E731
        h = _rms(x, c.norm_eps, W("attn_norm"))
        q, k, v = ((h @ W(n).T).view(len(h), -1, hd) for n in ("attn_q", "attn_k", "attn_v"))
        if c.qk_norm:
            q, k = _rms(q, c.norm_eps, W("attn_q_norm")), _rms(k, c.norm_eps, W("attn_k_norm"))
        q, k = turn(q), turn(k)
        o, at = [], 0
        for n in lens:
            o.append(_attend(q[at:at + n], k[at:at + n], v[at:at + n], n, hd ** -0.5, False))
            at += n
        x = x + torch.cat(o) @ W("attn_output").T
        h = _rms(x, c.norm_eps, W("ffn_norm"))
        gate, up, down = W("ffn_gate"), W("ffn_up"), W("ffn_down")
        for a in range(0, len(h), 4096):  # (rows in portions: the gate's numbers are the largest tensor)
            z = h[a:a + 4096] @ gate.T
            x[a:a + 4096] += (z * torch.sigmoid(z) * (h[a:a + 4096] @ up.T)) @ down.T
    last = torch.tensor(lens, device=DEV).cumsum(0) - 1
    return _rms(x[last], c.norm_eps, norm.values(F64)) @ out.values(F64).T


def _silu(z):
    return z * torch.sigmoid(z)


def _softplus(z):
    return torch.log1p(torch.exp(-z.abs())) + z.clamp(min=0)


def _seledra64(model, seqs):
    c, eps, B = model.cfg, model.cfg.norm_eps, len(seqs)
    lens, T = [len(s) for s in seqs], max(len(s) for s in seqs)
    tok = torch.tensor([s + [0] * (T - len(s)) for s in seqs], device=DEV)  # (causal: what follows a sequence's end is not read)
    emb, out, norm, _ = model.head()
    x = emb.values(F64)[tok] + model.positions().values(F64)[:T]
    first = None
    for i, l in enumerate(c.layers):
        w = {n: t.values(F64) for n, t in model.layer(i).items()}
        h = _rms(x, eps, w["attn_norm.weight"])
        if l.mixer == "gqa":
            H, G = l.heads, l.kv_heads
            q, k, v = (h @ w[f"attn_{n}.weight"].T + w[f"attn_{n}.bias"] for n in "qkv")
            q = _rms(q, eps, w["attn_q_norm.weight"]).view(B, T, H, l.dim) * w["attn_temp.weight"][:, None]
            k = _rms(k, eps, w["attn_k_norm.weight"]).view(B, T, G, l.dim)
            v = _rms(v.view(B, T, G, l.vdim), eps)
            if l.v_mix:
                lam = w["attn_v_mix.weight"]
                first, v = (v, v) if first is None else (first, (1 - lam) * v + lam * first)
            o = torch.stack([_attend(q[b], k[b], v[b], T, l.scale, True) for b in range(B)]).view(B, T, H, l.vdim)
            o = (o * torch.sigmoid(h @ w["attn_gate.weight"].T)[..., None]).reshape(B, T, -1) @ w["attn_output.weight"].T
        else:
            H, G, dk, dv = l.lin.heads, l.lin.groups, l.lin.dim, l.lin.vdim

            def conv(n):
                u, k = h @ w[f"delta_{n}.weight"].T, w[f"delta_{n}_conv1d.weight"]
                u = torch.cat([torch.zeros_like(u[:, :l.lin.conv - 1]), u], 1)
                return _silu(sum(k[:, j] * u[:, j:j + T] for j in range(l.lin.conv)))

            q, k, v = conv("q").view(B, T, G, dk), conv("k").view(B, T, G, dk), conv("v").view(B, T, H, dv)
            q, k = (y / torch.sqrt(y.pow(2).sum(-1, keepdim=True) + 1e-6) for y in (q, k))
            q, k = (q / math.sqrt(dk)).repeat_interleave(H // G, 2), k.repeat_interleave(H // G, 2)
            beta = torch.sigmoid(h @ w["delta_b.weight"].T)
            dec = torch.exp(-torch.exp(w["delta_a_log.bias"]) * _softplus(h @ w["delta_a.weight"].T + w["delta_dt.bias"]))
            S, o = torch.zeros(B, H, dk, dv, dtype=F64, device=DEV), torch.empty(B, T, H, dv, dtype=F64, device=DEV)
            for t in range(T):
                S *= dec[:, t, :, None, None]
                kt = k[:, t, :, :, None]
                u = beta[:, t, :, None] * (v[:, t] - (S * kt).sum(2))
                S += kt * u[:, :, None]
                o[:, t] = (S * q[:, t, :, :, None]).sum(2)
            o = (_rms(o, eps, w["delta_norm.weight"]).reshape(B, T, -1) * _silu(h @ w["delta_gate.weight"].T)) @ w["delta_output.weight"].T
        x = x + l.mixer_scale * o
        z = _rms(x, eps, w["ffn_norm.weight"]) @ w["ffn_up.weight"].T
        a, neg = w["ffn_act.bias"], z.clamp(max=0)
        z = z / 2 + torch.where(z > 0, _softplus(a[0]) * z * z, (0.5 + _softplus(a[1])) * (torch.expm1(neg) - neg))
        x = x + l.mlp_scale * (z @ w["ffn_down.weight"].T)
    x = x[torch.arange(B, device=DEV), torch.tensor(lens, device=DEV) - 1]
    return _rms(x, eps, norm.values(F64)) @ out.values(F64).T


def exact(case, seed):
    model, seqs = _model(case["engine"]), _tokens(case, seed)
    f = _seledra64 if case["engine"] == "seledra-bf16" else _llama64
    with torch.no_grad():
        if case["op"] == "prefill":
            return f(model, [before + now for before, now in seqs])[0].cpu()
        # the tokens that a model this sure of itself makes, whatever the temperature
        after, n = model.head()[3].cpu(), _steps(case)
        made = [[int(now[0]) for _, now in seqs]]
        for _ in range(n):
            made.append([int(after[t]) for t in made[-1]])
        logits = f(model, [before + [made[j][b] for j in range(n)] for b, (before, _) in enumerate(seqs)])
        return {"tokens": torch.tensor(made[1:]), "logits": logits.cpu()}
