"""Performance cases of the attention path: what the speech runtimes above this library have it do, through its public
entry points (flash_attn_ext, cpy, set_rows, flash_attn_relpos).

A case is a dict of plain values; `kind` says which of the runtimes' call sequences it is:

  encoder    an audio encoder's self-attention, layer by layer: no mask, [token][head][dim] activations.  kv "pad": K and V
             arrive as F32 and are copied into a zero-padded F16 buffer first, as Whisper's encoder graph does it;
             "f16" / "f32": K and V are handed over as they are
  cross      a decoder's cross-attention: few query rows against the encoder's K/V, no mask
  whisper    one step of a Whisper decoder with several beams, all layers: the beams' new K/V rows go into the unified
             cache, self-attention under the beams' mask of cells, cross-attention over the encoder's K/V
  step       one step of an LLM decoder, one token, all layers: the token's K/V rows go into the layer's cache slice, attention
             over the rows so far - or, with `fixed`, over the whole cache with the unwritten rows masked out
  batch      the same step for many sequences of different lengths in one call, one layer: a mask ends each of them
  prefill    a prompt (or a chunk of a long one behind `past` rows), layer by layer: K/V rows into the cache, causal mask
  bias       a FastConformer block's attention over a padded batch, the relative positions in a per-head F16 mask
  relpos     the same block with the position term computed by the call
  kv_cast    a quantised cache read back as F32, K and V of every layer

Inputs are unit-variance normal values (K scaled where the runtime scales it), masks hold 0 and -inf.
"""
from __future__ import annotations

import math

import torch

import crispasr_amd as ca
from crispasr_amd import ggml

TYPES = {"f32": ggml.F32, "f16": ggml.F16, "q8_0": ggml.Q8_0, "q4_0": ggml.Q4_0, "q4_1": ggml.Q4_1, "q5_0": ggml.Q5_0, "q5_1": ggml.Q5_1}


def listed():
    return [
        # the smallest call: one decoder token of a Moonshine-sized model (8 heads of 36) against 375 encoder frames
        dict(name="cross_token_d36", kind="cross", layers=1, hd=36, heads=8, tokens=1, frames=375, kv="f32"),
        # Whisper large-v3: a step of beam search, 5 beams, 32 layers
        dict(name="whisper_large_beam5", kind="whisper", layers=32, heads=20, beams=5, cells=560, prompt=60, frames=1500),
        # a Voxtral-style LLM (30 layers, 32 query / 8 KV heads of 128): a token near the end of an answer, Q8_0 cache
        dict(name="llm_step_q8_0", kind="step", layers=30, hd=128, hq=32, hkv=8, kv="q8_0", past=662, ctx=704, fixed=False),
        # a Qwen3-ASR-style LLM (28 layers, 16 query / 8 KV heads): the graph of fixed cache length, an early token
        dict(name="llm_step_fixed_f16", kind="step", layers=28, hd=128, hq=16, hkv=8, kv="f16", past=419, ctx=2048, fixed=True),
        # a server's step: 64 sequences of 500 to 4096 tokens in one call
        dict(name="llm_batch64_q8_0", kind="batch", batch=64, hd=128, hq=32, hkv=8, kv="q8_0", shortest=500, ctx=4096),
        # Voxtral's prompt: 375 audio and 32 text tokens into a Q8_0 cache
        dict(name="prefill_407_q8_0", kind="prefill", layers=4, hd=128, hq=32, hkv=8, kv="q8_0", tokens=407, past=0),
        # a chunk of a long transcript's context behind 2048 rows
        dict(name="prefill_2048_f16", kind="prefill", layers=1, hd=128, hq=32, hkv=8, kv="f16", tokens=2048, past=2048),
        # Whisper base: the encoder of one window, 6 layers, as its graph runs it
        dict(name="encoder_base", kind="encoder", layers=6, hd=64, heads=8, tokens=1500, batch=1, kv="pad"),
        # Whisper large-v3: encoder layers over four windows at once
        dict(name="encoder_large_x4", kind="encoder", layers=4, hd=64, heads=20, tokens=1500, batch=4, kv="f16"),
        # Parakeet / Canary-CTC: a block over 8 utterances of 400 to 750 frames, both forms of the call
        dict(name="conformer_mask_x8", kind="bias", hd=128, heads=8, tokens=750, shortest=400, batch=8, kv="f16"),
        dict(name="conformer_750_x8", kind="relpos", hd=128, heads=8, tokens=750, shortest=400, batch=8, kv="f32", table="f32"),
        # an LLM runtime that casts its quantised cache before it expands the heads: one step's reads
        dict(name="kv_cast_q8_0", kind="kv_cast", layers=30, hd=128, heads=8, tokens=663, ctx=704, kv="q8_0"),
    ]


def draw(rng):
    def between(lo, hi):             # over the logarithm
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["encoder", "encoder", "cross", "whisper", "step", "step", "batch", "prefill", "prefill", "bias", "relpos", "kv_cast"])
    if kind == "encoder":
        hd = rng.choice([64, 64, 64, 80, 96, 128])
        heads = rng.choice([h for h in (6, 8, 10, 12, 16, 20) if h * hd <= 1280])
        tokens = between(150, 1536)
        kv = rng.choice(["pad", "f16", "f32"])
        batch = 1 if kv == "pad" else rng.choice([1, 2, 3, 4])
        return dict(kind=kind, layers=rng.choice([1, 4]) if batch > 1 else rng.choice([4, 6, 12]), hd=hd, heads=heads, tokens=tokens, batch=batch, kv=kv)
    if kind == "cross":
        hd = rng.choice([36, 52, 64, 64, 80, 128])
        return dict(kind=kind, layers=rng.choice([1, 6, 8]), hd=hd, heads=rng.choice([8, 12, 16, 20]), tokens=rng.choice([1, 1, 2, 5, 24]),
                    frames=between(40, 1536), kv=rng.choice(["f32", "f16", "f16"]))
    if kind == "whisper":
        layers, heads = rng.choice([(4, 6), (6, 8), (12, 12), (24, 16), (32, 20), (4, 20)])
        beams, prompt = rng.randint(1, 5), between(4, 200)
        return dict(kind=kind, layers=layers, heads=heads, beams=beams, cells=prompt + beams * between(1, 180), prompt=prompt, frames=between(100, 1536))
    if kind == "step":
        hd, hq, hkv = rng.choice([(128, 32, 8), (128, 16, 8), (128, 8, 8), (64, 16, 16), (64, 32, 8)])
        ctx, fixed = rng.choice([704, 1024, 2048, 4096]), rng.random() < 0.4
        return dict(kind=kind, layers=rng.choice([8, 24, 28, 30]), hd=hd, hq=hq, hkv=hkv, kv=rng.choice(["f16", "f16", "q8_0", "q8_0", "q4_0", "q5_1"]),
                    past=min(between(32, 4095), ctx - 1), ctx=ctx, fixed=fixed)
    if kind == "batch":
        hd, hq, hkv = rng.choice([(128, 32, 8), (128, 16, 8), (128, 8, 8), (64, 32, 8)])
        ctx = between(256, 4096)
        kv = rng.choice(["f16", "q8_0", "q8_0", "q4_0"])
        return dict(kind=kind, batch=between(2, 32 if kv == "f16" else 64), hd=hd, hq=hq, hkv=hkv, kv=kv,
                    shortest=max(1, int(ctx * rng.uniform(0.05, 1.0))), ctx=ctx)
    if kind == "prefill":
        hd, hq, hkv = rng.choice([(128, 32, 8), (128, 16, 8), (128, 8, 8), (64, 16, 16), (64, 32, 8)])
        tokens = between(16, 2048)
        return dict(kind=kind, layers=rng.choice([1, 4]) if tokens < 600 else 1, hd=hd, hq=hq, hkv=hkv, kv=rng.choice(["f16", "f16", "q8_0", "q8_0", "q4_0"]),
                    tokens=tokens, past=rng.choice([0, 0, between(1, 2048)]))
    if kind in ("bias", "relpos"):
        tokens = between(50, 1000)
        c = dict(kind=kind, hd=rng.choice([64, 128, 128]), heads=rng.choice([4, 8]), tokens=tokens, shortest=max(1, int(tokens * rng.uniform(0.3, 1.0))),
                 batch=rng.choice([1, 1, 2, 4, 8]), kv=rng.choice(["f32", "f32", "f16"]))
        return dict(c, table=rng.choice(["f32", "f16"])) if kind == "relpos" else c
    ctx = rng.choice([704, 1024, 2048])
    return dict(kind=kind, layers=rng.choice([8, 28, 30]), hd=rng.choice([64, 128]), heads=8, tokens=min(between(32, 2048), ctx), ctx=ctx,
                kv=rng.choice(["q8_0", "q8_0", "q4_0", "q5_1"]))


# ---- inputs -------------------------------------------------------------------------------------------------------------

class _Random:
    """Seeded normal values on the GPU, as buffers of the storage types."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(int(seed))

    def normal(self, *shape, gain=1.0):
        x = torch.randn(*shape, device="cuda", generator=self.gen)
        return x.mul_(gain) if gain != 1.0 else x

    def shuffled(self, values):
        order = torch.randperm(len(values), generator=self.gen, device="cuda").tolist()
        return [values[i] for i in order]

    def tensor(self, type_, ne, nb=None, gain=1.0):
        """a whole buffer of normal values in a storage type, seen through (ne, nb); dimension 0 is contiguous in it"""
        n = ne[0] * ne[1] * (ne[2] if len(ne) > 2 else 1) * (ne[3] if len(ne) > 3 else 1)
        x = self.normal(n, gain=gain)
        if type_ == ggml.F32:
            return ca.Tensor(x.view(torch.uint8), type_, ne, nb)
        if type_ == ggml.F16:
            return ca.Tensor(x.half().view(torch.uint8), type_, ne, nb)
        flat = ca.Tensor.empty(type_, (n,))
        ca.cpy(ca.Tensor(x.view(torch.uint8), ggml.F32, (n,)), flat)
        return ca.Tensor(flat.buf, type_, ne, nb)


def _thd(type_, hd, n, heads):
    """strides of [batch][token][head][dim] memory seen as [dim, token, head, batch]"""
    rs = ggml.row_size(type_, hd)
    return (ggml.TYPE_SIZE[type_], rs * heads, rs, rs * heads * n)


def _out(hd, heads, n, batch, layers):
    """one F32 buffer for the results of all layers, and each layer's result tensor in it"""
    size = 4 * hd * heads * n * batch
    buf = torch.zeros(size * layers, dtype=torch.uint8, device="cuda")
    return buf.view(torch.float32), [ca.Tensor(buf, ggml.F32, (hd, heads, n, batch), None, il * size) for il in range(layers)]


def _mask(m):
    """a [Bm, Hm, rows, keys] bool tensor, True = visible, as an F16 mask tensor of 0 and -inf"""
    x = torch.zeros(m.shape, dtype=torch.float16, device="cuda").masked_fill_(~m, float("-inf")).contiguous()
    return ca.Tensor(x.view(torch.uint8).reshape(-1), ggml.F16, tuple(reversed(m.shape)))


def _lengths(case, n):
    """lengths from `shortest` to the longest, evenly spread: the same work for every seed"""
    lo, B = case["shortest"], case["batch"]
    return [n - (n - lo) * i // max(1, B - 1) for i in range(B)]


def _cells(case):
    """which cell of a unified cache belongs to whom: -1 the prompt that all beams share, else the beam"""
    own = (case["cells"] - case["prompt"]) // case["beams"]
    return [-1] * case["prompt"] + [b for _ in range(own) for b in range(case["beams"])]


# ---- the cases ------------------------------------------------------------------------------------------------------------

class _Encoder:
    def __init__(self, c, rnd):
        hd, H, N, B, L = c["hd"], c["heads"], c["tokens"], c["batch"], c["layers"]
        self.scale = hd ** -0.5
        F32, F16 = ggml.F32, ggml.F16
        self.q = [rnd.tensor(F32, (hd, N, H, B), _thd(F32, hd, N, H)) for _ in range(L)]
        t = F16 if c["kv"] == "f16" else F32
        self.pad = c["kv"] == "pad"
        if self.pad:             # K and V as the projections leave them: [n_state, tokens]
            self.k = [rnd.tensor(F32, (hd * H, N)) for _ in range(L)]
            self.v = [rnd.tensor(F32, (hd * H, N)) for _ in range(L)]
            rows = (N + 255) // 256 * 256
            bufs = [torch.zeros(2 * hd * H * rows, dtype=torch.uint8, device="cuda") for _ in range(2)]
            self.kp, self.vp = (ca.Tensor(b, F16, (hd, rows, H), _thd(F16, hd, rows, H)) for b in bufs)
            self.kw, self.vw = (ca.Tensor(b, F16, (hd * H, N)) for b in bufs)
        else:
            self.k = [rnd.tensor(t, (hd, N, H, B), _thd(t, hd, N, H)) for _ in range(L)]
            self.v = [rnd.tensor(t, (hd, N, H, B), _thd(t, hd, N, H)) for _ in range(L)]
        self.res, self.out = _out(hd, H, N, B, L)

    def run(self):
        for q, k, v, out in zip(self.q, self.k, self.v, self.out):
            if self.pad:
                ca.cpy(k, self.kw)
                ca.cpy(v, self.vw)
                k, v = self.kp, self.vp
            ca.flash_attn_ext(q, k, v, None, self.scale, out=out)
        return self.res

    @staticmethod
    def work(c):
        hd, H, N, B, L = c["hd"], c["heads"], c["tokens"], c["batch"], c["layers"]
        keys = (N + 255) // 256 * 256 if c["kv"] == "pad" else N
        return L * B * N * hd * H * (4 + 4 + 2 * (2 if c["kv"] == "f16" else 4)), 4.0 * L * B * N * keys * hd * H


class _Cross:
    def __init__(self, c, rnd):
        hd, H, T, N, L = c["hd"], c["heads"], c["tokens"], c["frames"], c["layers"]
        t = TYPES[c["kv"]]
        self.scale = hd ** -0.5
        self.q = [rnd.tensor(ggml.F32, (hd, T, H), _thd(ggml.F32, hd, T, H)) for _ in range(L)]
        self.k = [rnd.tensor(t, (hd, N, H)) for _ in range(L)]
        self.v = [rnd.tensor(t, (hd, N, H)) for _ in range(L)]
        self.res, self.out = _out(hd, H, T, 1, L)

    def run(self):
        for q, k, v, out in zip(self.q, self.k, self.v, self.out):
            ca.flash_attn_ext(q, k, v, None, self.scale, out=out)
        return self.res

    @staticmethod
    def work(c):
        n = c["hd"] * c["heads"] * c["layers"]
        return n * (8 * c["tokens"] + 2 * c["frames"] * ggml.TYPE_SIZE[TYPES[c["kv"]]]), 4.0 * n * c["tokens"] * c["frames"]


class _Whisper:
    HD = 64

    def __init__(self, c, rnd):
        hd, H, T, L, N = self.HD, c["heads"], c["beams"], c["layers"], c["frames"]
        F32, F16 = ggml.F32, ggml.F16
        self.hd, self.H, self.T, self.L = hd, H, T, L
        self.state = hd * H
        owner = torch.tensor(_cells(c), device="cuda")
        self.n_kv = owner.numel()
        self.ctx = self.n_kv + 64                  # the beams' newest cells are the last ones of n_kv
        self.cache_k = rnd.tensor(F16, (self.state, self.ctx, L), gain=hd ** -0.25)
        self.cache_v = rnd.tensor(F16, (self.state, self.ctx, L))
        self.mask = _mask((owner[None, :] < 0) | (owner[None, :] == torch.arange(T, device="cuda")[:, None]))
        self.new_k = [rnd.tensor(F32, (self.state, T), gain=hd ** -0.25) for _ in range(L)]
        self.new_v = [rnd.tensor(F32, (self.state, T)) for _ in range(L)]
        self.q_self = [rnd.tensor(F32, (hd, T, H), _thd(F32, hd, T, H), gain=hd ** -0.25) for _ in range(L)]
        self.q_cross = [rnd.tensor(F32, (hd, T, H), _thd(F32, hd, T, H)) for _ in range(L)]
        # (K is stored with the second half of 1/sqrt(hd) in it)
        self.k_cross = [rnd.tensor(F16, (hd, N, H), _thd(F16, hd, N, H), gain=hd ** -0.25) for _ in range(L)]
        self.v_cross = [rnd.tensor(F16, (hd, N, H), _thd(F16, hd, N, H)) for _ in range(L)]
        self.res_self, self.out_self = _out(hd, H, T, 1, L)
        self.res_cross, self.out_cross = _out(hd, H, T, 1, L)

    def run(self):
        hd, H, T, n_state, n_kv = self.hd, self.H, self.T, self.state, self.n_kv
        nb = (2, 2 * n_state, 2 * hd, 0)
        for il in range(self.L):
            off = 2 * n_state * self.ctx * il
            new = off + 2 * n_state * (n_kv - T)
            ca.cpy(self.new_k[il], self.cache_k.view((n_state * T,), (2, 0, 0, 0), new))
            ca.cpy(self.new_v[il], self.cache_v.view((n_state * T,), (2, 0, 0, 0), new))
            ca.flash_attn_ext(self.q_self[il], self.cache_k.view((hd, n_kv, H), nb, off), self.cache_v.view((hd, n_kv, H), nb, off),
                              self.mask, 1.0, out=self.out_self[il])
            ca.flash_attn_ext(self.q_cross[il], self.k_cross[il], self.v_cross[il], None, hd ** -0.25, out=self.out_cross[il])
        return [self.res_self, self.res_cross, self.cache_k.buf, self.cache_v.buf]

    @classmethod
    def work(cls, c):
        n_state, T, L, N = cls.HD * c["heads"], c["beams"], c["layers"], c["frames"]
        cells = len(_cells(c))
        seen = c["prompt"] * T + (cells - c["prompt"])
        bytes_ = L * n_state * (4 * 4 * T + 2 * (4 + 2) * T + 4 * (cells - T) + 4 * N) + L * 2 * cells * T
        return bytes_, 4.0 * L * n_state * (seen + T * N)


def _write_rows(cache, rows, idx, n_past):
    """K or V rows of new tokens into their cache: a copy into the view behind the rows so far for F16 caches, SET_ROWS for
    quantised ones (as the runtimes' graphs do it)"""
    if idx is None:
        hd, T, heads, _ = rows.ne
        ca.cpy(rows, cache.view((hd, T, heads), cache.nb, n_past * cache.nb[1]))
    else:
        ca.set_rows(cache, rows, idx)


class _Llm:
    """step (one token) and prefill (a prompt), over a [hd, ctx, kv heads, layers] cache"""

    def __init__(self, c, rnd):
        T = c.get("tokens", 1)
        hd, hq, hkv, L, past = c["hd"], c["hq"], c["hkv"], c["layers"], c["past"]
        ctx = c.get("ctx", past + T)
        t = TYPES[c["kv"]]
        rs = ggml.row_size(t, hd)
        self.nb = (ggml.TYPE_SIZE[t], rs, rs * ctx, rs * ctx * hkv)
        self.hd, self.hkv, self.ctx, self.past, self.scale = hd, hkv, ctx, past, hd ** -0.5
        self.n_kv = ctx if c.get("fixed") else past + T
        self.cache_k = rnd.tensor(t, (hd, ctx, hkv, L), self.nb)
        self.cache_v = rnd.tensor(t, (hd, ctx, hkv, L), self.nb)
        rows_nb = _thd(ggml.F32, hd, T, hkv)
        self.new_k = [rnd.tensor(ggml.F32, (hd, T, hkv), rows_nb) for _ in range(L)]
        self.new_v = [rnd.tensor(ggml.F32, (hd, T, hkv), rows_nb) for _ in range(L)]
        self.q = [rnd.tensor(ggml.F32, (hd, T, hq)) for _ in range(L)]
        self.idx = None if t == ggml.F16 else torch.arange(past, past + T, dtype=torch.int64, device="cuda")
        self.mask = None
        if T > 1 or c.get("fixed"):
            key, query = torch.arange(self.n_kv, device="cuda"), torch.arange(T, device="cuda")
            self.mask = _mask(key[None, :] <= query[:, None] + past)
        self.res, self.out = _out(hd, hq, T, 1, L)

    def run(self):
        ne, nb = (self.hd, self.n_kv, self.hkv), self.nb
        for il, out in enumerate(self.out):
            off = il * nb[3]
            for cache, new in ((self.cache_k, self.new_k[il]), (self.cache_v, self.new_v[il])):
                _write_rows(cache.view((self.hd, self.ctx, self.hkv), nb, off), new, self.idx, self.past)
            ca.flash_attn_ext(self.q[il], self.cache_k.view(ne, nb, off), self.cache_v.view(ne, nb, off), self.mask, self.scale, out=out)
        return [self.res, self.cache_k.buf, self.cache_v.buf]

    @staticmethod
    def work(c):
        T, hd, hq, hkv, L, past = c.get("tokens", 1), c["hd"], c["hq"], c["hkv"], c["layers"], c["past"]
        row = ggml.row_size(TYPES[c["kv"]], hd)
        # q and result, new rows in and out, the rows from before, the mask
        bytes_ = L * (8 * T * hd * hq + 2 * hkv * (T * (4 * hd + row) + past * row))
        if T > 1 or c.get("fixed"):
            bytes_ += L * 2 * T * (c["ctx"] if c.get("fixed") else past + T)
        return bytes_, 4.0 * L * hd * hq * (T * past + T * (T + 1) // 2)


class _Batch:
    def __init__(self, c, rnd):
        hd, hq, hkv, B, ctx = c["hd"], c["hq"], c["hkv"], c["batch"], c["ctx"]
        t = TYPES[c["kv"]]
        rs = ggml.row_size(t, hd)
        nb = (ggml.TYPE_SIZE[t], rs, rs * ctx, rs * ctx * hkv)
        self.scale = hd ** -0.5
        n = torch.tensor(rnd.shuffled(_lengths(c, ctx)), device="cuda")
        self.cache_k = rnd.tensor(t, (hd, ctx, hkv, B), nb)
        self.cache_v = rnd.tensor(t, (hd, ctx, hkv, B), nb)
        self.new_k = rnd.tensor(ggml.F32, (hd, 1, hkv, B))
        self.new_v = rnd.tensor(ggml.F32, (hd, 1, hkv, B))
        self.q = rnd.tensor(ggml.F32, (hd, 1, hq, B))
        self.idx = (n - 1).reshape(B, 1, 1)                # every sequence's own position
        self.mask = _mask((torch.arange(ctx, device="cuda")[None, :] < n[:, None])[:, None, None, :])
        self.res, self.out = _out(hd, hq, 1, B, 1)

    def run(self):
        ca.set_rows(self.cache_k, self.new_k, self.idx)
        ca.set_rows(self.cache_v, self.new_v, self.idx)
        ca.flash_attn_ext(self.q, self.cache_k, self.cache_v, self.mask, self.scale, out=self.out[0])
        return [self.res, self.cache_k.buf, self.cache_v.buf]

    @staticmethod
    def work(c):
        hd, hq, hkv, B = c["hd"], c["hq"], c["hkv"], c["batch"]
        row, seen = ggml.row_size(TYPES[c["kv"]], hd), sum(_lengths(c, c["ctx"]))
        return B * (8 * hd * hq + 2 * hkv * 4 * hd + 2 * c["ctx"]) + 2 * hkv * row * seen, 4.0 * hd * hq * seen


class _Bias:
    def __init__(self, c, rnd):
        hd, H, T, B = c["hd"], c["heads"], c["tokens"], c["batch"]
        t = TYPES[c["kv"]]
        self.scale = hd ** -0.5
        self.q = rnd.tensor(ggml.F32, (hd, T, H, B), _thd(ggml.F32, hd, T, H))
        self.k, self.v = (rnd.tensor(t, (hd, T, H, B), _thd(t, hd, T, H)) for _ in range(2))
        n = torch.tensor(rnd.shuffled(_lengths(c, T)), device="cuda")
        unseen = torch.arange(T, device="cuda")[None, None, None, :] >= n[:, None, None, None]
        m = rnd.normal(B, H, T, T, gain=0.5).masked_fill_(unseen, float("-inf")).half()
        self.mask = ca.Tensor(m.view(torch.uint8).reshape(-1), ggml.F16, (T, T, H, B))
        self.res, self.out = _out(hd, H, T, B, 1)

    def run(self):
        ca.flash_attn_ext(self.q, self.k, self.v, self.mask, self.scale, out=self.out[0])
        return self.res

    @staticmethod
    def work(c):
        hd, H, T, B = c["hd"], c["heads"], c["tokens"], c["batch"]
        seen = sum(_lengths(c, T))
        return hd * H * (8 * T * B + 2 * ggml.TYPE_SIZE[TYPES[c["kv"]]] * seen) + 2 * T * T * H * B, 4.0 * hd * H * T * seen


class _Relpos:
    def __init__(self, c, rnd):
        hd, H, T, B = c["hd"], c["heads"], c["tokens"], c["batch"]
        F32, t = ggml.F32, TYPES[c["kv"]]
        self.scale = hd ** -0.5
        # (content and position terms of std 0.7 each: scores of unit variance)
        self.qu, self.qv = (rnd.tensor(F32, (hd, T, H, B), _thd(F32, hd, T, H), gain=0.7) for _ in range(2))
        self.k, self.v = (rnd.tensor(t, (hd, T, H, B), _thd(t, hd, T, H)) for _ in range(2))
        if c["table"] == "f32":          # the position projection's output as it is
            self.r = rnd.tensor(F32, (hd, 2 * T - 1, H), _thd(F32, hd, 2 * T - 1, H))
        else:                            # rounded once for this length, rows contiguous
            self.r = rnd.tensor(ggml.F16, (hd, 2 * T - 1, H))
        n = torch.tensor(rnd.shuffled(_lengths(c, T)), device="cuda")
        seen = (torch.arange(T, device="cuda")[None, None, None, :] < n[:, None, None, None]).expand(B, 1, T, T)
        add = torch.zeros(B, 1, T, T, device="cuda").masked_fill_(~seen, float("-inf"))
        self.add = ca.Tensor(add.view(torch.uint8).reshape(-1), F32, (T, T, 1, B))
        self.res, self.out = _out(hd, H, T, B, 1)

    def run(self):
        ggml.flash_attn_relpos(self.qu, self.qv, self.k, self.v, self.r, self.add, self.scale, out=self.out[0])
        return self.res

    @staticmethod
    def work(c):
        hd, H, T, B = c["hd"], c["heads"], c["tokens"], c["batch"]
        lengths = _lengths(c, T)
        es = ggml.TYPE_SIZE[TYPES[c["kv"]]]
        bytes_ = hd * H * (12 * T * B + 2 * es * sum(lengths) + (2 * T - 1) * ggml.TYPE_SIZE[TYPES[c["table"]]]) + 4 * T * T * B
        return bytes_, 6.0 * hd * H * T * sum(lengths)


class _KvCast:
    def __init__(self, c, rnd):
        hd, H, N, L, ctx, t = c["hd"], c["heads"], c["tokens"], c["layers"], c["ctx"], TYPES[c["kv"]]
        rs = ggml.row_size(t, hd)
        nb = (ggml.TYPE_SIZE[t], rs, rs * ctx, rs * ctx * H)
        caches = [rnd.tensor(t, (hd, ctx, H, L), nb) for _ in range(2)]
        self.src = [caches[i % 2].view((hd, N, H), nb, (i // 2) * nb[3]) for i in range(2 * L)]
        nbytes = 4 * hd * N * H
        buf = torch.zeros(nbytes * 2 * L, dtype=torch.uint8, device="cuda")
        self.res = buf.view(torch.float32)
        self.dst = [ca.Tensor(buf, ggml.F32, (hd, N, H), None, i * nbytes) for i in range(2 * L)]

    def run(self):
        for src, dst in zip(self.src, self.dst):
            ca.cpy(src, dst)
        return self.res

    @staticmethod
    def work(c):
        n = 2 * c["layers"] * c["tokens"] * c["heads"]
        return n * (4 * c["hd"] + ggml.row_size(TYPES[c["kv"]], c["hd"])), 0.0


KINDS = {"encoder": _Encoder, "cross": _Cross, "whisper": _Whisper, "step": _Llm, "prefill": _Llm, "batch": _Batch, "bias": _Bias,
         "relpos": _Relpos, "kv_cast": _KvCast}


def prepare(case, seed):
    return KINDS[case["kind"]](case, _Random(seed))


def run(state):
    return state.run()


def work(case):
    bytes_, flops = KINDS[case["kind"]].work(case)
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    # copies are exact, and so are the caches' bytes ("differ" 0); attention rounds its probabilities and its F32 or dequantised operands to f16
    if case["kind"] == "kv_cast":
        return "exact"
    if case["kind"] == "cross" and case["hd"] % 8:        # head sizes outside the matrix cores' forms: F32 throughout
        return {"rel": 1e-5, "max": 1e-3}
    return {"rel": 1e-3, "max": 0.02}
