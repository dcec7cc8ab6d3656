"""What this framework is timed on: attention over the paged KV cache, the
cache's own writes, and the model calls built on both, each through the entry
points that a program calls (``tvara_amd.kv``, ``tvara_amd.attention``,
``tvara_amd.native``).

``listed()`` names the cases and ``draw()`` gives others of the same ranges.
A case is a plain dict; its sequences' lengths follow from its own fields, so
they are the same for every seed, while every value that is computed on follows
from the seed.  Five kinds:

decode   one ``DecodePlan.launch``: a generated token of every sequence of a
         batch attends to that sequence's cached tokens in one layer.
chunk    one ``PrefillPlan.launch``: a prompt chunk of every sequence attends
         causally to what is cached and to itself in one layer.
step     the cache and attention work of one whole generation step: append a
         token to every sequence for all layers, plan, launch every layer; the
         step is rolled back (a rejected speculative token).
tokens   one model call that advances every listed sequence by a token and
         returns the logits; rolled back likewise.
prompt   one model call that takes a prompt in and returns its last logits;
         rolled back likewise.

The plans are kept between passes as a serving loop keeps them over the layers
of a step (kinds decode and chunk); the step kind makes its own each pass,
since the append outdates it.
"""

import math
import os
import random
import shutil
import tempfile
import zlib

import numpy as np
import torch

from tvara_amd import attention, gguf_writer, kv, native

CONTEXT = 1 << 20
DEVICE = "cuda"

# (query heads, KV heads, head_dim) of the attention layers in use here:
# SmolLM2-135M, Llama-3.2-1B, Llama-3-8B, Llama-3-70B, TinyLlama-1.1B
SMOL, L1B, L8B, L70B, TINY = (9, 3, 64), (32, 8, 64), (32, 8, 128), (64, 8, 128), (32, 4, 64)


def _shape(s):
    return {"heads": s[0], "kv_heads": s[1], "dim": s[2]}


def listed():
    return [
        # one user's stream on a small model: the smallest call, launch-bound;
        # the token's own K/V ride along as the tail, as in a decode step
        {"name": "decode-smol-1x512", "kind": "decode", **_shape(SMOL), "n": 1, "low": 512, "high": 512,
         "block": 16, "q8": False, "tail": True, "spread": 1},
        # a serving batch of unequal contexts in f32 blocks
        {"name": "decode-1b-64-ragged", "kind": "decode", **_shape(L1B), "n": 64, "low": 128, "high": 4096,
         "block": 16, "q8": False, "tail": False, "spread": 2},
        # a mid-sized batch of a wide-GQA model over quantised blocks
        {"name": "decode-70b-q8-16", "kind": "decode", **_shape(L70B), "n": 16, "low": 2048, "high": 6144,
         "block": 16, "q8": True, "tail": False, "spread": 3},
        # long contexts over quantised blocks: the largest decode
        {"name": "decode-8b-q8-16x32k", "kind": "decode", **_shape(L8B), "n": 16, "low": 32768, "high": 32768,
         "block": 16, "q8": True, "tail": False, "spread": 4},
        # one generation step of 32 sequences: append, plan, 16 layers
        {"name": "step-1b-32x16-layers", "kind": "step", **_shape(L1B), "n": 32, "low": 64, "high": 1024,
         "layers": 16, "block": 16, "q8": False, "spread": 5},
        # chunked prefill on the bf16 tiles: eight users' 512-token chunks
        {"name": "chunk-1b-bf16-8x512", "kind": "chunk", **_shape(L1B), "n": 8, "plow": 2048, "phigh": 2048,
         "clow": 512, "chigh": 512, "block": 16, "q8": False, "precision": "bf16", "spread": 6},
        # the default precision (the reference's arithmetic), prompts and
        # prefixes of unequal, odd lengths
        {"name": "chunk-1b-f32-ragged", "kind": "chunk", **_shape(L1B), "n": 6, "plow": 0, "phigh": 2047,
         "clow": 33, "chigh": 700, "block": 16, "q8": False, "precision": "f32", "spread": 7},
        # f32 accuracy on the tiles, at head_dim 128
        {"name": "chunk-8b-f32x3-ragged", "kind": "chunk", **_shape(L8B), "n": 4, "plow": 500, "phigh": 3000,
         "clow": 200, "chigh": 900, "block": 16, "q8": False, "precision": "f32x3", "spread": 8},
        # a long document continued over quantised blocks of 64 tokens
        {"name": "chunk-8b-q8-bf16-long", "kind": "chunk", **_shape(L8B), "n": 2, "plow": 12000, "phigh": 16000,
         "clow": 1000, "chigh": 1024, "block": 64, "q8": True, "precision": "bf16", "spread": 9},
        # the whole model (Llama-3.2-1B shape, Q8_0 weights): one user's token
        {"name": "model-1b-token", "kind": "tokens", "n": 1, "low": 512, "high": 512, "spread": 10},
        # ... a batch of users' tokens
        {"name": "model-1b-64-tokens", "kind": "tokens", "n": 64, "low": 32, "high": 480, "spread": 11},
        # ... and a long prompt
        {"name": "model-1b-prompt-2048", "kind": "prompt", "prefix": 0, "tokens": 2048},
    ]


def _log(rng, low, high):
    """An integer from low to high, evenly over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "chunk", "chunk", "chunk", "step", "tokens", "prompt"])
    spread = rng.randrange(1 << 30)
    if kind == "tokens":
        low = _log(rng, 1, 256)
        return {"kind": kind, "n": _log(rng, 1, 64), "low": low, "high": low + _log(rng, 1, 224), "spread": spread}
    if kind == "prompt":
        return {"kind": kind, "prefix": rng.choice([0, _log(rng, 1, 1024)]), "tokens": _log(rng, 2, 2048)}
    block = rng.choice([16, 16, 16, 32, 64])
    if kind == "step":
        shape = rng.choice([SMOL, L1B, TINY])
        low = _log(rng, 1, 256)
        return {"kind": kind, **_shape(shape), "n": _log(rng, 1, 48), "low": low, "high": low + _log(rng, 1, 600),
                "layers": rng.randrange(2, 17), "block": block, "q8": rng.random() < 0.3, "spread": spread}
    q8 = rng.random() < 0.4
    if kind == "decode":
        heads, kvh, dim = rng.choice([SMOL, L1B, L1B, L8B, L8B, L70B, TINY])
        # total cached tokens from a few hundred to what the largest listed case reads
        per_token = 2 * kvh * dim * (34 / 32 if q8 else 4)
        n = _log(rng, 1, 64)
        mean = _log(rng, 16, max(17, min(32768, int(1.1e9 / per_token / n))))
        low = max(1, int(mean * rng.choice([1.0, 0.5, 0.1])))
        return {"kind": kind, "heads": heads, "kv_heads": kvh, "dim": dim, "n": n, "low": low,
                "high": max(low, 2 * mean - low), "block": block, "q8": q8, "tail": rng.random() < 0.3,
                "spread": spread}
    heads, kvh, dim = rng.choice([SMOL, L1B, L1B, L8B, L8B, TINY])
    precision = rng.choice(["bf16", "f32", "f32x3"])
    n = _log(rng, 1, 8)
    chunk = _log(rng, 16, 1024)
    most = 60e9 if precision == "f32" else 200e9  # flops of the largest drawn chunk
    reach = most / (4 * dim * heads * n * chunk) - chunk / 2
    prefix = min(int(reach), rng.choice([0, _log(rng, 1, 16000)]))
    while prefix < 0:
        chunk, prefix = chunk // 2, 0
        if most / (4 * dim * heads * n * chunk) < chunk / 2:
            prefix = -1
    low, clow = int(prefix * rng.uniform(0, 1)), max(1, int(chunk * rng.uniform(0.3, 1)))
    return {"kind": kind, "heads": heads, "kv_heads": kvh, "dim": dim, "n": n, "plow": low, "phigh": prefix,
            "clow": clow, "chigh": chunk, "block": block, "q8": q8, "precision": precision, "spread": spread}


# ------------------------------------------------------------------ sizes

def _lengths(case, low="low", high="high", tag=0):
    r = random.Random(case["spread"] * 4 + tag)
    return [r.randint(case[low], case[high]) for _ in range(case["n"])]


def _cached(case):
    """Cached tokens per sequence when the call is made."""
    if case["kind"] == "chunk":
        return [p + c for p, c in zip(*_chunks(case))]
    return _lengths(case)


def _chunks(case):
    return _lengths(case, "plow", "phigh", 1), _lengths(case, "clow", "chigh", 2)


def work(case):
    kind = case["kind"]
    if kind in ("tokens", "prompt"):
        s = _SPEC
        kvw = s.hidden // s.heads * s.kv_heads
        layer = s.hidden * (2 * s.hidden + 2 * kvw) + 3 * s.hidden * s.intermediate
        head = s.vocab * s.hidden
        weights = (layer * s.layers + head) * 34 / 32
        if kind == "tokens":
            ctx = _lengths(case)
            kvb = sum(ctx) * s.layers * kvw * 2 * 4
            return {"bytes": weights + kvb + case["n"] * s.vocab * 4,
                    "flops": 2 * case["n"] * (layer * s.layers + head) + 4 * s.hidden * s.layers * sum(c + 1 for c in ctx)}
        p, t = case["prefix"], case["tokens"]
        pairs = t * p + t * (t + 1) // 2
        return {"bytes": weights + (p + 2 * t) * s.layers * kvw * 2 * 4 + s.vocab * 4,
                "flops": 2 * t * layer * s.layers + 2 * head + 4 * s.hidden * s.layers * pairs}
    hidden, kvw = case["heads"] * case["dim"], case["kv_heads"] * case["dim"]
    element = 34 / 32 if case["q8"] else 4
    if kind == "chunk":
        pre, chunk = _chunks(case)
        pairs = sum(c * p + c * (c + 1) // 2 for p, c in zip(pre, chunk))
        return {"bytes": sum(_cached(case)) * 2 * kvw * element + 2 * sum(chunk) * hidden * 4, "flops": 4 * hidden * pairs}
    tail = int(bool(case.get("tail")))
    ctx = _lengths(case)
    layers = case.get("layers", 1)
    one = sum(ctx) * 2 * kvw * element + case["n"] * (2 * hidden + 2 * tail * kvw) * 4
    if kind == "step":  # the appended token is read from the batch, written, and read back by the attention
        one += case["n"] * 2 * kvw * (4 + 2 * element)
        tail = 1
    return {"bytes": layers * one, "flops": layers * 4 * hidden * sum(c + tail for c in ctx)}


# Relative errors (2-norm) against exact(), measured on an MI355X when these
# cases were written: f32 attention 1e-7 to 4.3e-7, the three-product tiles
# 4.3e-6, the bf16 tiles 4.0e-3 to 5.4e-3, the model 6.7e-6 to 7.4e-6 (tokens)
# and 1.5e-5 (prompts: their attention runs on the three-product tiles).  Another
# correct order of the same sums stays within about four times that.
def tolerance(case):
    if case["kind"] in ("tokens", "prompt"):
        return {"rel": 6e-5, "max": 1e-3}
    if case["kind"] == "chunk" and case["precision"] == "bf16":
        return {"rel": 1.5e-2, "max": 2e-1}
    if case["kind"] == "chunk" and case["precision"] == "f32x3":
        return {"rel": 3e-5, "max": 6e-4}
    return {"rel": 2e-6, "max": 4e-5}


# ------------------------------------------------------------- attention data

def _gen(seed, *tags):
    g = torch.Generator(device=DEVICE)
    g.manual_seed((int(seed) * 1000003 + zlib.crc32(repr(tags).encode())) % (1 << 62))
    return g


def _kv_rows(case, seed, which, rows, layers=1):
    """[rows, layers * kv_width]: normal, each channel at a scale of its own."""
    w = layers * case["kv_heads"] * case["dim"]
    g = _gen(seed, which)
    scale = torch.exp(0.4 * torch.randn(w, generator=g, device=DEVICE)) if which.endswith("k") else 1.0
    return torch.randn(rows, w, generator=g, device=DEVICE) * scale


def _queries(case, seed, rows, layers=1):
    """[layers, rows, heads * head_dim]"""
    return 1.5 * torch.randn(layers, rows, case["heads"] * case["dim"], generator=_gen(seed, "q"), device=DEVICE)


def _append_order(case, lengths):
    """(sequence, token) of every append: blocks of the sequences in turn, as
    sequences that grow side by side take them from the pool."""
    r = np.random.default_rng(case["spread"])
    seq, tok = [], []
    b = case["block"]
    for lo in range(0, max(lengths, default=0), b):
        live = np.array([i for i, n in enumerate(lengths) if n > lo], dtype=np.int64)
        for i in r.permutation(live):
            t = np.arange(lo, min(lo + b, lengths[i]))
            seq.append(np.full(t.size, i))
            tok.append(t)
    return (np.concatenate(seq), np.concatenate(tok)) if seq else (np.zeros(0, int), np.zeros(0, int))


class _State:
    pass


def _fill(case, seed, layers=1):
    """The cache with every sequence's tokens appended."""
    lengths = _cached(case)
    total = sum(lengths)
    blocks = sum(-(-n // case["block"]) + 2 for n in lengths) + 8
    st = _State()
    st.cache = kv.PagedCache(layers, case["kv_heads"], case["dim"], case["block"], blocks,
                             kv.Q8_0 if case["q8"] else kv.F32)
    st.seqs = np.array([st.cache.create_sequence() for _ in lengths], dtype=np.uint64)
    if total:
        seq, tok = _append_order(case, lengths)
        first = np.concatenate([[0], np.cumsum(lengths)[:-1]])
        rows = torch.from_numpy(first[seq] + tok).to(DEVICE)
        k, v = (_kv_rows(case, seed, which, total, layers)[rows] for which in ("k", "v"))
        ids = st.seqs[seq]
        for lo in range(0, total, 1 << 16):
            part = np.ascontiguousarray(ids[lo:lo + (1 << 16)])
            st.cache.append_batch_device(part, k[lo:].data_ptr(), v[lo:].data_ptr())
        st.cache.synchronize()
    st.lengths = np.array(lengths, dtype=np.uintp)
    return st


# ----------------------------------------------------------------- the model

_SPEC = gguf_writer.llama32_1b()
_MODEL = []
_POOL_BLOCKS = 12288


def _weight_seed(name):
    return _gen(_SPEC.seed, "weight", name)


def _weight(name, rows, cols):
    """(fp16 scales [rows, cols/32], int8 [rows, cols/32, 32]) of a matrix."""
    g = _weight_seed(name)
    d = (1 / math.sqrt(cols) / 64 * (0.5 + torch.rand(rows, cols // 32, generator=g, device=DEVICE))).half()
    q = torch.randint(-127, 128, (rows, cols // 32, 32), generator=g, device=DEVICE, dtype=torch.int8)
    return d, q


def _norm(name):
    return 1.0 + 0.1 * torch.randn(_SPEC.hidden, generator=_weight_seed(name), device=DEVICE)


def _tensors():
    out = []
    for name, dims, kind, _ in _SPEC.tensors():
        if kind == gguf_writer.T_F32:
            out.append((name, dims, kind, _norm(name).cpu().numpy().tobytes()))
            continue
        cols, rows = dims

        def make(name=name, rows=rows, cols=cols):
            d, q = _weight(name, rows, cols)
            raw = torch.cat([d.view(torch.uint8).reshape(rows, cols // 32, 2), q.view(torch.uint8)], 2)
            return raw.cpu().numpy().tobytes()

        out.append((name, dims, kind, gguf_writer.Lazy(rows * cols // 32 * 34, make)))
    return out


def _model():
    """The loaded checkpoint, one for all requests, as a server holds it."""
    if not _MODEL:
        folder = tempfile.mkdtemp(prefix="tvara-cases-")
        try:
            path = os.path.join(folder, "model.gguf")
            gguf_writer.write_gguf(path, _SPEC.metadata(), _tensors())
            _MODEL.append(native.NativeModel(path, max_blocks=_POOL_BLOCKS, block_tokens=16))
        finally:
            shutil.rmtree(folder, ignore_errors=True)
    return _MODEL[0]


class _Requests(_State):
    """The sequences that a server holds for its requests; dropped with it."""

    def __init__(self, model, count):
        self.model, self.seqs = model, []
        for _ in range(count):
            self.seqs.append(model.new_sequence())

    def __del__(self):
        for s in self.seqs:
            self.model.drop_sequence(s)


def _ids(seed, tag, n):
    return torch.randint(0, _SPEC.vocab, (n,), generator=_gen(seed, "ids", tag), device=DEVICE).cpu().numpy()


# ----------------------------------------------------------------- the calls

def prepare(case, seed):
    kind = case["kind"]
    if kind in ("tokens", "prompt"):
        m = _model()
        before = _lengths(case) if kind == "tokens" else [case["prefix"]]
        st = _Requests(m, len(before))
        for i, (s, n) in enumerate(zip(st.seqs, before)):
            if n:
                m.prefill(s, _ids(seed, i, n))
        st.kind = kind
        st.cache = m.cache()
        st.ids = np.array(st.seqs, dtype=np.uint64)
        st.lengths = np.array(before, dtype=np.uintp)
        st.tokens = _ids(seed, "next", case["n"] if kind == "tokens" else case["tokens"]).astype(np.uint32)
        return st
    layers = case.get("layers", 1)
    st = _fill(case, seed, layers)
    st.kind, st.layers, st.heads = kind, layers, case["heads"]
    if kind == "chunk":
        pre, chunk = _chunks(case)
        st.q = _queries(case, seed, sum(chunk))[0].contiguous()
        st.plan = attention.PrefillPlan(st.cache, st.seqs, pre, chunk, case["heads"], CONTEXT, case["precision"])
    else:
        st.q = _queries(case, seed, case["n"], layers)
        st.k, st.v = (_kv_rows(case, seed, which, case["n"], layers) for which in ("tk", "tv"))
        st.tail = bool(case.get("tail"))
        if kind == "decode":
            st.plan = attention.DecodePlan(st.cache, st.seqs, case["heads"], CONTEXT, with_tail=st.tail)
    st.out = torch.empty_like(st.q)
    return st


def run(st):
    if st.kind == "decode":
        tk, tv = (st.k.data_ptr(), st.v.data_ptr()) if st.tail else (None, None)
        st.plan.launch(0, st.q.data_ptr(), st.out.data_ptr(), tk, tv)
        return st.out
    if st.kind == "chunk":
        st.plan.launch(0, st.q.data_ptr(), st.out.data_ptr())
        return st.out
    if st.kind == "step":
        st.cache.append_batch_device(st.seqs, st.k.data_ptr(), st.v.data_ptr())
        plan = attention.DecodePlan(st.cache, st.seqs, st.heads, CONTEXT)
        for layer in range(st.layers):
            plan.launch(layer, st.q[layer].data_ptr(), st.out[layer].data_ptr())
        st.cache.truncate_batch(st.seqs, st.lengths)
        return st.out
    if st.kind == "tokens":
        if len(st.seqs) == 1:
            logits = st.model.logits(st.seqs[0], int(st.tokens[0]))
        else:
            logits = st.model.decode_sequences(st.ids, st.tokens)
    else:
        logits = st.model.prefill(st.seqs[0], st.tokens)
    st.cache.truncate_batch(st.ids, st.lengths)
    return logits


# ------------------------------------------------------------ in 64 bits

def _stored(x, q8):
    """What the cache holds of f32 values, as float64: Q8_0 blocks hold int8
    times an fp16 scale per 32 (scale max|x| / 127, quotients by that scale in
    f32 rounded to even)."""
    if not q8:
        return x.double()
    g = x.reshape(*x.shape[:-1], -1, 32)
    scale = g.abs().amax(-1, keepdim=True).double() / 127
    s32 = scale.float()
    q = torch.where(s32 > 0, torch.round(g / torch.where(s32 > 0, s32, 1.0)), 0.0).clamp(-127, 127)
    return (q.double() * scale.half().double()).reshape(x.shape)


def _attend(q, k, v, first):
    """q [rows, heads, d] over k, v [tokens, kv_heads, d]; row i sees tokens
    0 .. first + i (all in float64)."""
    rows, heads, d = q.shape
    kvh = k.shape[1]
    kt, vt = k.permute(1, 2, 0).contiguous(), v.permute(1, 0, 2).contiguous()
    out = torch.empty_like(q)
    part = max(1, (1 << 27) // (heads * k.shape[0]))
    col = torch.arange(k.shape[0], device=q.device)
    for lo in range(0, rows, part):
        qq = q[lo:lo + part]
        n = qq.shape[0]
        g = qq.reshape(n, kvh, heads // kvh, d).permute(1, 2, 0, 3).reshape(kvh, -1, d).contiguous()
        s = torch.matmul(g, kt) / math.sqrt(d)
        seen = col[None, :] <= (first + lo + torch.arange(n, device=q.device))[:, None]
        s = s.reshape(kvh, heads // kvh, n, -1).masked_fill(~seen, -math.inf)
        p = torch.softmax(s, -1).reshape(kvh, -1, k.shape[0])
        o = torch.matmul(p, vt).reshape(kvh, heads // kvh, n, d)
        out[lo:lo + n] = o.permute(2, 0, 1, 3).reshape(n, heads, d)
    return out


def _exact_attention(case, seed):
    lengths, layers = _cached(case), case.get("layers", 1)
    heads, kvh, d = case["heads"], case["kv_heads"], case["dim"]
    kind, kvw = case["kind"], kvh * d
    total = sum(lengths)
    k, v = _kv_rows(case, seed, "k", total, layers), _kv_rows(case, seed, "v", total, layers)
    if kind == "chunk":
        pre, chunk = _chunks(case)
    else:
        pre, chunk = lengths, [1] * case["n"]
    q = _queries(case, seed, sum(chunk), layers)
    extra = kind == "step" or case.get("tail")
    if kind != "chunk":
        tk, tv = (_kv_rows(case, seed, which, case["n"], layers) for which in ("tk", "tv"))
    out = torch.empty(q.shape, dtype=torch.float64, device=DEVICE)
    for layer in range(layers):
        cols = slice(layer * kvw, (layer + 1) * kvw)
        t0 = r0 = 0
        for i, n in enumerate(lengths):
            kk, vv = (_stored(x[t0:t0 + n, cols], case["q8"]) for x in (k, v))
            if extra:
                # an appended token is stored in the cache's form, a tail is not
                more = [_stored(x[i:i + 1, cols], case["q8"] and kind == "step") for x in (tk, tv)]
                kk, vv = torch.cat([kk, more[0]]), torch.cat([vv, more[1]])
            qq = q[layer, r0:r0 + chunk[i]].double().reshape(-1, heads, d)
            first = pre[i] if kind == "chunk" else kk.shape[0] - 1
            out[layer, r0:r0 + chunk[i]] = _attend(qq, kk.reshape(-1, kvh, d), vv.reshape(-1, kvh, d), first).reshape(
                chunk[i], -1)
            t0, r0 = t0 + n, r0 + chunk[i]
    return out[0] if kind != "step" and layers == 1 else out


def _exact_model(case, seed):
    s = _SPEC
    d, kvh = s.hidden // s.heads, s.kv_heads
    if case["kind"] == "tokens":
        before = _lengths(case)
        nxt = _ids(seed, "next", case["n"])
        runs = [np.append(_ids(seed, i, n) if n else np.zeros(0, int), nxt[i]) for i, n in enumerate(before)]
    else:
        runs = [np.concatenate([_ids(seed, 0, case["prefix"]) if case["prefix"] else np.zeros(0, int),
                                _ids(seed, "next", case["tokens"])])]

    def matrix(name, rows, cols):
        sc, q = _weight(name, rows, cols)
        return (q.double() * sc.double()[:, :, None]).reshape(rows, cols)

    def norm(x, name):
        return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + s.rms_epsilon) * _norm(name).double()

    ids = torch.from_numpy(np.concatenate(runs).astype(np.int64)).to(DEVICE)
    pos = np.concatenate([np.arange(len(r)) for r in runs]).astype(np.float32)
    # the angle is defined in f32: position / theta^(2i/d)
    freq = np.power(float(s.rope_theta), (2 * np.arange(d // 2) / d).astype(np.float32).astype(np.float64))
    angle = torch.from_numpy((pos[:, None] / freq.astype(np.float32)[None, :]).astype(np.float64)).to(DEVICE)
    cos, sin = torch.cos(angle)[:, None], torch.sin(angle)[:, None]

    def rope(x):  # pairs (2i, 2i + 1)
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([a * cos - b * sin, b * cos + a * sin], -1).reshape(x.shape)

    embedding = matrix("token_embd.weight", s.vocab, s.hidden)
    x = embedding[ids]
    for layer in range(s.layers):
        p = "blk.%d." % layer
        h = norm(x, p + "attn_norm.weight")
        q = rope((h @ matrix(p + "attn_q.weight", s.hidden, s.hidden).T).reshape(-1, s.heads, d))
        k = rope((h @ matrix(p + "attn_k.weight", kvh * d, s.hidden).T).reshape(-1, kvh, d))
        v = (h @ matrix(p + "attn_v.weight", kvh * d, s.hidden).T).reshape(-1, kvh, d)
        a, at = torch.empty_like(q), 0
        for r in runs:
            part = slice(at, at + len(r))
            a[part] = _attend(q[part], k[part], v[part], 0)
            at += len(r)
        x = x + a.reshape(x.shape) @ matrix(p + "attn_output.weight", s.hidden, s.hidden).T
        h = norm(x, p + "ffn_norm.weight")
        gate = h @ matrix(p + "ffn_gate.weight", s.intermediate, s.hidden).T
        gate = gate * torch.sigmoid(gate)
        gate *= h @ matrix(p + "ffn_up.weight", s.intermediate, s.hidden).T
        x = x + gate @ matrix(p + "ffn_down.weight", s.hidden, s.intermediate).T
        del gate
    last = torch.from_numpy(np.cumsum([len(r) for r in runs]) - 1).to(DEVICE)
    logits = norm(x[last], "output_norm.weight") @ embedding.T
    return logits[0] if case["kind"] == "prompt" or case["n"] == 1 else logits


def exact(case, seed):
    """run()'s answer in plain torch, in 64 bits."""
    return (_exact_model if case["kind"] in ("tokens", "prompt") else _exact_attention)(case, seed)
