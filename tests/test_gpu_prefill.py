"""Paged chunked-prefill attention on the GPU against the oracle's
fused_prompt_attention (attention.hpp:85-89, FP64).

f32 path: |gpu - ref| <= 1e-4 * (1 + |ref|).

f32x3 path (the MFMA tiles with every operand split as hi + lo and three
products, hi*hi + hi*lo + lo*hi): the score operands q*log2(e)/sqrt(d) and K
as fp16 parts (22 significant bits), V and the probabilities as bf16 parts
(16 bits), the dropped lo*lo term below 2^-16 of its product, so every
rounding term below shrinks by 2^7 or more against the bf16 path: the
short-row worst case becomes ~8e-2 / 128 ~ 6e-4 at |ref| ~ 5, within the f32
bar's 1e-4 * (1 + |ref|), and the long rows sit two orders below it.  The
f32 bar applies.

bf16 MFMA path.  q*log2(e)/sqrt(d), K, V and the probabilities P are rounded
to bf16 (unit roundoff u = 2^-9); products and sums are f32.  To first order
the output error of one row is
    sum_t w_t * (dv_t + v_t * dp_t + (v_t - o) * ds_t)
with |dv_t| <= u|v_t|, |dp_t| <= u, and a score error ds_t (natural-log units)
that is a sum of d independent rounding terms, so its standard deviation is
    sigma_s = u / sqrt(3) * sqrt(2 * sum_i (q_i k_i)^2) / sqrt(d)  ~ 2^-9 * 0.8
for N(0,1) inputs at d = 64.  The three terms are independent across keys:
  * a row with few visible keys keeps them whole: with |v| <= 5 (the largest of
    ~10^6 N(0,1) draws) and |v - o| <= 10, a 4-sigma score error gives
    10 * 4 * 1.6e-3 + 2 * 5 * u ~ 8e-2 in the worst element, and the batch RMS
    is ~ |v| * sigma_s ~ 2e-3;
  * a row of the chunked-prefill shape sees >= 2,049 keys; N(0,1) scores give
    n_eff = n / e >= 750 effective keys, so every term shrinks by
    1/sqrt(n_eff) < 0.04: the worst element stays below 1e-2 and the RMS below
    1e-3.
Bars: short rows  max |gpu - ref| <= 8e-2 * (1 + |ref|), RMS <= 2e-3;
      long rows   max |gpu - ref| <= 1e-2 * (1 + |ref|), RMS <= 1e-3.
"""

import sys

import numpy as np
import pytest

import refmath
from tvara_amd import attention, synth, workloads

pytestmark = pytest.mark.gpu
TOL_F32 = 1e-4
SHORT_ROWS = (8e-2, 2e-3)
LONG_ROWS = (1e-2, 1e-3)


def say(*a):
    print(*a, flush=True, file=sys.stderr)


def bf16_ok(got, want, bars):
    d = np.asarray(got, np.float64) - np.asarray(want, np.float64)
    rms = float(np.sqrt(np.mean(d * d)))
    return refmath.close(got, want, bars[0]) and rms <= bars[1], (refmath.max_rel(got, want), rms)


def build(device, oracle, heads, kv_heads, dim, specs, seed, tpb=16, q8=False):
    """specs: (cached tokens, chunk start, chunk rows) per sequence.  q8: Q8_0
    blocks, with the oracle holding the dequantised values."""
    nb = sum((n + tpb - 1) // tpb for n, _, _ in specs) + 4
    dev = device.PagedCache(1, kv_heads, dim, tpb, nb, fmt=device.Q8_0 if q8 else device.F32)
    ref = oracle.Cache(1, kv_heads, dim, tpb, nb)
    w = kv_heads * dim
    ds, rs, qs = [], [], []
    for i, (n, start, rows) in enumerate(specs):
        k = synth.normal(seed, f"k{i}", n * w).reshape(n, w)
        v = synth.normal(seed, f"v{i}", n * w).reshape(n, w)
        if q8:
            k = oracle.dequantize_q8_0(oracle.quantize_q8_0(k)).reshape(n, w)
            v = oracle.dequantize_q8_0(oracle.quantize_q8_0(v)).reshape(n, w)
        sd, sr = dev.create_sequence(), ref.create_sequence()
        dev.append_many(sd, k, v)
        ref.append_many(sr, k, v)
        ds.append(sd)
        rs.append(sr)
        qs.append(synth.normal(seed, f"q{i}", rows * heads * dim).reshape(rows, heads * dim))
    return dev, ref, ds, rs, qs


@pytest.mark.parametrize("fmt", ["f32", "q8_0"])
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("group", [1, 2, 3, 4, 5, 6, 7, 8, 10, 16])  # 10, 16: slices of 5 and 8 heads
def test_bf16_small_shapes(device, oracle, group, dim, fmt):
    heads, kv_heads = 2 * group, 2
    specs = [(137, 100, 37), (64, 0, 64), (20, 3, 17)]
    say("prefill bf16 group", group, "dim", dim, fmt)
    dev, ref, ds, rs, qs = build(device, oracle, heads, kv_heads, dim, specs, seed=group, q8=fmt == "q8_0")
    starts = [s for _, s, _ in specs]
    counts = [r for _, _, r in specs]
    got = attention.prefill_batch(dev, np.concatenate(qs), ds, starts, counts, 0, heads, 4096, precision="bf16")
    f32 = attention.prefill_batch(dev, np.concatenate(qs), ds, starts, counts, 0, heads, 4096, precision="f32")
    want = np.concatenate([ref.fused_prompt_attention(q, s, 0, st, c, heads, 4096).reshape(c, -1)
                           for q, s, st, c in zip(qs, rs, starts, counts)])
    assert refmath.close(f32, want, TOL_F32), refmath.max_rel(f32, want)
    ok, err = bf16_ok(got, want, SHORT_ROWS)
    assert ok, err


@pytest.mark.parametrize("fmt", ["f32", "q8_0"])
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("tpb", [32, 64, 128, 1024])
def test_bf16_block_sizes(device, oracle, tpb, dim, fmt):
    """Blocks above 16 tokens: a 64-key tile lies inside one block (tpb >= 64)
    or spans several (32); at 128 and 1,024 a block holds several tiles, so a
    key's slot depends on the tile index as well as its row."""
    heads, kv_heads = 8, 2
    specs = [(1100, 900, 200), (300, 0, 300), (20, 3, 17)]
    say("prefill bf16 tpb", tpb, "dim", dim, fmt)
    dev, ref, ds, rs, qs = build(device, oracle, heads, kv_heads, dim, specs, seed=tpb + dim, tpb=tpb,
                                 q8=fmt == "q8_0")
    starts = [s for _, s, _ in specs]
    counts = [r for _, _, r in specs]
    got = attention.prefill_batch(dev, np.concatenate(qs), ds, starts, counts, 0, heads, 4096, precision="bf16")
    f32 = attention.prefill_batch(dev, np.concatenate(qs), ds, starts, counts, 0, heads, 4096, precision="f32")
    want = np.concatenate([ref.fused_prompt_attention(q, s, 0, st, c, heads, 4096).reshape(c, -1)
                           for q, s, st, c in zip(qs, rs, starts, counts)])
    assert refmath.close(f32, want, TOL_F32), refmath.max_rel(f32, want)
    ok, err = bf16_ok(got, want, SHORT_ROWS)
    assert ok, err


@pytest.mark.parametrize("fmt", ["f32", "q8_0"])
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("group", [1, 2, 3, 4, 5, 6, 7, 8, 10, 16])
def test_f32x3_small_shapes(device, oracle, group, dim, fmt):
    # Q8_0 blocks: d * q dequantised when staged, against the oracle over the
    # dequantised values the blocks hold
    heads, kv_heads = 2 * group, 2
    specs = [(137, 100, 37), (64, 0, 64), (20, 3, 17), (1, 0, 1)]
    say("prefill f32x3 group", group, "dim", dim, fmt)
    dev, ref, ds, rs, qs = build(device, oracle, heads, kv_heads, dim, specs, seed=50 + group, q8=fmt == "q8_0")
    starts = [s for _, s, _ in specs]
    counts = [r for _, _, r in specs]
    got = attention.prefill_batch(dev, np.concatenate(qs), ds, starts, counts, 0, heads, 4096, precision="f32x3")
    want = np.concatenate([ref.fused_prompt_attention(q, s, 0, st, c, heads, 4096).reshape(c, -1)
                           for q, s, st, c in zip(qs, rs, starts, counts)])
    say("f32x3 max rel", refmath.max_rel(got, want))
    assert refmath.close(got, want, TOL_F32), refmath.max_rel(got, want)


@pytest.mark.parametrize("fmt", ["f32", "q8_0"])
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("tpb", [32, 64, 128, 1024])
def test_f32x3_block_sizes(device, oracle, tpb, dim, fmt):
    heads, kv_heads = 8, 2
    specs = [(1100, 900, 200), (300, 0, 300), (20, 3, 17)]
    say("prefill f32x3 tpb", tpb, "dim", dim, fmt)
    dev, ref, ds, rs, qs = build(device, oracle, heads, kv_heads, dim, specs, seed=60 + tpb + dim, tpb=tpb,
                                 q8=fmt == "q8_0")
    starts = [s for _, s, _ in specs]
    counts = [r for _, _, r in specs]
    got = attention.prefill_batch(dev, np.concatenate(qs), ds, starts, counts, 0, heads, 4096, precision="f32x3")
    want = np.concatenate([ref.fused_prompt_attention(q, s, 0, st, c, heads, 4096).reshape(c, -1)
                           for q, s, st, c in zip(qs, rs, starts, counts)])
    assert refmath.close(got, want, TOL_F32), refmath.max_rel(got, want)


@pytest.mark.parametrize("dim", [64, 128])
def test_f32x3_sharp_scores(device, oracle, dim):
    # queries and keys of N(0, 36) put the scores' standard deviation near 36:
    # a score's error enters the softmax's exponent unscaled, so score
    # operands carried in two bf16 parts (16 bits) leave 4.1e-4 on these rows
    # at d=64 (a float64 simulation of the split products), over the f32 bar;
    # with fp16 parts (22 bits) the same simulation gives 1.1e-5
    heads, kv_heads = 8, 2
    w = kv_heads * dim
    specs = [(700, 500, 200), (130, 0, 130)]
    nb = sum((n + 15) // 16 for n, _, _ in specs) + 4
    dev = device.PagedCache(1, kv_heads, dim, 16, nb)
    ref = oracle.Cache(1, kv_heads, dim, 16, nb)
    ds, rs, qs = [], [], []
    for i, (n, _, rows) in enumerate(specs):
        k = (6.0 * synth.normal(90, f"k{i}", n * w)).astype(np.float32).reshape(n, w)
        v = synth.normal(90, f"v{i}", n * w).reshape(n, w)
        sd, sr = dev.create_sequence(), ref.create_sequence()
        dev.append_many(sd, k, v)
        ref.append_many(sr, k, v)
        ds.append(sd)
        rs.append(sr)
        qs.append((6.0 * synth.normal(90, f"q{i}", rows * heads * dim)).astype(np.float32).reshape(rows, -1))
    starts = [s for _, s, _ in specs]
    counts = [r for _, _, r in specs]
    say("prefill f32x3 sharp", dim)
    got = attention.prefill_batch(dev, np.concatenate(qs), ds, starts, counts, 0, heads, 4096, precision="f32x3")
    want = np.concatenate([ref.fused_prompt_attention(q, s, 0, st, c, heads, 4096).reshape(c, -1)
                           for q, s, st, c in zip(qs, rs, starts, counts)])
    say("f32x3 sharp max rel", refmath.max_rel(got, want))
    assert refmath.close(got, want, TOL_F32), refmath.max_rel(got, want)


def test_f32x3_refusals(device):
    # the three-product tiles take the bf16 tiles' shapes: head_dim 64 or 128
    # and power-of-two blocks of 16 to 1,024 tokens; the f32 rows take the rest
    for dim, tpb in [(32, 16), (64, 24)]:
        dev = device.PagedCache(1, 2, dim, tpb, 8, fmt=device.Q8_0)
        s = dev.create_sequence()
        x = synth.normal(1, "x", 20 * 2 * dim).reshape(20, -1)
        dev.append_many(s, x, x)
        q = synth.normal(1, "q", 4 * 4 * dim).reshape(4, -1)
        with pytest.raises(device.InvalidArgument):
            attention.prefill_batch(dev, q, [s], [10], [4], 0, 4, 64, precision="f32x3")
        assert np.isfinite(attention.prefill_batch(dev, q, [s], [10], [4], 0, 4, 64, precision="f32")).all()


def bf16_rne(x):
    """float32 -> the nearest bfloat16 (ties to even), as float32."""
    u = np.ascontiguousarray(x, np.float32).view(np.uint32).astype(np.uint64)
    u = (u + 0x7FFF + ((u >> 16) & 1)) >> 16 << 16
    return u.astype(np.uint32).view(np.float32)


@pytest.mark.parametrize("tpb", [16, 64])
@pytest.mark.parametrize("fmt", ["f32", "q8_0"])
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("group", [1, 4, 8])
def test_bf16_against_bf16_operands(device, oracle, group, dim, fmt, tpb):
    """The MFMA path against the FP64 oracle run on the operands the kernel
    actually multiplies: K and V rounded to bf16 (Q8_0: d * q rounded), and
    the query bf16(q * log2(e)/sqrt(d)) carried back to natural units.  The
    scores then agree to f32 summation error, and what is left is the bf16
    rounding of the probabilities, p~ = p (1 + e), |e| <= u = 2^-9, which
    enters numerator and normaliser alike:
        |o~ - o| = |sum w e (v - o)| / (1 + sum w e) <= u (max|v| + |o|) / (1 - u).
    A dropped or duplicated key in a short row, a wrong scale or a stale
    running maximum breaks this bound by far."""
    heads, kv_heads = 2 * group, 2
    specs = [(137, 100, 37), (64, 0, 64), (20, 3, 17), (300, 250, 50)]
    say("prefill bf16 operands group", group, "dim", dim, fmt, "tpb", tpb)
    nb = sum((n + tpb - 1) // tpb for n, _, _ in specs) + 4
    q8 = fmt == "q8_0"
    dev = device.PagedCache(1, kv_heads, dim, tpb, nb, fmt=device.Q8_0 if q8 else device.F32)
    ref = oracle.Cache(1, kv_heads, dim, tpb, nb)
    w, seed = kv_heads * dim, 100 + group + dim + tpb
    qscale = np.float32(1.4426950408889634 / np.sqrt(float(dim)))
    ds, rs, qs, qo, vmax = [], [], [], [], 0.0
    for i, (n, start, rows) in enumerate(specs):
        k = synth.normal(seed, f"k{i}", n * w).reshape(n, w)
        v = synth.normal(seed, f"v{i}", n * w).reshape(n, w)
        kr, vr = k, v
        if q8:
            kr = oracle.dequantize_q8_0(oracle.quantize_q8_0(k)).reshape(n, w)
            vr = oracle.dequantize_q8_0(oracle.quantize_q8_0(v)).reshape(n, w)
        kr, vr = bf16_rne(kr), bf16_rne(vr)
        vmax = max(vmax, float(np.abs(vr).max()))
        sd, sr = dev.create_sequence(), ref.create_sequence()
        dev.append_many(sd, k, v)
        ref.append_many(sr, kr, vr)
        ds.append(sd)
        rs.append(sr)
        q = synth.normal(seed, f"q{i}", rows * heads * dim).reshape(rows, heads * dim)
        qs.append(q)
        qb = bf16_rne((q * qscale).astype(np.float32))
        qo.append((qb.astype(np.float64) * np.sqrt(float(dim)) / 1.4426950408889634).astype(np.float32))
    starts = [s for _, s, _ in specs]
    counts = [r for _, _, r in specs]
    got = attention.prefill_batch(dev, np.concatenate(qs), ds, starts, counts, 0, heads, 4096, precision="bf16")
    want = np.concatenate([ref.fused_prompt_attention(q, s, 0, st, c, heads, 4096).reshape(c, -1)
                           for q, s, st, c in zip(qo, rs, starts, counts)])
    u = 2.0 ** -9
    bound = u * (vmax + np.abs(want).astype(np.float64)) / (1 - u) + 1e-5
    err = np.abs(np.asarray(got, np.float64) - want)
    assert np.all(err <= bound), (float((err / bound).max()), float(err.max()))
    say("bf16 operands: worst error / bound", float((err / bound).max()), "max error", float(err.max()))


@pytest.mark.parametrize("make,fmt", [(workloads.prefill_c4, "f32"), (workloads.prefill_8b, "f32"),
                                      (workloads.prefill_c4, "q8_0")], ids=["d64", "d128", "d64-q8_0"])
def test_bf16_c4_shape(device, oracle, make, fmt):
    w = make()
    say("prefill", w.name, fmt)
    g = (1, w.kv_heads, w.head_dim, w.tokens_per_block, w.pool_blocks())
    q8 = fmt == "q8_0"
    dev, ref = device.PagedCache(*g, fmt=device.Q8_0 if q8 else device.F32), oracle.Cache(*g)
    ds = workloads.fill_prefill(dev, w)
    q = np.concatenate([w.chunk_queries(i) for i in range(w.sequences)])
    got = attention.prefill_batch(dev, q, ds, [w.prefix] * w.sequences, [w.chunk] * w.sequences, 0, w.heads,
                                  w.context, precision="bf16").reshape(w.sequences, w.chunk, -1)
    f32 = attention.prefill_batch(dev, q, ds, [w.prefix] * w.sequences, [w.chunk] * w.sequences, 0, w.heads,
                                  w.context, precision="f32").reshape(w.sequences, w.chunk, -1)
    # every 37th row and the last, 24 seeded random rows per sequence, and a
    # seeded run of 256 consecutive rows (whole query tiles) in one sequence
    rng = np.random.default_rng(4242)
    run_seq, run_at = int(rng.integers(w.sequences)), int(rng.integers(w.chunk - 256 + 1))
    want, gsel, fsel = [], [], []
    for i in range(w.sequences):
        rows = sorted(set(range(0, w.chunk, 37)) | {w.chunk - 1} |
                      set(rng.choice(w.chunk, 24, replace=False).tolist()))
        s = ref.create_sequence()
        k, v = w.keys(i), w.values(i)
        if q8:  # the oracle holds the dequantised values the Q8_0 blocks store
            k = oracle.dequantize_q8_0(oracle.quantize_q8_0(k)).reshape(k.shape)
            v = oracle.dequantize_q8_0(oracle.quantize_q8_0(v)).reshape(v.shape)
        ref.append_many(s, k, v)
        qi = w.chunk_queries(i)
        for r in rows:
            want.append(ref.fused_prompt_attention(qi[r], s, 0, w.prefix + r, 1, w.heads, w.context))
            gsel.append(got[i, r])
            fsel.append(f32[i, r])
        if i == run_seq:
            run = ref.fused_prompt_attention(qi[run_at:run_at + 256], s, 0, w.prefix + run_at, 256, w.heads,
                                             w.context).reshape(256, -1)
            want.extend(run)
            gsel.extend(got[i, run_at:run_at + 256])
            fsel.extend(f32[i, run_at:run_at + 256])
        ref.drop(s)
    want = np.stack(want)
    assert refmath.close(np.stack(fsel), want, TOL_F32), refmath.max_rel(np.stack(fsel), want)
    ok, err = bf16_ok(np.stack(gsel), want, LONG_ROWS)
    assert ok, err
    say("c4 bf16 vs oracle (max rel, rms):", err)
    # over the whole batch the bf16 path tracks the f32 path
    ok, err = bf16_ok(got, f32, LONG_ROWS)
    assert ok, err
    say("c4 bf16 vs f32 path (max rel, rms):", err)


@pytest.mark.parametrize("make,fmt", [(workloads.prefill_c4, "f32"), (workloads.prefill_8b, "f32"),
                                      (workloads.prefill_c4, "q8_0")], ids=["d64", "d128", "d64-q8_0"])
def test_c4_every_row_against_reference(device, oracle, ref, make, fmt):
    # every one of the batch's 8 x 512 rows, on both paths, against the
    # reference's own fused_prompt_attention (attention.hpp:85-89, built from
    # its sources in oracle/_ref) run over the same K/V on the host's threads:
    # the f32 path within the f32 bar, the bf16 path within its derived bars
    import os

    w = make()
    say("prefill every row", w.name, fmt)
    g = (1, w.kv_heads, w.head_dim, w.tokens_per_block, w.pool_blocks())
    q8 = fmt == "q8_0"
    dev = device.PagedCache(*g, fmt=device.Q8_0 if q8 else device.F32)
    ds = workloads.fill_prefill(dev, w)
    q = np.concatenate([w.chunk_queries(i) for i in range(w.sequences)])
    args = (ds, [w.prefix] * w.sequences, [w.chunk] * w.sequences, 0, w.heads, w.context)
    got = attention.prefill_batch(dev, q, *args, precision="bf16").reshape(w.sequences, w.chunk, -1)
    f32 = attention.prefill_batch(dev, q, *args, precision="f32").reshape(w.sequences, w.chunk, -1)
    x3 = attention.prefill_batch(dev, q, *args, precision="f32x3").reshape(f32.shape)
    threads = max(1, min(16, os.cpu_count() or 1))
    rc = ref.RefCache(*g)
    want = np.empty_like(f32)
    for i in range(w.sequences):
        k, v = w.keys(i), w.values(i)
        if q8:  # the reference holds the dequantised values the Q8_0 blocks store
            k = oracle.dequantize_q8_0(oracle.quantize_q8_0(k)).reshape(k.shape)
            v = oracle.dequantize_q8_0(oracle.quantize_q8_0(v)).reshape(v.shape)
        s = rc.create_sequence()
        rc.append_many(s, k, v)
        want[i] = rc.prompt_batch(w.chunk_queries(i), s, 0, w.prefix, w.chunk, w.heads, w.context, 16,
                                  threads).reshape(w.chunk, -1)
        rc.drop(s)
    assert refmath.close(f32, want, TOL_F32), refmath.max_rel(f32, want)
    ok, err = bf16_ok(got, want, LONG_ROWS)
    assert ok, err
    say("every row: f32 max rel", refmath.max_rel(f32, want), "bf16 (max rel, rms)", err)
    say("every row: f32x3 max rel", refmath.max_rel(x3, want))
    assert refmath.close(x3, want, TOL_F32), refmath.max_rel(x3, want)


@pytest.mark.parametrize("precision", ["bf16", "f32", "f32x3"])
def test_prefill_plan_matches_call(device, oracle, precision):
    # a resident plan launched on two layers gives the one-shot call's bytes,
    # and refuses to run once the cache has changed
    from tvara_amd import hip

    heads, kv_heads, dim = 8, 2, 64
    specs = [(137, 100, 37), (64, 0, 64), (20, 3, 17)]
    g = (2, kv_heads, dim, 16, 40)
    dev = device.PagedCache(*g)
    w = 2 * kv_heads * dim
    ds, qs = [], []
    for i, (n, _, rows) in enumerate(specs):
        s = dev.create_sequence()
        dev.append_many(s, synth.normal(9, f"k{i}", n * w).reshape(n, w), synth.normal(9, f"v{i}", n * w).reshape(n, w))
        ds.append(s)
        qs.append(synth.normal(9, f"q{i}", rows * heads * dim).reshape(rows, heads * dim))
    q = np.concatenate(qs)
    starts, counts = [st for _, st, _ in specs], [r for _, _, r in specs]
    plan = attention.PrefillPlan(dev, ds, starts, counts, heads, 4096, precision)
    dq, out = hip.DeviceArray.from_numpy(q), hip.DeviceArray(q.shape)
    for layer in (1, 0):
        want = attention.prefill_batch(dev, q, ds, starts, counts, layer, heads, 4096, precision=precision)
        out.zero()
        plan.launch(layer, dq.ptr, out.ptr)
        plan.check()
        assert np.array_equal(out.numpy(), want.reshape(q.shape))
    dev.append(ds[0], synth.normal(9, "x", w), synth.normal(9, "y", w))
    with pytest.raises(device.InvalidArgument):
        plan.launch(0, dq.ptr, out.ptr)


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("group", [1, 4])
def test_bf16_nan_poisoned_unused_slots(device, oracle, group, dim):
    # prefill_t174.cpp for the MFMA path: NaN in the unused slots of the last
    # block (past the cached length, inside the last 64-key tile) never reaches
    # a row; chunks that end at the cache end, 16-key boundaries and mid-block
    heads, kv_heads = 2 * group, 2
    w = kv_heads * dim
    for n, rows in [(137, 37), (33, 33), (80, 16), (1, 1)]:
        say("prefill bf16 poison", group, dim, n, rows)
        dev = device.PagedCache(1, kv_heads, dim, 16, n // 16 + 3)
        ref = oracle.Cache(1, kv_heads, dim, 16, n // 16 + 3)
        k = synth.normal(21, "k", n * w).reshape(n, w)
        v = synth.normal(21, "v", n * w).reshape(n, w)
        sd, sr = dev.create_sequence(), ref.create_sequence()
        dev.append_many(sd, k, v)
        ref.append_many(sr, k, v)
        h = dev.physical_block(sd, n - 1)
        for slot in range(n % 16 or 16, 16):
            for kind in (0, 1):
                dev.block_write(h, dev.kv_offset(0, kind, slot), np.full(w, np.nan, np.float32))
        q = synth.normal(21, "q", rows * heads * dim).reshape(rows, heads * dim)
        got = attention.prefill_batch(dev, q, [sd], [n - rows], [rows], 0, heads, 4096, precision="bf16")
        want = ref.fused_prompt_attention(q, sr, 0, n - rows, rows, heads, 4096).reshape(rows, -1)
        assert np.isfinite(got).all()
        ok, err = bf16_ok(got.reshape(rows, -1), want, SHORT_ROWS)
        assert ok, err


def test_bf16_rejections(device):
    dev = device.PagedCache(1, 2, 32, 16, 8)
    s = dev.create_sequence()
    x = synth.normal(1, "x", 20 * 64).reshape(20, 64)
    dev.append_many(s, x, x)
    q = synth.normal(1, "q", 4 * 4 * 32)
    with pytest.raises(device.InvalidArgument):  # bf16 tile kernels cover head_dim 64 and 128
        attention.prefill_batch(dev, q, [s], [10], [4], 0, 4, 64, precision="bf16")
    dev = device.PagedCache(1, 2, 64, 16, 8)
    s = dev.create_sequence()
    x = synth.normal(1, "x", 20 * 128).reshape(20, 128)
    dev.append_many(s, x, x)
    q = synth.normal(1, "q", 4 * 4 * 64).reshape(4, -1)
    q[1, 3] = np.inf
    with pytest.raises(device.InvalidArgument):  # non-finite input
        attention.prefill_batch(dev, q, [s], [10], [4], 0, 4, 64, precision="bf16")
    with pytest.raises(device.InvalidArgument):  # chunk past the cached tokens
        attention.prefill_batch(dev, q, [s], [18], [4], 0, 4, 64, precision="bf16")
    q[1, 3] = 0.0
    for tpb in (8, 24):  # bf16 tile kernels take power-of-two blocks of 16 to 1,024 tokens
        dev = device.PagedCache(1, 2, 64, tpb, 8)
        s = dev.create_sequence()
        dev.append_many(s, x, x)
        with pytest.raises(device.InvalidArgument):
            attention.prefill_batch(dev, q, [s], [10], [4], 0, 4, 64, precision="bf16")
        f32 = attention.prefill_batch(dev, q, [s], [10], [4], 0, 4, 64, precision="f32")
        assert np.all(np.isfinite(f32))


@pytest.mark.parametrize("dim", [64, 128])
def test_x3_range(device, dim):
    # f32x3 carries queries and keys as fp16 parts: a visible key beyond the
    # fp16 range (65,504), or a query beyond it once multiplied by
    # log2(e)/sqrt(head_dim) (1e6 at both widths), makes scores non-finite and
    # the launch fails as a non-finite input does; the f32 rows take the same
    # inputs
    heads, kv_heads = 4, 2
    w = kv_heads * dim
    x = synth.normal(2, "x", 20 * w).reshape(20, w)
    q = synth.normal(2, "q", 4 * heads * dim).reshape(4, -1)
    for where in ("key", "query"):
        dev = device.PagedCache(1, kv_heads, dim, 16, 8)
        s = dev.create_sequence()
        k, qq = x.copy(), q.copy()
        if where == "key":
            k[5, 7] = 7e4
        else:
            qq[2, dim + 3] = -1e6
        dev.append_many(s, k, x)
        say("prefill x3 range", dim, where)
        with pytest.raises(device.InvalidArgument):
            attention.prefill_batch(dev, qq, [s], [10], [4], 0, heads, 4096, precision="f32x3")
        f32 = attention.prefill_batch(dev, qq, [s], [10], [4], 0, heads, 4096, precision="f32")
        assert np.isfinite(f32).all()
        # within the range the launch goes through
        k[5, 7], qq[2, dim + 3] = 6e4, -6e4
        dev.block_write(dev.physical_block(s, 5), dev.kv_offset(0, 0, 5), k[5])
        got = attention.prefill_batch(dev, qq, [s], [10], [4], 0, heads, 4096, precision="f32x3")
        assert np.isfinite(got).all()


@pytest.mark.parametrize("precision", ["bf16", "f32", "f32x3"])
@pytest.mark.parametrize("dim", [64, 128])
def test_chunk_invariant_under_future_tokens(device, precision, dim):
    # prefill_t173.cpp:6: tokens appended after a chunk (here huge and NaN
    # values, in the chunk's last block and in new blocks) leave the chunk's
    # rows byte-identical
    heads, kv_heads, tpb = 8, 2, 16
    w = kv_heads * dim
    dev = device.PagedCache(1, kv_heads, dim, tpb, 24)
    s = dev.create_sequence()
    n, start, rows = 150, 110, 40
    dev.append_many(s, synth.normal(41, "k", n * w).reshape(n, w), synth.normal(41, "v", n * w).reshape(n, w))
    q = synth.normal(41, "q", rows * heads * dim).reshape(rows, heads * dim)
    before = attention.prefill_batch(dev, q, [s], [start], [rows], 0, heads, 4096, precision=precision)
    junk = np.full((60, w), 3e4, np.float32)
    junk[::3] = np.nan
    dev.append_many(s, junk, junk)
    after = attention.prefill_batch(dev, q, [s], [start], [rows], 0, heads, 4096, precision=precision)
    assert np.isfinite(before).all()
    assert np.array_equal(before, after)


@pytest.mark.parametrize("precision", ["bf16", "f32", "f32x3"])
@pytest.mark.parametrize("fmt", ["f32", "q8_0"])
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("group", [1, 3, 4, 8, 12])
def test_zero_query_averages_every_visible_key(device, oracle, group, dim, fmt, precision):
    # With q = 0 every score is 0, every probability exp2(0) = 1 exactly, and
    # with V of integers (exact in bf16, Q8_0 and every f32 partial sum) each
    # output row is the exact mean of the V rows its causal mask admits.
    # A dropped or repeated key moves the mean by at least 1/(2n) of a unit,
    # far above the 1e-6 bar, so the mask boundary of every row, the chunk
    # tiling, the GQA row mapping and the paged block walk are checked exactly
    # (the bf16 bars above cannot see a single key among thousands).  The f32
    # path (decode kernels, split merges) is exact here too.
    heads, kv_heads = 2 * group, 2
    w = kv_heads * dim
    specs = [(1100, 1000, 100), (300, 0, 300), (77, 60, 17), (2100, 1600, 500)]
    nb = sum((n + 15) // 16 for n, _, _ in specs) + 4
    q8 = fmt == "q8_0"
    dev = device.PagedCache(1, kv_heads, dim, 16, nb, fmt=device.Q8_0 if q8 else device.F32)
    ref = oracle.Cache(1, kv_heads, dim, 16, nb)
    rng = np.random.default_rng(83 + group + dim)
    ds, rs, vals = [], [], []
    for i, (n, _, _) in enumerate(specs):
        k = synth.normal(83, f"k{i}", n * w).reshape(n, w)
        # integers (exact in bf16); one 127 per 32-column group makes the
        # Q8_0 scale exactly 1, so the blocks hold the same integers
        v = rng.integers(-4, 5, size=(n, w)).astype(np.float32)
        v[:, ::32] = 127.0
        if q8:
            k = oracle.dequantize_q8_0(oracle.quantize_q8_0(k)).reshape(n, w)
            assert np.array_equal(oracle.dequantize_q8_0(oracle.quantize_q8_0(v)).reshape(n, w), v)
        sd, sr = dev.create_sequence(), ref.create_sequence()
        dev.append_many(sd, k, v)
        ref.append_many(sr, k, v)
        ds.append(sd)
        rs.append(sr)
        vals.append(v)
    starts = [s for _, s, _ in specs]
    counts = [r for _, _, r in specs]
    rows = sum(counts)
    q = np.zeros((rows, heads * dim), np.float32)
    say("prefill zero query", group, dim, fmt, precision)
    got = attention.prefill_batch(dev, q, ds, starts, counts, 0, heads, 4096, precision=precision)
    got = got.reshape(rows, heads, dim)
    at = 0
    for i, (n, start, cnt) in enumerate(specs):
        csum = np.cumsum(vals[i].reshape(n, kv_heads, dim).astype(np.float64), axis=0)
        for r in range(cnt):
            want = csum[start + r] / (start + r + 1)  # keys 0 .. start + r
            for h in range(heads):
                assert np.allclose(got[at + r, h], want[h // group], rtol=1e-6, atol=1e-6), (i, r, h)
        at += cnt


def _every_kernel(monkeypatch, run):
    """run() under TVARA_PREFILL_PIPE = 0 (prefill_bf16_kernel) and 1 (the
    software-pipelined kernel)."""
    out = []
    for flag in ("0", "1"):
        monkeypatch.setenv("TVARA_PREFILL_PIPE", flag)
        out.append(run())
    monkeypatch.delenv("TVARA_PREFILL_PIPE")
    return out


def _same_bits(plain, *others):
    return all(np.array_equal(plain.view(np.uint32), o.view(np.uint32)) for o in others)


@pytest.mark.parametrize("make,fmt", [(workloads.prefill_c4, "f32"), (workloads.prefill_c4, "q8_0"),
                                      (workloads.prefill_8b, "f32")], ids=["d64", "d64-q8_0", "d128"])
def test_pipelined_kernel_matches_plain_kernel(device, monkeypatch, make, fmt):
    """The pipelined kernels perform the plain kernel's products, exponentials
    and rescales in the same order, so the whole chunked-prefill batch must
    agree bit for bit (the plain kernel is pinned to the oracle above)."""
    w = make()
    say("pipelined vs plain prefill", w.name, fmt)
    g = (1, w.kv_heads, w.head_dim, w.tokens_per_block, w.pool_blocks())
    dev = device.PagedCache(*g, fmt=device.Q8_0 if fmt == "q8_0" else device.F32)
    ds = workloads.fill_prefill(dev, w)
    q = np.concatenate([w.chunk_queries(i) for i in range(w.sequences)])
    plain, pipe = _every_kernel(monkeypatch, lambda: attention.prefill_batch(
        dev, q, ds, [w.prefix] * w.sequences, [w.chunk] * w.sequences, 0, w.heads, w.context, precision="bf16"))
    assert np.isfinite(plain).all()
    assert _same_bits(plain, pipe)


@pytest.mark.parametrize("tpb", [16, 32, 1024])
@pytest.mark.parametrize("group", [1, 3, 4, 8])
def test_pipelined_kernel_ragged_chunks(device, oracle, monkeypatch, group, tpb):
    """Ragged chunks (a row alone, chunks ending inside a tile, a chunk with no
    cached prefix, odd and even tile counts) through every kernel: equal bits,
    and the pipelined ones within the short-row bars of the oracle."""
    heads, kv_heads, dim = 2 * group, 2, 64
    specs = [(1, 0, 1), (65, 64, 1), (200, 137, 63), (129, 0, 129), (700, 300, 400)]
    say("pipelined prefill ragged, group", group, "tpb", tpb)
    dev, ref, ds, rs, qs = build(device, oracle, heads, kv_heads, dim, specs, seed=31 + group, tpb=tpb)
    starts = [s for _, s, _ in specs]
    counts = [r for _, _, r in specs]
    plain, pipe = _every_kernel(monkeypatch, lambda: attention.prefill_batch(
        dev, np.concatenate(qs), ds, starts, counts, 0, heads, 4096, precision="bf16"))
    assert _same_bits(plain, pipe)
    want = np.concatenate([ref.fused_prompt_attention(q, s, 0, st, c, heads, 4096).reshape(c, -1)
                           for q, s, st, c in zip(qs, rs, starts, counts)])
    ok, err = bf16_ok(pipe, want, SHORT_ROWS)
    assert ok, err


@pytest.mark.parametrize("fmt", ["f32", "q8_0"])
@pytest.mark.parametrize("tpb", [16, 32, 64, 128])
def test_pipelined_kernel_over_blocks(device, oracle, monkeypatch, tpb, fmt):
    # the two kernels over both block forms and their sizes, in launches that are
    # not split (as the choice between them has it): equal bits, within the
    # short-row bars; without the choice this batch runs as splits
    heads, kv_heads, dim = 8, 2, 64
    specs = [(1100, 900, 200), (300, 0, 300), (20, 3, 17)]
    say("pipelined prefill over blocks", tpb, fmt)
    dev, ref, ds, rs, qs = build(device, oracle, heads, kv_heads, dim, specs, seed=170 + tpb, tpb=tpb, q8=fmt == "q8_0")
    starts = [s for _, s, _ in specs]
    counts = [r for _, _, r in specs]

    def run():
        attention.profile_reset()
        out = attention.prefill_batch(dev, np.concatenate(qs), ds, starts, counts, 0, heads, 4096, precision="bf16")
        return out, attention.profile_read("paged_prefill_merge")[1]

    attention.profile_enable(True)
    try:
        (plain, m0), (pipe, m1) = _every_kernel(monkeypatch, run)
        split, m2 = run()
    finally:
        attention.profile_enable(False)
    assert (m0, m1, m2) == (0, 0, 1)
    assert _same_bits(plain, pipe)
    want = np.concatenate([ref.fused_prompt_attention(q, s, 0, st, c, heads, 4096).reshape(c, -1)
                           for q, s, st, c in zip(qs, rs, starts, counts)])
    for got in (pipe, split):
        ok, err = bf16_ok(got, want, SHORT_ROWS)
        assert ok, err


F32_TILE_SPECS = [(1510, 1000, 500), (300, 0, 300), (70, 67, 3), (1, 0, 1)]


@pytest.mark.parametrize("fmt", ["f32", "q8_0"])
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("group,tpb", [(1, 16), (3, 64), (4, 1024), (8, 16), (12, 32)])  # 12: slices of six heads
def test_f32_tiles(device, oracle, group, tpb, dim, fmt):
    # a batch above the f32 tiles' threshold of work, with key splits (some of
    # them empty for the short sequences), rows and keys that fill neither a
    # wave nor a tile, and ten cached tokens past the chunk; rows at the chunk's
    # ends and at tile and workgroup edges against the oracle
    heads = 24
    say("prefill f32 tiles group", group, "tpb", tpb, "dim", dim, fmt)
    dev, ref, ds, rs, qs = build(device, oracle, heads, heads // group, dim, F32_TILE_SPECS, seed=90 + group, tpb=tpb,
                                 q8=fmt == "q8_0")
    starts = [s for _, s, _ in F32_TILE_SPECS]
    counts = [r for _, _, r in F32_TILE_SPECS]
    got = attention.prefill_batch(dev, np.concatenate(qs), ds, starts, counts, 0, heads, 4096, precision="f32")
    row0 = 0
    for q, s, st, c in zip(qs, rs, starts, counts):
        for lo, n in [(0, 3), (22, 4), (30, 4), (126, 4), (c - 3, 3)]:
            lo, n = max(0, min(lo, c - 1)), min(n, c)
            n = min(n, c - lo)
            want = ref.fused_prompt_attention(q[lo:lo + n], s, 0, st + lo, n, heads, 4096).reshape(n, -1)
            part = got[row0 + lo:row0 + lo + n]
            assert refmath.close(part, want, 1e-5), (lo, refmath.max_rel(part, want))
        row0 += c


@pytest.mark.parametrize("precision", ["f32", "bf16", "f32x3"])
def test_key_splits_of_one_long_sequence(device, oracle, precision):
    # a few rows after a long prefix beside fresh prompts: the long rows' runs
    # are many, the prompts' one or two, and partials exist for rows of several
    # runs only (a slot per row and run of the longest would take 213 MB in f32
    # and 202 MB on the bf16 tiles; these take 1 MB and 3), on a plan held open
    # while the device's free memory is read
    import ctypes as C

    from tvara_amd import hip

    heads, kv_heads, dim = 8, 2, 64
    specs = [(16000 + 16, 16000, 16)] + [(512, 0, 512)] * 7 if precision == "f32" else \
        [(16000 + 16, 16000, 16)] + [(300, 0, 300)] * 5
    say("prefill splits, one long sequence", precision)
    dev, ref, ds, rs, qs = build(device, oracle, heads, kv_heads, dim, specs, seed=140)
    starts = [s for _, s, _ in specs]
    counts = [r for _, _, r in specs]

    def free():
        hip.synchronize()
        n, total = C.c_size_t(), C.c_size_t()
        hip.check(hip.runtime().hipMemGetInfo(C.byref(n), C.byref(total)))
        return n.value

    dq, out = hip.DeviceArray.from_numpy(np.concatenate(qs)), hip.DeviceArray((sum(counts), heads * dim))
    before = free()
    plan = attention.PrefillPlan(dev, ds, starts, counts, heads, 1 << 20, precision)
    used = before - free()
    plan.launch(0, dq.ptr, out.ptr)
    plan.check()
    got, row0 = out.numpy(), 0
    for q, s, st, c in zip(qs, rs, starts, counts):
        for lo in sorted({0, 31, 32, c // 2, c - 1} & set(range(c))):
            want = ref.fused_prompt_attention(q[lo], s, 0, st + lo, 1, heads, 1 << 20)
            part = got[row0 + lo]
            if precision == "bf16":
                ok, err = bf16_ok(part, want, SHORT_ROWS)
                assert ok, (st, lo, err)
            else:
                assert refmath.close(part, want, 1e-5 if precision == "f32" else TOL_F32), (st, lo)
        row0 += c
    assert used < 48 << 20, used


# (heads, KV heads, dim, format, [(prefix, rows)], tiles): few rows after long
# prefixes, where a tile of 128 rows would be nearly empty, stay row by row
F32_ROUTES = [(32, 8, 64, "f32", [(30000, 4)], False), (32, 8, 64, "f32", [(30000, 16)], True),
              (32, 8, 64, "f32", [(1500, 4)] * 32, False), (32, 8, 64, "f32", [(1500, 4)] * 32 + [(0, 1500)], True),
              (32, 8, 128, "f32", [(8000, 4)] * 2, False), (32, 8, 128, "f32", [(8000, 32)] * 2, True),
              (9, 3, 64, "f32", [(100000, 4)], False), (9, 3, 64, "f32", [(16000, 40)], True),
              (32, 32, 64, "f32", [(16000, 6)], False), (32, 32, 64, "f32", [(4000, 64)], True),
              (64, 8, 128, "f32", [(8000, 1)] * 4, False), (64, 8, 128, "f32", [(8000, 8)] * 4, True),
              (64, 8, 128, "q8_0", [(30000, 4)], False), (32, 8, 64, "q8_0", [(4000, 256)], True)]


@pytest.mark.parametrize("heads,kv_heads,dim,fmt,chunks,tiles", F32_ROUTES)
def test_f32_route(device, oracle, heads, kv_heads, dim, fmt, chunks, tiles):
    specs = [(p + r, p, r) for p, r in chunks]
    say("prefill f32 route", heads, kv_heads, dim, fmt, chunks[0], len(chunks))
    dev, ref, ds, rs, qs = build(device, oracle, heads, kv_heads, dim, specs, seed=160, q8=fmt == "q8_0")
    attention.profile_enable(True)
    attention.profile_reset()
    try:
        got = attention.prefill_batch(dev, np.concatenate(qs), ds, [s for _, s, _ in specs], [r for _, _, r in specs],
                                      0, heads, 1 << 20, precision="f32")
        assert attention.profile_read("paged_prefill_f32")[1] == int(tiles)
        assert attention.profile_read("paged_decode")[1] == int(not tiles)
    finally:
        attention.profile_enable(False)
    last = ref.fused_prompt_attention(qs[-1][-1], rs[-1], 0, specs[-1][0] - 1, 1, heads, 1 << 20)
    assert refmath.close(got.reshape(sum(len(q) for q in qs), -1)[-1], last, 1e-5)


@pytest.mark.parametrize("dim", [64, 128])
def test_f32_tiles_split_a_long_sequence_of_a_large_batch(device, oracle, dim):
    # 1,024 workgroups and more (33 sequences of 128 rows, eight KV heads) run
    # unsplit, unless one of them alone takes longer than a CU's share of the
    # whole batch; whether a merge ran says which
    heads, kv_heads = 32, 8
    for start, merges in [(20000, 1), (0, 0)]:
        specs = [(start + 33, start, 33)] + [(128, 0, 128)] * 33
        say("prefill f32 large batch", dim, start)
        dev, ref, ds, rs, qs = build(device, oracle, heads, kv_heads, dim, specs, seed=150)
        attention.profile_enable(True)
        attention.profile_reset()
        try:
            got = attention.prefill_batch(dev, np.concatenate(qs), ds, [s for _, s, _ in specs],
                                          [r for _, _, r in specs], 0, heads, 1 << 20, precision="f32")
            assert attention.profile_read("paged_prefill_merge")[1] == merges
            assert attention.profile_read("paged_prefill_f32")[1] == 1
        finally:
            attention.profile_enable(False)
        row0 = 0
        for q, s, (_, st, c) in zip(qs, rs, specs):
            for lo in (0, 31, c - 1):
                want = ref.fused_prompt_attention(q[lo], s, 0, st + lo, 1, heads, 1 << 20)
                assert refmath.close(got[row0 + lo], want, 1e-5), (st, lo)
            row0 += c


@pytest.mark.parametrize("dim", [64, 128])
def test_f32_tiles_non_finite(device, dim):
    # values that are not finite reach the rows that see them and no others (a
    # masked probability is not multiplied by them); a key that is not finite
    # fails the call if a row sees it, and does not if none does
    heads, kv_heads, n, start, rows = 24, 6, 1510, 1000, 500
    w = kv_heads * dim
    k, v = (synth.normal(3, t, n * w).reshape(n, w) for t in "kv")
    q = synth.normal(3, "q", rows * heads * dim).reshape(rows, heads * dim)

    def run(k, v):
        c = device.PagedCache(1, kv_heads, dim, 16, n // 16 + 4, fmt=device.F32)
        s = c.create_sequence()
        c.append_many(s, k, v)
        return attention.prefill_batch(c, q, [s], [start], [rows], 0, heads, 4096, precision="f32")

    clean = run(k, v)
    at = 1203
    for bad in (np.nan, np.inf):
        vb = v.copy()
        vb[at, dim + 5] = bad
        vb[n - 1] = np.nan  # past the chunk
        got = run(k, vb).reshape(rows, heads, dim)
        hit = np.zeros(got.shape, bool)
        hit[at - start:, 4:8, 5] = True
        assert np.array_equal(~np.isfinite(got), hit)
        keep = clean.reshape(rows, heads, dim)
        assert refmath.close(got[~hit], keep[~hit], 1e-6)
    kb = k.copy()
    kb[n - 1] = np.inf
    assert np.array_equal(run(kb, v), clean)
    kb[at, 3] = np.inf
    with pytest.raises(ValueError, match="invalid online attention input"):
        run(kb, v)


@pytest.mark.parametrize("precision", ["bf16", "f32x3"])
@pytest.mark.parametrize("fmt", ["f32", "q8_0"])
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("group,tpb", [(1, 16), (3, 64), (4, 16), (8, 1024), (12, 16)])
def test_tile_key_splits(device, oracle, group, tpb, dim, fmt, precision):
    # few workgroups, so their key tiles run as splits: a chunk whose last split
    # takes the rest of the keys, chunks of one split beside it (written without
    # a merge), and a chunk whose rows start mid-tile; every row against the
    # oracle, with the bars of the short rows (above)
    heads, kv_heads = 2 * group, 2
    specs = [(2615, 2500, 100), (300, 0, 300), (70, 67, 3), (1, 0, 1), (1000, 865, 135)]
    say("prefill splits", precision, "group", group, "tpb", tpb, "dim", dim, fmt)
    dev, ref, ds, rs, qs = build(device, oracle, heads, kv_heads, dim, specs, seed=120 + group, tpb=tpb, q8=fmt == "q8_0")
    starts = [s for _, s, _ in specs]
    counts = [r for _, _, r in specs]
    got = attention.prefill_batch(dev, np.concatenate(qs), ds, starts, counts, 0, heads, 4096, precision=precision)
    want = np.concatenate([ref.fused_prompt_attention(q, s, 0, st, c, heads, 4096).reshape(c, -1)
                           for q, s, st, c in zip(qs, rs, starts, counts)])
    if precision == "bf16":
        ok, err = bf16_ok(got, want, SHORT_ROWS)
        assert ok, err
    else:
        assert refmath.close(got, want, TOL_F32), refmath.max_rel(got, want)


@pytest.mark.parametrize("precision", ["bf16", "f32x3"])
@pytest.mark.parametrize("dim", [64, 128])
def test_tile_key_splits_reject_what_unsplit_tiles_reject(device, dim, precision):
    # a chunk whose keys run as splits: a value that is not finite (seen by rows
    # of one split only), a key or query outside the fp16 range in three
    # products, and values whose weighted sum overflows f32 only once the splits
    # are added (equal scores: every weight is 1, and 4,000 of 2e35 pass f32's
    # largest while the 256 of a split stay below); the largest sum that fits
    # goes through
    heads, kv_heads, n, rows = 8, 2, 4000, 40
    w = kv_heads * dim
    k, v = (synth.normal(7, t, n * w).reshape(n, w) for t in "kv")
    q = synth.normal(7, "q", rows * heads * dim).reshape(rows, -1)

    def run(k, v, q):
        c = device.PagedCache(1, kv_heads, dim, 16, n // 16 + 4)
        s = c.create_sequence()
        c.append_many(s, k, v)
        return attention.prefill_batch(c, q, [s], [n - rows], [rows], 0, heads, 1 << 20, precision=precision)

    say("prefill split rejections", dim, precision)
    assert np.isfinite(run(k, v, q)).all()
    for at in (5, n - 20):
        bad = v.copy()
        bad[at, 3] = np.nan
        with pytest.raises(device.InvalidArgument):
            run(k, bad, q)
        bad = k.copy()
        bad[at, 3] = np.inf
        with pytest.raises(device.InvalidArgument):
            run(bad, v, q)
        if precision == "f32x3":
            bad[at, 3] = 7e4
            with pytest.raises(device.InvalidArgument):
                run(bad, v, q)
    if precision == "f32x3":
        bad = q.copy()
        bad[rows - 1, 2] = -1e6
        with pytest.raises(device.InvalidArgument):
            run(k, v, bad)
    zero = np.zeros_like(q)
    with pytest.raises(device.InvalidArgument):
        run(k, np.full_like(v, 2e35), zero)
    got = run(k, np.full_like(v, 2e34), zero)
    assert refmath.close(got / 2e34, np.ones_like(got), 1e-2)
