"""The batched decode's work split at its edges: pieces of one unit per workgroup (few keys),
equal segments past them, head groups that are no power of two, and head_dim 64."""
import numpy as np
import pytest

import mi_attn
from helpers import assert_parity, f16, oracle_attention

pytestmark = pytest.mark.gpu


def rand(seed, shape, scale=1.0):
    return (scale * np.random.default_rng(seed).standard_normal(shape)).astype(np.float16).view(np.uint16)


def run(ctx, q, k, v, lengths, hq, hkv, d, cap):
    qt, lt = ctx.tensor(q), ctx.tensor(np.asarray(lengths, np.uint32), mi_attn.U32)
    kt, vt = (ctx.tensor(np.ascontiguousarray(x.transpose(0, 2, 1, 3))) for x in (k, v))
    strides = (hkv * cap * d, d, cap * d, 1)
    kview, vview = kt.view(k.shape, strides), vt.view(v.shape, strides)
    ctx.take_kernel_profiles()
    ctx.set_kernel_profiling(True)
    try:
        batch = ctx.begin_batch()
        out = batch.attention_decode_batched(qt, kview, vview, lt, mi_attn.AttentionConfig(hq, hkv, d, True, 0))
        batch.finish()
        names = [name for name, _ in ctx.take_kernel_profiles()]
    finally:
        ctx.set_kernel_profiling(False)
    fixed = ctx.empty(q.shape)
    batch = ctx.begin_batch()
    batch.attention_decode_batched_noalloc(qt, kview, vview, lt, mi_attn.AttentionConfig(hq, hkv, d, True, 0), 0,
                                           fixed)
    batch.finish()
    got = ctx.download(out)
    assert (ctx.download(fixed) == got).all()
    return got, names


@pytest.mark.parametrize("hq,hkv,d,cap,lengths", [
    (16, 8, 128, 1300, [1, 127, 128, 129, 1300]),           # 128-key pieces, more than 8 of a unit
    (8, 1, 128, 6000, [6000, 0, 5]),                        # 47 pieces of one unit: overflow slots
    (32, 8, 128, 1100, [256, 257, 512, 1100, 1, 900] * 3),  # 256-key pieces
    (32, 8, 128, 1200, [1200] * 20),                        # past the pieces: equal segments
    (40, 8, 128, 500, [500, 33, 64, 0, 499]),               # groups of 5
    (34, 2, 128, 400, [400, 399]),                          # groups of 17: chunks of 9 and 8
    (24, 2, 128, 4000, [4000, 3073, 37]),                   # 32 pieces of 12 heads: two merge workgroups
    (64, 8, 64, 1000, [1000, 33, 64, 0, 999]),
    (64, 8, 64, 3000, [3000, 2999, 1, 768] * 4),
    (40, 8, 64, 800, [(b * 97) % 250 for b in range(60)] + [800]),  # groups of 5, pieces
    (34, 2, 64, 800, [(b * 97) % 801 for b in range(70)]),          # chunks of 9 and 8
    (8, 2, 64, 8192, [(b * 97) % 300 for b in range(90)]),          # groups of 4 by the capacity
    (64, 8, 64, 800, [(b * 5) % 129 for b in range(150)]),          # whole units, several per workgroup
    (16, 8, 128, 130, [(b * 5) % 129 for b in range(150)]),
    (16, 8, 128, 130, [(b * 5) % 130 for b in range(150)]),         # one key too many: equal segments
    (8, 4, 128, 20, [1] * 600),
])
def test_batched_decode_work_split(ctx, hq, hkv, d, cap, lengths):
    B = len(lengths)
    q, k, v = rand(1, (B, hq, d), 2.0), rand(2, (B, cap, hkv, d)), rand(3, (B, cap, hkv, d))
    got, names = run(ctx, q, k, v, lengths, hq, hkv, d, cap)
    assert names == ["attn_decode_stream", "attn_decode_stream_merge"], names
    for b, n in enumerate(lengths):
        if n == 0:
            assert np.isnan(f16(got[b])).all()
            continue
        ref = oracle_attention(q[b:b + 1], k[b, :n], v[b, :n], hq=hq, hkv=hkv, d=d, off=n - 1)
        assert_parity(got[b:b + 1], ref, label=f"seq {b} len {n}")
        if d == 64:  # f32 probabilities: one rounding of the output and a few of the sums
            bound = np.abs(ref["f32"]) * 2.0 ** -11 + 2.0 ** -24 + 1e-5
            assert (np.abs(f16(got[b:b + 1]).astype(np.float64) - ref["f32"]) <= bound).all()


@pytest.mark.parametrize("B,hq,hkv,cap", [
    (900, 34, 1, 40),   # compact, with chunks that divide the group: 17 of 2 heads
    (700, 34, 1, 40),   # compact: three chunks of 12, 12 and 10
    (200, 34, 1, 40),   # fixed slots
])
def test_batched_decode_of_wide_groups_in_the_fixed_buffer(ctx, B, hq, hkv, cap):
    """Near the fixed buffer's size the call without allocations still gives the other call's bits,
    so the head chunks, which move the pieces' boundaries, are the same in both."""
    lengths = [1 + (11 * b) % cap for b in range(B)]
    q, k, v = rand(1, (B, hq, 128), 2.0), rand(2, (B, cap, hkv, 128)), rand(3, (B, cap, hkv, 128))
    got, _ = run(ctx, q, k, v, lengths, hq, hkv, 128, cap)  # compares the two calls
    for b in range(0, B, 97):
        n = lengths[b]
        ref = oracle_attention(q[b:b + 1], k[b, :n], v[b, :n], hq=hq, hkv=hkv, d=128, off=n - 1)
        assert_parity(got[b:b + 1], ref, label=f"seq {b} len {n}")


@pytest.mark.parametrize("B,hq,hkv,cap,fits", [
    (190, 32, 8, 8192, False),  # groups of 4, whose units alone keep to the rows kernel
    (190, 32, 8, 7680, True),   # one rows split fewer
    (500, 16, 8, 8192, False),  # groups of 2
    (1000, 8, 8, 6200, False),  # groups of 1
    (1000, 8, 1, 6200, False),  # one KV head
])
def test_calls_past_the_fixed_buffer_by_their_capacity_take_the_kernel_that_fits(ctx, B, hq, hkv, cap, fits):
    """The rows kernel's partials grow with the capacity; where they pass the no-allocation buffer the
    stream kernel serves both calls. All sequences read one cache."""
    d, lengths = 64, [1 + (7 * b) % 900 for b in range(B)]
    assert (B * hq * -(-cap // 768) * (d + 2) * 4 <= 16 << 20) == fits
    q, k, v = rand(1, (B, hq, d), 2.0), rand(2, (cap, hkv, d)), rand(3, (cap, hkv, d))
    qt, lt = ctx.tensor(q), ctx.tensor(np.asarray(lengths, np.uint32), mi_attn.U32)
    ks, vs = ctx.tensor(k), ctx.tensor(v)  # the views do not own the memory
    kt, vt = (x.view((B, cap, hkv, d), (0, hkv * d, d, 1)) for x in (ks, vs))
    cfg = mi_attn.AttentionConfig(hq, hkv, d, True, 0)
    ctx.take_kernel_profiles()
    ctx.set_kernel_profiling(True)
    try:
        batch = ctx.begin_batch()
        out = batch.attention_decode_batched(qt, kt, vt, lt, cfg)
        batch.finish()
        names = [name for name, _ in ctx.take_kernel_profiles()]
    finally:
        ctx.set_kernel_profiling(False)
    assert names == (["attn_rows_batched"] if fits else ["attn_decode_stream", "attn_decode_stream_merge"]), names
    fixed = ctx.empty(q.shape)
    batch = ctx.begin_batch()
    batch.attention_decode_batched_noalloc(qt, kt, vt, lt, cfg, 0, fixed)
    batch.finish()
    got = ctx.download(out)
    assert (ctx.download(fixed) == got).all()
    for b in range(0, B, 97):
        n = lengths[b]
        ref = oracle_attention(q[b:b + 1], k[:n], v[:n], hq=hq, hkv=hkv, d=d, off=n - 1)
        assert_parity(got[b:b + 1], ref, label=f"seq {b} len {n}")


@pytest.mark.parametrize("hq,hkv,cap,B", [
    (32, 8, 4096, 8),    # groups of 4, few sequences
    (32, 8, 1024, 32),   # two rows splits of each unit
    (32, 8, 4096, 70),   # groups of 4, between one unit and six per CU
    (40, 8, 1024, 8),    # fewer than nine heads per CU
    (16, 8, 1024, 20),
    (8, 1, 4096, 8),     # one KV head
    (64, 8, 700, 8),     # one rows split
])
def test_short_sequences_at_head_dim_64_stay_on_the_rows_kernel(ctx, hq, hkv, cap, B):
    """Calls whose sequences may be short, where the rows kernel's one launch is the faster one."""
    d, lengths = 64, [1 + (7 * b) % 60 for b in range(B)]
    q, k, v = rand(1, (B, hq, d), 2.0), rand(2, (B, 64, hkv, d)), rand(3, (B, 64, hkv, d))
    kt = ctx.empty((B, cap, hkv, d))
    vt = ctx.empty((B, cap, hkv, d))
    pad = np.zeros((B, cap - 64, hkv, d), np.uint16)
    ctx.upload(kt, np.concatenate([k, pad], 1))
    ctx.upload(vt, np.concatenate([v, pad], 1))
    qt, lt = ctx.tensor(q), ctx.tensor(np.asarray(lengths, np.uint32), mi_attn.U32)
    ctx.take_kernel_profiles()
    ctx.set_kernel_profiling(True)
    try:
        batch = ctx.begin_batch()
        out = batch.attention_decode_batched(qt, kt, vt, lt, mi_attn.AttentionConfig(hq, hkv, d, True, 0))
        batch.finish()
        names = [name for name, _ in ctx.take_kernel_profiles()]
    finally:
        ctx.set_kernel_profiling(False)
    assert names == ["attn_rows_batched"], names
    got = ctx.download(out)
    for b in range(0, B, 5):
        n = lengths[b]
        ref = oracle_attention(q[b:b + 1], k[b, :n], v[b, :n], hq=hq, hkv=hkv, d=d, off=n - 1)
        assert_parity(got[b:b + 1], ref, label=f"seq {b} len {n}")


def test_batched_decode_with_infinite_values_at_head_dim_64(ctx):
    """An infinite value gives the infinity that the weighted sum gives, in its own column only."""
    hq, hkv, d, cap, lengths = 64, 8, 64, 800, [800, 37, 300, 65] * 4
    q, k, v = rand(4, (16, hq, d)), rand(5, (16, cap, hkv, d)), rand(6, (16, cap, hkv, d))
    for b, n in enumerate(lengths):
        v[b, n - 1, b % hkv, b] = np.float16(np.inf if b % 2 else -np.inf).view(np.uint16)
    got, _ = run(ctx, q, k, v, lengths, hq, hkv, d, cap)
    for b, n in enumerate(lengths):
        ref = oracle_attention(q[b:b + 1], k[b, :n], v[b, :n], hq=hq, hkv=hkv, d=d, off=n - 1)["f32"]
        x = f16(got[b:b + 1])
        assert (np.isposinf(ref) == np.isposinf(x)).all() and (np.isneginf(ref) == np.isneginf(x)).all()
        fine = np.isfinite(ref)
        assert np.isfinite(x[fine]).all() and np.abs(x[fine] - ref[fine]).max() <= 2e-3
