"""The few-row MFMA attention (attn_decode.hip) at the edges of its tiles, splits, head
chunks and row packing, against the oracle."""
import numpy as np
import pytest

import mi_attn
import oracle
from helpers import KINDS, assert_parity, f16, oracle_attention, run_attention, upload_kv

pytestmark = pytest.mark.gpu


def rand(seed, shape, scale=1.0):
    return (scale * np.random.default_rng(seed).standard_normal(shape)).astype(np.float16).view(np.uint16)


# Splits and keys per split of the cases below that are there for them (256 CUs).
SPLITS = {(64, 31): (1, 32), (64, 128): (2, 96), (64, 384): (4, 128), (64, 4999): (32, 160), (8, 9000): (71, 128)}


@pytest.mark.parametrize("hq,hkv,d,T,off,extra,causal,kind", [
    (8, 1, 128, 1, 0, 0, True, "flash-decode"),        # one key
    (64, 8, 128, 1, 31, 0, True, "decode-split-kv"),   # one whole tile, one split
    (64, 8, 128, 1, 128, 0, True, "flash-decode"),     # 129 keys: splits of 96 and 33
    (64, 8, 128, 1, 384, 0, True, "flash-decode"),     # a fourth split of one key
    (32, 8, 128, 1, 255, 9, True, "flash-decode"),     # keys past the window are not read
    (32, 8, 128, 1, 99, 57, False, "flash-decode"),    # non-causal: every key
    (64, 8, 128, 1, 4999, 0, True, "flash-decode"),    # 32 splits: a whole merge pass
    (8, 1, 128, 1, 9000, 0, True, "flash-decode"),     # 71 splits: three merge passes
    (17, 1, 128, 1, 9000, 0, True, "flash-decode"),    # two head chunks of 9 and 8
    (40, 2, 64, 1, 777, 0, True, "decode-split-kv"),   # two head chunks of 10
    (32, 8, 64, 1, 300, 0, True, "flash-decode"),
    (16, 8, 64, 1, 5000, 0, True, "flash-decode"),
    (32, 8, 128, 2, 30, 0, True, "tiled"),             # two tokens, windows across a tile edge
    (32, 8, 128, 4, 3001, 0, True, "tiled"),           # 16 rows
    (15, 3, 128, 3, 4400, 5, True, "tiled"),           # 15 rows of 5 heads
    (16, 8, 64, 8, 1900, 0, False, "tiled"),
    (12, 1, 64, 1, 2047, 0, True, "tiled"),
])
def test_few_row_attention(ctx, hq, hkv, d, T, off, extra, causal, kind):
    L = off + T + extra
    q, k, v = rand(1, (T, hq, d), 2.0), rand(2, (L, hkv, d)), rand(3, (L, hkv, d))
    geo = dict(hq=hq, hkv=hkv, d=d, off=off, causal=causal)
    qt, (ko, kview) = ctx.tensor(q), upload_kv(ctx, k, "head_major")
    info = ctx.plan(qt, kview, kview, mi_attn.AttentionConfig(hq, hkv, d, causal, off), KINDS[kind])
    if (hq, off) in SPLITS:
        assert (info["splits"], info["block_keys"]) == SPLITS[hq, off], info
    group, chunks = hq // hkv, 1 if T > 1 else -(-hq // hkv // 16)
    rows = T * -(-group // chunks)
    assert info["kernel"] == "attn_decode" and info["block_threads"] == 512 and info["grid"][1] == hkv * chunks, info
    assert info["scratch_bytes"] in (0, info["grid"][1] * info["splits"] * rows * (d + 2) * 4), info
    out = run_attention(ctx, q, k, v, kind=kind, layout="position_major", **geo)
    again = run_attention(ctx, q, k, v, kind=kind, layout="head_major", **geo)
    # f16 inputs, f32 probabilities (22 bits in the products) and sums: one
    # rounding of the output, a few f32 roundings of the sums before it.
    ref = oracle_attention(q, k, v, **geo)["f32"]
    bound = np.abs(ref) * 2.0 ** -11 + 2.0 ** -24 + 1e-5
    assert (np.abs(f16(out).astype(np.float64) - ref) <= bound).all()
    assert (again == out).all()


@pytest.mark.parametrize("d,T,off,kind", [(128, 1, 2300, "flash-decode"), (64, 1, 700, "flash-decode"),
                                          (128, 2, 400, "tiled")])
def test_few_row_attention_with_infinite_values(ctx, d, T, off, kind):
    """An infinite value reaches the rows that see its key and no others, as a weighted sum over
    the visible keys gives it."""
    hq, hkv, L = 8, 1, off + T
    q, k, v = rand(4, (T, hq, d)), rand(5, (L, hkv, d)), rand(6, (L, hkv, d))
    v[L - 1, 0, 5] = np.float16(np.inf).view(np.uint16)      # the last token's own key
    v[off // 2, 0, d - 1] = np.float16(-np.inf).view(np.uint16)
    geo = dict(hq=hq, hkv=hkv, d=d, off=off)
    ref = oracle_attention(q, k, v, **geo)["f32"]
    got = f16(run_attention(ctx, q, k, v, kind=kind, **geo))
    assert (np.isposinf(ref) == np.isposinf(got)).all() and (np.isneginf(ref) == np.isneginf(got)).all()
    fine = np.isfinite(ref)
    assert np.isfinite(got[fine]).all() and np.abs(got[fine] - ref[fine]).max() <= 2e-3


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("T,off,kind", [(1, 2300, "flash-decode"), (2, 400, "tiled"), (90, 600, "tiled"),
                                        (90, 0, "tiled")])
@pytest.mark.parametrize("what", ["nan key", "nan value", "nan row", "infinite row"])
def test_values_that_are_not_finite(ctx, d, T, off, kind, what):
    """A NaN or an infinity in a key or value row reaches the rows that see it, in the columns that
    it has, and no others."""
    hq, hkv, L = 16, 2, off + T
    q, k, v = rand(4, (T, hq, d)), rand(5, (L, hkv, d)), rand(6, (L, hkv, d))
    at = off + T // 2 if T > 2 else L // 2
    bad = np.float16(np.inf if what == "infinite row" else np.nan).view(np.uint16)
    if what == "nan key":
        k[at, 0, 3] = bad
    elif what == "nan value":
        v[at, 0, d - 1] = bad
    else:
        v[at, 0] = bad
    geo = dict(hq=hq, hkv=hkv, d=d, off=off)
    ref = oracle_attention(q, k, v, **geo)["f32"]
    got = f16(run_attention(ctx, q, k, v, kind=kind, **geo))
    assert (np.isnan(ref) == np.isnan(got)).all() and (np.isposinf(ref) == np.isposinf(got)).all()
    fine = np.isfinite(ref)
    assert not fine.all() and np.abs(got[fine] - ref[fine]).max() <= 2e-3


def fastest(ctx, call, runs=5):
    """The fastest of a few calls, in ns of its kernels."""
    best = float("inf")
    ctx.set_kernel_profiling(True)
    try:
        for _ in range(runs):
            ctx.take_kernel_profiles()
            batch = ctx.begin_batch()
            keep = call(batch)
            batch.finish()
            best = min(best, sum(ns for _, ns in ctx.take_kernel_profiles()))
            del keep
    finally:
        ctx.set_kernel_profiling(False)
    return best


@pytest.mark.parametrize("hq,hkv,d,T,L,kind,most", [
    (64, 8, 64, 1, 20000, "flash-decode", 2.6),
    (32, 8, 64, 200, 2000, "tiled", 7.0),
    (32, 8, 128, 200, 2000, "tiled", 8.0),
])
def test_a_row_that_is_not_finite_costs_no_serial_walk(ctx, hq, hkv, d, T, L, kind, most):
    """One NaN value row takes its tiles to the vector units, not every key of the call to a chain of
    loads: at most `most` times the finite call (a key at a time measured 4 and 11 to 14 times)."""
    q, k, v = rand(1, (T, hq, d)), rand(2, (L, hkv, d)), rand(3, (L, hkv, d))
    qt, (ko, kview), (vo, vview) = ctx.tensor(q), upload_kv(ctx, k, "head_major"), upload_kv(ctx, v, "head_major")
    cfg = mi_attn.AttentionConfig(hq, hkv, d, True, L - T)
    v[L // 2] = np.float16(np.nan).view(np.uint16)
    bo, bview = upload_kv(ctx, v, "head_major")
    finite = fastest(ctx, lambda b: b.attention(qt, kview, vview, cfg, KINDS[kind]))
    nan = fastest(ctx, lambda b: b.attention(qt, kview, bview, cfg, KINDS[kind]))
    assert nan <= most * finite, (nan, finite)


@pytest.mark.parametrize("hq,hkv,pos", [(64, 8, 0), (64, 8, 32), (8, 1, 300), (40, 2, 1700), (32, 8, 3500),
                                        (17, 1, 9000)])
def test_decode_step_on_the_mfma_kernel(ctx, hq, hkv, pos):
    """The one-launch step: no cached key, splits and head chunks; the cache row that it writes is
    the only one that changes, and what the row held before has no influence."""
    d, cap = 128, pos + 2
    q, k, v = rand(1, (1, hq, d)), rand(2, (1, hkv, d)), rand(3, (1, hkv, d))
    qw, kw = rand(4, (d,), 0.3), rand(5, (d,), 0.3)
    hist_k, hist_v = rand(6, (cap, hkv, d)), rand(7, (cap, hkv, d))
    hist_k[pos], hist_v[pos] = 0x7e00, 0x7e00  # NaN until the step writes it
    cache = ctx.kv_cache(1, hkv, d, cap)
    key, value = cache.layer(0)
    ctx.upload(key, hist_k)
    ctx.upload(value, hist_v)
    tensors = [ctx.tensor(x) for x in (q, k, v, qw, kw)]
    ctx.take_kernel_profiles()
    ctx.set_kernel_profiling(True)
    batch = ctx.begin_batch()
    out = batch.decode_step_attention(*tensors, key, value, mi_attn.QkNormRopeCacheConfig(pos, 1e6, 1e-6),
                                      mi_attn.AttentionConfig(hq, hkv, d, True, pos))
    batch.finish()
    ctx.set_kernel_profiling(False)
    assert [name for name, _ in ctx.take_kernel_profiles()] == ["attn_decode_step_mfma"]
    got, key_now, value_now = ctx.download(out), ctx.download(key), ctx.download(value)
    others = np.arange(cap) != pos
    assert (key_now[others] == hist_k[others]).all() and (value_now[others] == hist_v[others]).all()
    assert (value_now[pos] == v[0]).all()
    want_q, want_k = oracle.qk_norm_rope(q, k, qw, kw, offset=pos, theta=1e6, epsilon=1e-6)
    assert np.abs(f16(key_now[pos]) - f16(want_k[0])).max() <= 2e-3
    ref = oracle_attention(want_q, key_now[:pos + 1], value_now[:pos + 1], hq=hq, hkv=hkv, d=d, off=pos)
    assert_parity(got, ref, label=f"{hq}/{hkv} pos {pos}")
    cache.close()


@pytest.mark.parametrize("at", [0, 700, 899, 900])
def test_decode_step_with_infinite_values(ctx, at):
    """An infinite value in the cache (900 is the new token's own) reaches its column of every head."""
    hq, hkv, d, pos = 16, 2, 128, 900
    q, k, v = rand(1, (1, hq, d)), rand(2, (1, hkv, d)), rand(3, (1, hkv, d))
    qw, kw = rand(4, (d,), 0.3), rand(5, (d,), 0.3)
    hist_k, hist_v = rand(6, (pos + 1, hkv, d)), rand(7, (pos + 1, hkv, d))
    (v[0] if at == pos else hist_v[at])[1, 5] = np.float16(-np.inf).view(np.uint16)
    cache = ctx.kv_cache(1, hkv, d, pos + 1)
    key, value = cache.layer(0)
    ctx.upload(key, hist_k)
    ctx.upload(value, hist_v)
    tensors = [ctx.tensor(x) for x in (q, k, v, qw, kw)]
    batch = ctx.begin_batch()
    out = batch.decode_step_attention(*tensors, key, value, mi_attn.QkNormRopeCacheConfig(pos, 1e6, 1e-6),
                                      mi_attn.AttentionConfig(hq, hkv, d, True, pos))
    batch.finish()
    got = f16(ctx.download(out))
    want_q, _ = oracle.qk_norm_rope(q, k, qw, kw, offset=pos, theta=1e6, epsilon=1e-6)
    ref = oracle_attention(want_q, ctx.download(key), ctx.download(value), hq=hq, hkv=hkv, d=d, off=pos)["f32"]
    assert (np.isneginf(ref) == np.isneginf(got)).all() and np.isneginf(got).sum() == hq // hkv
    fine = np.isfinite(ref)
    assert np.abs(got[fine] - ref[fine]).max() <= 2e-3
    cache.close()
