"""Tiled attention of several tokens on MFMA (attn_tiled.hip) at the edges of its row tiles, key
tiles and splits, against the oracle."""
import numpy as np
import pytest

import mi_attn
from helpers import f16, oracle_attention, run_attention, upload_kv

pytestmark = pytest.mark.gpu


def rand(seed, shape, scale=1.0):
    return (scale * np.random.default_rng(seed).standard_normal(shape)).astype(np.float16).view(np.uint16)


@pytest.mark.parametrize("hq,hkv,d,T,off,extra,causal", [
    (32, 8, 128, 24, 1100, 0, True),   # 96 rows: the last wave only loads
    (32, 8, 128, 32, 480, 0, True),    # 128 rows, 8 whole key tiles
    (32, 8, 128, 33, 480, 0, True),    # a second row tile of 4 rows; a key tile of one key
    (10, 2, 128, 31, 700, 40, True),   # rows of 5 heads across the waves; keys past the window
    (10, 2, 128, 31, 700, 40, False),
    (16, 8, 64, 29, 3000, 0, True),
    (8, 1, 64, 300, 5, 0, True),       # many row tiles, splits cut at each one's window
    (8, 8, 128, 500, 0, 0, True),      # one head per group, no split
    (4, 1, 128, 31, 20000, 0, True),   # 157 splits of two tiles
])
def test_tiled_attention(ctx, hq, hkv, d, T, off, extra, causal):
    L = off + T + extra
    q, k, v = rand(1, (T, hq, d), 2.0), rand(2, (L, hkv, d)), rand(3, (L, hkv, d))
    geo = dict(hq=hq, hkv=hkv, d=d, off=off, causal=causal)
    qt, (ko, kview) = ctx.tensor(q), upload_kv(ctx, k, "head_major")
    info = ctx.plan(qt, kview, kview, mi_attn.AttentionConfig(hq, hkv, d, causal, off), mi_attn.TILED)
    assert info["kernel"] == "attn_tiled" and info["grid"][1] == -(-T * hq // hkv // 128), info
    out = run_attention(ctx, q, k, v, kind="tiled", layout="position_major", **geo)
    again = run_attention(ctx, q, k, v, kind="tiled", layout="head_major", **geo)
    # f16 inputs, f32 probabilities (22 bits in the products) and sums: one
    # rounding of the output, a few f32 roundings of the sums before it.
    ref = oracle_attention(q, k, v, **geo)["f32"]
    bound = np.abs(ref) * 2.0 ** -11 + 2.0 ** -24 + 1e-5
    assert (np.abs(f16(out).astype(np.float64) - ref) <= bound).all(), info
    assert (again == out).all()


@pytest.mark.parametrize("off", [0, 900])
def test_tiled_attention_with_infinite_values(ctx, off):
    """An infinite value reaches the rows that see its key and no others."""
    hq, hkv, d, T = 8, 2, 128, 90
    L = off + T
    q, k, v = rand(4, (T, hq, d)), rand(5, (L, hkv, d)), rand(6, (L, hkv, d))
    v[off + 50, 0, 5] = np.float16(np.inf).view(np.uint16)
    v[L - 1, 1, 0] = np.float16(-np.inf).view(np.uint16)
    geo = dict(hq=hq, hkv=hkv, d=d, off=off)
    ref = oracle_attention(q, k, v, **geo)["f32"]
    got = f16(run_attention(ctx, q, k, v, kind="tiled", **geo))
    assert (np.isposinf(ref) == np.isposinf(got)).all() and (np.isneginf(ref) == np.isneginf(got)).all()
    fine = np.isfinite(ref)
    assert np.isfinite(got[fine]).all() and np.abs(got[fine] - ref[fine]).max() <= 2e-3
