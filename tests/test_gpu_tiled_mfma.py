"""Tiled attention of several tokens on MFMA (attn_tiled.hip) at the edges of its row tiles, key
tiles and splits, against the oracle."""
import numpy as np
import pytest

import mi_attn
from helpers import f16, oracle_attention, run_attention, upload_kv

pytestmark = pytest.mark.gpu


def rand(seed, shape, scale=1.0):
    return (scale * np.random.default_rng(seed).standard_normal(shape)).astype(np.float16).view(np.uint16)


@pytest.mark.parametrize("hq,hkv,d,T,off,extra,causal,splits,split_keys", [
    (32, 8, 128, 24, 1100, 0, True, 9, 128),    # 96 rows: the last wave only loads
    (32, 8, 128, 32, 480, 0, True, 4, 128),     # 128 rows, 8 whole key tiles
    (32, 8, 128, 33, 480, 0, True, 3, 192),     # a second row tile of 4 rows; a key tile of one key
    (10, 2, 128, 31, 700, 40, True, 6, 128),    # rows of 5 heads across the waves; keys past the window
    (10, 2, 128, 31, 700, 40, False, 5, 192),
    (16, 8, 64, 29, 3000, 0, True, 24, 128),
    (8, 1, 64, 300, 5, 0, True, 1, 0),          # 19 row tiles, no split
    (8, 1, 64, 500, 5, 0, True, 4, 128),        # row tiles whose windows need 1 to 4 splits
    (8, 8, 128, 500, 0, 0, True, 4, 128),       # one head per group, the same
    (4, 1, 128, 31, 20000, 0, True, 105, 192),  # 105 splits of three tiles
])
def test_tiled_attention(ctx, hq, hkv, d, T, off, extra, causal, splits, split_keys):
    L = off + T + extra
    q, k, v = rand(1, (T, hq, d), 2.0), rand(2, (L, hkv, d)), rand(3, (L, hkv, d))
    geo = dict(hq=hq, hkv=hkv, d=d, off=off, causal=causal)
    qt, (ko, kview) = ctx.tensor(q), upload_kv(ctx, k, "head_major")
    info = ctx.plan(qt, kview, kview, mi_attn.AttentionConfig(hq, hkv, d, causal, off), mi_attn.TILED)
    assert info["kernel"] == "attn_tiled" and info["grid"][1] == -(-T * hq // hkv // 128), info
    assert (info["splits"], info["block_keys"]) == (splits, split_keys), info
    out = run_attention(ctx, q, k, v, kind="tiled", layout="position_major", **geo)
    again = run_attention(ctx, q, k, v, kind="tiled", layout="head_major", **geo)
    # f16 inputs, f32 probabilities (22 bits in the products) and sums: one
    # rounding of the output, a few f32 roundings of the sums before it.
    ref = oracle_attention(q, k, v, **geo)["f32"]
    bound = np.abs(ref) * 2.0 ** -11 + 2.0 ** -24 + 1e-5
    assert (np.abs(f16(out).astype(np.float64) - ref) <= bound).all(), info
    assert (again == out).all()


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("off", [0, 900])
def test_tiled_attention_with_infinite_values(ctx, off, d):
    """An infinite value reaches the rows that see its key and no others."""
    hq, hkv, T = 8, 2, 90
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
