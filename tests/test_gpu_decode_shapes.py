"""Seeded random batched-decode geometries against the oracle: 1-48
sequences, GQA ratios 1-16, head_dim 128 (by default the stream-K MFMA kernel
and its merge launch) and 64 (by default that or the rows kernel, by heads and
units), per-sequence lengths from 0 to past the cache capacity (clamped),
head-major and token-major caches, the default plan and explicit split sizes
(the rows kernel, splits merged inside the launch). Every sequence is checked (a zero-length one must be NaN, the
reference's 0/0), a second call must be bit-identical, and the
no-allocation entry point must agree bit for bit where its buffer holds the
partials."""
from __future__ import annotations

import numpy as np
import pytest

import mi_attn
from helpers import assert_parity, oracle_attention

pytestmark = pytest.mark.gpu

CASES = 30


def _geometry(i: int):
    rng = np.random.default_rng(7000 + i)
    d = int(rng.choice([128, 128, 64]))
    hkv = int(rng.choice([1, 2, 4, 8]))
    g = int(rng.choice([1, 2, 4, 8, 16]))
    B = int(rng.integers(1, 49))
    cap = int(rng.integers(16, 1500))
    lengths = rng.integers(0, cap + 40, B)
    lengths[rng.random(B) < 0.1] = 0
    block = int(rng.choice([0, 0, 0, 64, 192]))
    token_major = bool(rng.random() < 0.3)
    return rng, d, hkv * g, hkv, B, cap, lengths.astype(np.uint32), block, token_major


# What each kind of call launches.
KERNELS = {
    "stream-128": ["attn_decode_stream", "attn_decode_stream_merge"],
    "stream-64": ["attn_decode_stream", "attn_decode_stream_merge"],
    "rows-default": ["attn_rows_batched"],
    "rows-split": ["attn_rows_batched"],
}


def _kind(cus, i):
    """The default at head_dim 64 is stream-K for groups of 8, for larger groups than 4 of nine
    heads per CU, and for groups of 4 whose rows splits come to six workgroups per CU (not
    between one unit and six per CU), as long as there are at least
    two KV heads and more keys than one rows split."""
    _, d, hq, hkv, B, cap, _, block, _ = _geometry(i)
    if block != 0:
        return "rows-split"
    if d == 128:
        return "stream-128"
    g, units = hq // hkv, B * hkv
    four = g == 4 and units * -(-cap // 768) >= 6 * cus and not cus < units < 6 * cus
    many = g == 8 or (g > 4 and B * hq >= 9 * cus) or four
    return "stream-64" if cap > 768 and hkv > 1 and many else "rows-default"


@pytest.mark.parametrize("i", range(CASES))
def test_random_batched_decode_geometry(ctx, i):
    rng, d, hq, hkv, B, cap, lengths, block, token_major = _geometry(i)
    q = rng.standard_normal((B, hq, d)).astype(np.float16).view(np.uint16)
    k = rng.standard_normal((B, cap, hkv, d)).astype(np.float16).view(np.uint16)
    v = rng.standard_normal((B, cap, hkv, d)).astype(np.float16).view(np.uint16)
    if token_major:
        kt, vt = ctx.tensor(k), ctx.tensor(v)
        kview, vview = kt, vt
    else:  # head-major storage [B, Hkv, cap, D] seen as [B, cap, Hkv, D]
        kt = ctx.tensor(np.ascontiguousarray(k.transpose(0, 2, 1, 3)))
        vt = ctx.tensor(np.ascontiguousarray(v.transpose(0, 2, 1, 3)))
        view = ((B, cap, hkv, d), (hkv * cap * d, d, cap * d, 1))
        kview, vview = kt.view(*view), vt.view(*view)
    qt, lt = ctx.tensor(q), ctx.tensor(lengths, mi_attn.U32)
    cfg = mi_attn.AttentionConfig(hq, hkv, d, True, 0)
    label = (f"case {i}: d={d} hq={hq} hkv={hkv} B={B} cap={cap} block={block} "
             f"token_major={token_major}")
    outs = []
    ctx.take_kernel_profiles()
    ctx.set_kernel_profiling(True)
    try:
        for _ in range(2):
            batch = ctx.begin_batch()
            out = batch.attention_decode_batched(qt, kview, vview, lt, cfg, block)
            batch.finish()
            outs.append(ctx.download(out))
        names = [name for name, _ in ctx.take_kernel_profiles()]
    finally:
        ctx.set_kernel_profiling(False)
    assert names == KERNELS[_kind(ctx.compute_units, i)] * 2, (label, names)
    got = outs[0]
    assert np.array_equal(got.view(np.uint16), outs[1].view(np.uint16)), label
    for b in range(B):
        n = min(int(lengths[b]), cap)
        if n == 0:
            assert np.isnan(got[b].view(np.float16).astype(np.float32)).all(), label
            continue
        ref = oracle_attention(q[b:b + 1], k[b, :n], v[b, :n], hq=hq, hkv=hkv, d=d, off=n - 1)
        assert_parity(got[b:b + 1], ref, label=f"{label} seq {b} len {n}")
    fixed = ctx.empty(q.shape)
    batch = ctx.begin_batch()
    try:
        batch.attention_decode_batched_noalloc(qt, kview, vview, lt, cfg, block, fixed)
    except mi_attn.MiError as err:  # partials larger than the fixed buffer
        batch.abandon()
        assert err.name == "MI_ERR_RESOURCE", (label, err)
    else:
        batch.finish()
        assert np.array_equal(ctx.download(fixed).view(np.uint16), got.view(np.uint16)), label


def test_random_decode_geometries_cover_every_route():
    """The sample above holds stream-K calls at both head dimensions, default
    calls that stay on the rows kernel and explicit splits (each call is checked
    to have run its kernels), both cache layouts, zero lengths and lengths past
    the capacity."""
    kinds, layouts, zero, clamped = set(), set(), 0, 0
    for i in range(CASES):
        _, _, _, _, _, cap, lengths, _, token_major = _geometry(i)
        kinds.add(_kind(256, i))
        layouts.add(token_major)
        zero += int((lengths == 0).any())
        clamped += int((lengths > cap).any())
    assert kinds == set(KERNELS), kinds
    assert layouts == {True, False}
    assert zero > 0 and clamped > 0
