"""The attention work that a program on this framework has it do, as cases to time.

Every case is the attention half of a transformer block, for `layers` layers with their own
weights and KV cache (as a model's forward pass meets them: cold), through the calls that a
program makes per layer: Q/K norm + RoPE with the KV append, attention, o_proj. Layers do not
feed one another, so each output carries the rounding of its own layer only.

`op` is what kind of pass it is:
  step     one token of one sequence, `mi_decode_step_attention` + o_proj, a captured graph
  token    one token of one sequence, the separate calls of the reference's forward_layer
           (norm + RoPE + key append, value append, FlashDecode, o_proj), a captured graph
  batch    one token of each of `batch` sequences of ragged lengths: batched decode + o_proj, a
           captured graph (lengths are device data, so a server replays it for many tokens)
  prefill  `tokens` new tokens of one sequence on `offset` cached ones, fused Q/K path, the
           attention kind by the framework's own policy; a captured graph at offset 0, else an
           eager batch per pass
  unfused  the same with the unfused Q/K path (rms_norm, rope, copy_into_cache)

Sizes: the repository's benchmark configurations (16/8, 32/8 and 64/8 heads of 128 with hidden
sizes 1024, 4096 and 5120), 40/8 heads, and the other head dimensions that its kernels serve.
"""
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "metal-infer-rs_amd"))
import mi_attn  # noqa: E402

THETA, EPS = 1_000_000.0, 1e-6
# (query heads, KV heads, hidden size) of the models that the repository is measured on, and 40/8.
GEOMETRIES = [(16, 8, 1024), (32, 8, 4096), (40, 8, 5120), (64, 8, 5120)]


def listed():
    return [
        # A short chat's next token on the smallest model: launches and latency.
        dict(name="step 16/8 L301", op="step", layers=28, tokens=1, offset=300, q_heads=16, kv_heads=8,
             head_dim=128, hidden=1024, batch=1),
        # A longer chat's next token with the reference's separate calls.
        dict(name="token 32/8 L4100", op="token", layers=12, tokens=1, offset=4099, q_heads=32, kv_heads=8,
             head_dim=128, hidden=4096, batch=1),
        # The next token over a long document, the largest heads.
        dict(name="token 64/8 L32768", op="token", layers=3, tokens=1, offset=32767, q_heads=64, kv_heads=8,
             head_dim=128, hidden=5120, batch=1),
        # A lightly loaded server: few sequences, short and ragged.
        dict(name="batch 8 16/8 L40-1000", op="batch", layers=14, tokens=1, offset=0, q_heads=16, kv_heads=8,
             head_dim=128, hidden=1024, batch=8, low=40, high=1000, capacity=1024),
        # The repository's headline: 32 sequences of 1024 to 8192 tokens.
        dict(name="batch 32 32/8 L1024-8192", op="batch", layers=2, tokens=1, offset=0, q_heads=32, kv_heads=8,
             head_dim=128, hidden=4096, batch=32, low=1024, high=8192, capacity=8192),
        # Many sequences at the other common head dimension.
        dict(name="batch 70 32/8/64 L100-4000", op="batch", layers=2, tokens=1, offset=0, q_heads=32, kv_heads=8,
             head_dim=64, hidden=2048, batch=70, low=100, high=4000, capacity=4096),
        # A short prompt on the smallest model.
        dict(name="prefill 16/8 T128", op="prefill", layers=28, tokens=128, offset=0, q_heads=16, kv_heads=8,
             head_dim=128, hidden=1024, batch=1),
        # A long prompt on the smallest model.
        dict(name="prefill 16/8 T2048", op="prefill", layers=8, tokens=2048, offset=0, q_heads=16, kv_heads=8,
             head_dim=128, hidden=1024, batch=1),
        # A chunk of a long prompt, the largest heads.
        dict(name="prefill 64/8 T4096@16384", op="prefill", layers=1, tokens=4096, offset=16384, q_heads=64,
             kv_heads=8, head_dim=128, hidden=5120, batch=1),
        # A ragged prompt at head dimension 64 with the unfused Q/K path.
        dict(name="unfused 32/8/64 T1100", op="unfused", layers=8, tokens=1100, offset=0, q_heads=32, kv_heads=8,
             head_dim=64, hidden=2048, batch=1),
        # A chat's next question: a few new tokens on a cached conversation.
        dict(name="turn 32/8 T24@6000", op="prefill", layers=8, tokens=24, offset=6000, q_heads=32, kv_heads=8,
             head_dim=128, hidden=4096, batch=1),
        # A longer question about a cached document, the largest heads.
        dict(name="turn 64/8 T200@12000", op="prefill", layers=4, tokens=200, offset=12000, q_heads=64,
             kv_heads=8, head_dim=128, hidden=5120, batch=1),
    ]


def _spread(rng, low, high):
    """A whole number from low to high, even over its logarithm."""
    return min(high, int(low * (high / low) ** rng.random() + rng.random()))


def draw(rng):
    op = rng.choice(["step", "token", "batch", "batch", "prefill", "prefill", "turn", "unfused"])
    q_heads, kv_heads, hidden = rng.choice(GEOMETRIES)
    head_dim = rng.choice([128, 128, 128, 128, 128, 128, 64, 64, 256])
    if head_dim == 256:
        q_heads = min(q_heads, 32)
    case = dict(op=op, layers=1, tokens=1, offset=0, q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim,
                hidden=hidden, batch=1)
    if op in ("step", "token"):
        case["offset"] = _spread(rng, 16, 40000)
        keys = case["offset"] + 1
    elif op == "batch":
        case["batch"] = _spread(rng, 2, 128)
        high = min(8192, 200_000 // case["batch"])
        case["high"] = _spread(rng, 64, high)
        case["low"] = max(1, int(case["high"] * rng.uniform(0.02, 0.9)))
        case["capacity"] = -(-case["high"] // 64) * 64 + 64 * rng.randint(0, 3)
        keys = case["batch"] * (case["low"] + case["high"]) // 2
    else:
        short = op == "turn"
        case["op"] = "prefill" if short else op
        case["tokens"] = _spread(rng, 2, 400) if short else _spread(rng, 33, 3000)
        case["offset"] = _spread(rng, 300, 20000) if short else rng.choice([0, 0, _spread(rng, 100, 8000)])
        keys = case["offset"] + case["tokens"]
    # As many layers as keep a pass near half a millisecond, at most what a model has.
    row = 4 * kv_heads * head_dim
    cost = keys * row + 2 * q_heads * head_dim * hidden + 20e6 + (work(case)["flops"] / 100)
    case["layers"] = max(1, min(28, int(1.5e9 / cost)))
    return case


# ------------------------------------------------------------------- inputs --

def _lengths(case, seed):
    r = np.random.default_rng(seed % (1 << 32))
    return r.integers(case["low"], case["high"] + 1, case["batch"]).astype(np.uint32)


def _inputs(case, seed):
    """Inputs and KV caches from the seed alone (torch tensors on the GPU)."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    n, t, hq, hkv, d = (case[k] for k in ("layers", "tokens", "q_heads", "kv_heads", "head_dim"))

    def normal(*shape, scale=1.0):
        return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float16).mul_(scale)

    def norm_weight():
        return torch.rand(n, d, generator=g, device="cuda").mul_(1.5).add_(0.5).half()

    x = {"proj_weight": normal(n, case["hidden"], hq * d, scale=(hq * d) ** -0.5)}
    if case["op"] == "batch":
        b, c = case["batch"], case["capacity"]
        x["q"] = normal(n, b, hq, d, scale=1.5)
        x["key"], x["value"] = normal(n, b, hkv, c, d), normal(n, b, hkv, c, d)
        x["lengths"] = torch.from_numpy(_lengths(case, seed).astype(np.int32)).cuda()
        return x
    c = -(-(case["offset"] + t + 1) // 512) * 512
    # The rows of a fused QKV projection, as a model hands them over.
    x["qkv"] = normal(n, t, hq + 2 * hkv, d)
    x["q_weight"], x["k_weight"] = norm_weight(), norm_weight()
    x["key"], x["value"] = normal(n, hkv, c, d), normal(n, hkv, c, d)
    return x


_context = None


def _ctx():
    """The program's one context."""
    global _context
    if _context is None:
        _context = mi_attn.Context(torch.cuda.current_device())
    return _context


def _view(t, shape=None, strides=None, dtype=mi_attn.F16):
    shape = tuple(t.shape) if shape is None else shape
    strides = tuple(t.stride()) if strides is None else strides
    return mi_attn.Tensor(mi_attn.describe(t.data_ptr(), shape, strides, dtype))


def _cache_view(t):
    """[Hkv, C, D] head-major storage as the logical [C, Hkv, D] (batched: [B, C, Hkv, D])."""
    return _view(t.transpose(-2, -3))


def prepare(case, seed):
    ctx = _ctx()
    x = _inputs(case, seed)
    n, t, hq, hkv, d = (case[k] for k in ("layers", "tokens", "q_heads", "kv_heads", "head_dim"))
    rows = case["batch"] if case["op"] == "batch" else t
    attn = torch.empty(n, rows, hq, d, device="cuda", dtype=torch.float16)
    proj = torch.empty(n, rows, case["hidden"], device="cuda", dtype=torch.float16)
    state = dict(x=x, out={"attention": attn, "proj": proj}, pending=None, graph=None)
    cfg = mi_attn.AttentionConfig(hq, hkv, d, True, case["offset"])
    layers = []
    for i in range(n):
        w = dict(cfg=cfg, attn=_view(attn[i]), rows=_view(attn[i].view(rows, hq * d)), proj=_view(proj[i]),
                 proj_weight=_view(x["proj_weight"][i]), key=_cache_view(x["key"][i]),
                 value=_cache_view(x["value"][i]))
        if case["op"] == "batch":
            w["q"] = _view(x["q"][i])
            w["lengths"] = _view(x["lengths"], dtype=mi_attn.U32)
        else:
            qkv = x["qkv"][i]
            w["q"], w["k"], w["v"] = _view(qkv[:, :hq]), _view(qkv[:, hq:hq + hkv]), _view(qkv[:, hq + hkv:])
            w["q_weight"], w["k_weight"] = _view(x["q_weight"][i]), _view(x["k_weight"][i])
            w["rope"] = mi_attn.QkNormRopeCacheConfig(case["offset"], THETA, EPS)
            length = case["offset"] + t
            w["active_key"], w["active_value"] = w["key"].prefix(length), w["value"].prefix(length)
            # The model's configured kind is Tiled, the reference's default.
            w["kind"] = mi_attn.attention_kind_for_tokens(mi_attn.TILED, t, length, hq // hkv)
        layers.append(w)
    if case["op"] != "batch":
        o = case["offset"]
        state["out"].update(key=x["key"], value=x["value"], new_key=x["key"][:, :, o:o + t],
                            new_value=x["value"][:, :, o:o + t])
    state["layers"], state["layer"] = layers, _LAYER[case["op"]]
    torch.cuda.synchronize()  # the inputs were made on torch's stream, the calls run on the context's
    # A program warms up once and captures what it replays: a token's launches, and prompts from
    # position 0 (padded to lengths that it keeps a graph for). A chunk or a turn at a position of
    # its own is enqueued as it comes.
    if t == 1 or case["offset"] == 0:
        batch = ctx.begin_batch()
        state["layer"](batch, layers[0])
        batch.finish()
        batch = ctx.begin_capture()
        for w in layers:
            state["layer"](batch, w)
        state["graph"] = batch.end_capture()
    return state


# --------------------------------------------------------------------- runs --

def _step(batch, w):
    batch.decode_step_attention(w["q"], w["k"], w["v"], w["q_weight"], w["k_weight"], w["key"], w["value"],
                                w["rope"], w["cfg"], out=w["attn"])
    batch.matmul(w["rows"], w["proj_weight"], out=w["proj"])


def _token(batch, w):
    q = batch.qk_norm_rope_cache(w["q"], w["k"], w["q_weight"], w["k_weight"], w["key"], w["rope"])
    batch.copy_into_cache(w["v"], w["value"], w["rope"].offset)
    batch.attention(q, w["active_key"], w["active_value"], w["cfg"], w["kind"], out=w["attn"])
    batch.matmul(w["rows"], w["proj_weight"], out=w["proj"])


def _batch(batch, w):
    batch.attention_decode_batched(w["q"], w["key"], w["value"], w["lengths"], w["cfg"], out=w["attn"])
    batch.matmul(w["rows"], w["proj_weight"], out=w["proj"])


def _prefill(batch, w):
    q = batch.qk_norm_rope_cache_value(w["q"], w["k"], w["v"], w["q_weight"], w["k_weight"], w["key"],
                                       w["value"], w["rope"])
    batch.attention(q, w["active_key"], w["active_value"], w["cfg"], w["kind"], out=w["attn"])
    batch.matmul(w["rows"], w["proj_weight"], out=w["proj"])


def _unfused(batch, w):
    offset = w["rope"].offset
    q = batch.rope(batch.rms_norm(w["q"], w["q_weight"], EPS), offset, THETA)
    k = batch.rope(batch.rms_norm(w["k"], w["k_weight"], EPS), offset, THETA)
    batch.copy_into_cache(k, w["key"], offset)
    batch.copy_into_cache(w["v"], w["value"], offset)
    batch.attention(q, w["active_key"], w["active_value"], w["cfg"], w["kind"], out=w["attn"])
    batch.matmul(w["rows"], w["proj_weight"], out=w["proj"])


_LAYER = {"step": _step, "token": _token, "batch": _batch, "prefill": _prefill, "unfused": _unfused}


def run(state):
    """One pass: a graph replay, or an eager batch that is committed and, as a program with
    two batches in flight does, waited for when its buffers are used again."""
    if state["graph"] is not None:
        state["graph"].launch()
        return state["out"]
    if state["pending"] is not None:
        state["pending"].wait()
    batch = _ctx().begin_batch()
    for w in state["layers"]:
        state["layer"](batch, w)
    state["pending"] = batch.commit()
    return state["out"]


# ------------------------------------------------------- work and exactness --

def _mean_keys(case):
    return case["batch"] * (case["low"] + case["high"]) / 2


def work(case):
    n, t, hq, hkv, d = (case[k] for k in ("layers", "tokens", "q_heads", "kv_heads", "head_dim"))
    rows = case["batch"] if case["op"] == "batch" else t
    if case["op"] == "batch":
        keys = pairs = _mean_keys(case)
        inputs = rows * hq * d
        written = 0
    else:
        keys = case["offset"] + t
        pairs = t * case["offset"] + t * (t + 1) // 2
        inputs = t * (hq + 2 * hkv) * d + 2 * d
        written = 2 * t * hkv * d
    halves = 2 * keys * hkv * d + inputs + written + rows * hq * d  # KV, Q/K/V rows, appended, attention
    halves += case["hidden"] * hq * d + rows * case["hidden"]       # o_proj weight and output
    flops = 4 * d * hq * pairs + 2 * rows * case["hidden"] * hq * d
    return {"bytes": 2 * halves * n, "flops": flops * n}


def tolerance(case):
    """f16 inputs and outputs with f32 sums, and f16 probabilities in prefill. Measured against
    exact() over the listed and ten drawn cases: relative error at most 7.5e-4, largest single
    difference 0.02 of the rms (a probability's rounding where the values cancel)."""
    return {"rel": 3e-3, "max": 0.08}


def _exact_norm_rope(x, weight, offset):
    """x [T, H, D] float64: RMSNorm by weight, then the half-split rotation."""
    x = x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS) * weight
    half = x.shape[-1] // 2
    freq = THETA ** (-torch.arange(half, device=x.device, dtype=torch.float64) / half)
    angle = (offset + torch.arange(x.shape[0], device=x.device, dtype=torch.float64))[:, None, None] * freq
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * angle.cos() - b * angle.sin(), a * angle.sin() + b * angle.cos()], -1)


def _exact_attention(q, key, value, offset):
    """q [T, Hq, D], key / value [Hkv, L, D] float64, causal from `offset`: [T, Hq, D]."""
    t, hq, d = q.shape
    hkv, length = key.shape[:2]
    out = torch.empty_like(q)
    step = max(1, int(1e8 / (length * (hq // hkv))))  # query rows a block
    at = torch.arange(length, device=q.device)
    for h in range(hkv):
        for t0 in range(0, t, step):
            rows = q[t0:t0 + step, h * (hq // hkv):(h + 1) * (hq // hkv)]
            s = (rows.reshape(-1, d) @ key[h].T) * d ** -0.5
            s = s.view(rows.shape[0], -1, length)
            last = offset + t0 + torch.arange(rows.shape[0], device=q.device)
            s = s.masked_fill(at[None, None, :] > last[:, None, None], float("-inf")).softmax(-1)
            out[t0:t0 + step, h * (hq // hkv):(h + 1) * (hq // hkv)] = \
                (s.view(-1, length) @ value[h]).view(rows.shape)
    return out


def exact(case, seed):
    x = _inputs(case, seed)
    n, t, hq, hkv, d = (case[k] for k in ("layers", "tokens", "q_heads", "kv_heads", "head_dim"))
    attn, proj = [], []
    keys, values = x["key"].double(), x["value"].double()
    o = case["offset"]
    for i in range(n):
        if case["op"] == "batch":
            a = torch.cat([_exact_attention(x["q"][i, b:b + 1].double(), keys[i, b, :, :m], values[i, b, :, :m], m - 1)
                           for b, m in enumerate(x["lengths"].tolist())])
        else:
            qkv = x["qkv"][i].double()
            q = _exact_norm_rope(qkv[:, :hq], x["q_weight"][i].double(), o)
            keys[i, :, o:o + t] = _exact_norm_rope(qkv[:, hq:hq + hkv], x["k_weight"][i].double(), o).transpose(0, 1)
            values[i, :, o:o + t] = qkv[:, hq + hkv:].transpose(0, 1)
            a = _exact_attention(q, keys[i, :, :o + t], values[i, :, :o + t], o)
        attn.append(a)
        proj.append(a.reshape(a.shape[0], hq * d) @ x["proj_weight"][i].double().T)
    out = {"attention": torch.stack(attn), "proj": torch.stack(proj)}
    if case["op"] != "batch":
        out.update(key=keys, value=values, new_key=keys[:, :, o:o + t], new_value=values[:, :, o:o + t])
    return out
