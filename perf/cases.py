"""Performance cases of the k-quant path: what a user's program has the library do.

Listed cases are decode and prefill work at the sizes this repository is used
at (the Qwen3-8B geometry, and the 5120-wide projections of the reference's own
GEMV bench); draw() spreads the same kinds over their whole ranges. Each kind
goes through the public entry points:

  proj    projections sharing one input (q/k/v, o): execute_warp,
          execute_warp_batch, execute_group with the fused RMSNorm
  mlp     a layer's FFN: RMSNorm-fused gate/up SwiGLU pair, then down
  attn    a layer's decode attention over filled caches
  chunk   a layer's causal attention for a prompt chunk
  gemm    the prefill matmul, f32 or bf16 activations, RMSNorm fused or not
  decode  a whole decoder step (embedding to logits)
  prompt  a whole prompt into the cache, then the step that samples it

Weights are k-quant blocks with the magnitudes of trained ones (zero mean, a
row's variance 1/K); proj, mlp and the decode kinds walk several distinct
layers in a pass, as a model does, so weights come from HBM.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import engine_amd as E

DEV = "cuda:0"
EPS = 1e-6
ROPE_BASE = 1.0e6
HEAD = 128
TYPES = {"q4_k": 12, "q5_k": 13, "q6_k": 14}
BLOCK = {12: 144, 13: 176, 14: 210}
# Standard deviation of (quant - mean) * scale over uniform quants and scales.
SPREAD = {12: 4.61 * 36.5, 13: 9.23 * 36.5, 14: 18.47 * 18.5}
MEAN_Q = {12: 7.5, 13: 15.5}


def listed():
    return [
        # One token's o projections: the smallest calls, all launch and latency.
        dict(name="proj_o_1", kind="proj", type="q4_k", k=4096, rows="4096", members=1, norm=False, layers=2),
        # The 5120-wide FFN projection of the reference's GEMV bench, one token.
        dict(name="proj_5120_1", kind="proj", type="q5_k", k=5120, rows="17408", members=1, norm=False, layers=4),
        # One token through the FFNs of a few layers (interactive decode).
        dict(name="mlp_1", kind="mlp", type="q4_k", down="q5_k", hidden=4096, ffn=12288, members=1, layers=6),
        # Eight sequences, the reference's batch cap.
        dict(name="mlp_8", kind="mlp", type="q4_k", down="q5_k", hidden=4096, ffn=12288, members=8, layers=6),
        # Serving batches past it: ordinary, and large and ragged.
        dict(name="mlp_16", kind="mlp", type="q4_k", down="q5_k", hidden=4096, ffn=12288, members=16, layers=6),
        dict(name="mlp_61", kind="mlp", type="q4_k", down="q5_k", hidden=4096, ffn=12288, members=61, layers=6),
        # Decode attention of eight sequences of different lengths.
        dict(name="attn_8", kind="attn", q_heads=32, kv_heads=8, members=8, context=3000, layers=4),
        # Prompt attention over a whole chunk.
        dict(name="chunk_2047", kind="chunk", q_heads=32, kv_heads=8, tokens=2047, position=0),
        # Prefill matmuls: a short prompt in bf16, a long ragged one in f32.
        dict(name="gemm_512", kind="gemm", type="q4_k", k=4096, n=12288, members=512, dtype="bf16", norm=False),
        dict(name="gemm_1999", kind="gemm", type="q6_k", k=12288, n=4096, members=1999, dtype="f32", norm=False),
        # A whole decode step at 2,048 cached tokens: embedding, 36 layers, head.
        dict(name="decode_1", kind="decode", hidden=4096, ffn=12288, q_heads=32, kv_heads=8, vocab=151936, layers=36,
             members=1, context=2047),
        # A whole prompt through a stack of layers, then the step that samples it.
        dict(name="prompt_2047", kind="prompt", hidden=4096, ffn=12288, q_heads=32, kv_heads=8, vocab=32000, layers=4,
             tokens=2047),
    ]


def _log_int(rng, low, high, step=1):
    v = math.exp(rng.uniform(math.log(low), math.log(high)))
    return max(low, min(high, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(("proj", "proj", "mlp", "mlp", "attn", "chunk", "gemm", "gemm", "decode", "prompt"))
    t = rng.choice(tuple(TYPES))
    if kind == "proj":
        rows = [_log_int(rng, 256, 17408, rng.choice((1, 16, 256))) for _ in range(rng.choice((1, 1, 2, 3)))]
        k = _log_int(rng, 1024, 17408, 256)
        return dict(kind="proj", type=t, k=k, rows=",".join(str(n) for n in rows), members=_log_int(rng, 1, 64),
                    norm=k <= 16384 and rng.random() < 0.5, layers=rng.randint(1, 4))
    if kind == "mlp":
        return dict(kind="mlp", type=rng.choice(("q4_k", "q4_k", "q5_k")), down=t, hidden=_log_int(rng, 1024, 4096, 256),
                    ffn=_log_int(rng, 2816, 12288, 256), members=_log_int(rng, 1, 61), layers=rng.randint(2, 6))
    if kind == "attn":
        return dict(kind="attn", q_heads=rng.choice((8, 16, 32, 64)), kv_heads=8, members=_log_int(rng, 1, 16),
                    context=_log_int(rng, 16, 4096), layers=rng.randint(1, 4))
    if kind == "chunk":
        return dict(kind="chunk", q_heads=rng.choice((8, 16, 32)), kv_heads=8, tokens=_log_int(rng, 16, 2047),
                    position=rng.choice((0, 0, rng.randint(1, 2048))))
    if kind == "gemm":
        return dict(kind="gemm", type=t, k=_log_int(rng, 1024, 12288, 256), n=_log_int(rng, 512, 12288, rng.choice((1, 16, 256))),
                    members=_log_int(rng, 65, 1999), dtype=rng.choice(("f32", "bf16")), norm=rng.random() < 0.4)
    geo = rng.choice(((4096, 12288, 32), (2560, 9728, 32), (2048, 6144, 16), (1024, 3072, 16)))
    if kind == "decode":
        return dict(kind="decode", hidden=geo[0], ffn=geo[1], q_heads=geo[2], kv_heads=8, vocab=_log_int(rng, 8000, 100000),
                    layers=rng.randint(2, 8), members=_log_int(rng, 1, 16), context=_log_int(rng, 16, 4000))
    return dict(kind="prompt", hidden=geo[0], ffn=geo[1], q_heads=geo[2], kv_heads=8, vocab=_log_int(rng, 8000, 32000),
                layers=rng.randint(2, 4), tokens=_log_int(rng, 64, 2047))


# ------------------------------------------------------------------ inputs

def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(1000003 * seed + 17)
    return g


def _encode(t, k, n, g):
    """Random k-quant blocks of an [n][k] weight with zero mean and variance 1/k."""
    nb = n * (k // 256)
    blocks = torch.randint(0, 256, (nb, BLOCK[t]), dtype=torch.uint8, device=DEV, generator=g)
    d = torch.empty(nb, device=DEV).uniform_(0.5, 1.5, generator=g).mul_(1.0 / (SPREAD[t] * math.sqrt(k))).half()

    def halfs(v):
        return v.view(torch.uint8).view(nb, 2)

    if t == 14:
        scales = torch.randint(-32, 32, (nb, 16), dtype=torch.int8, device=DEV, generator=g)
        blocks[:, 192:208] = scales.view(torch.uint8)
        blocks[:, 208:210] = halfs(d)
    else:
        blocks[:, 0:2] = halfs(d)
        blocks[:, 2:4] = halfs((d.float() * MEAN_Q[t]).half())
    return blocks.view(-1)


def _gamma(n, g):
    return torch.randn(n, device=DEV, generator=g).mul_(0.02).add_(1.0)


class _DeviceArray:
    """An f16 device range of the library's, for torch.as_tensor."""

    def __init__(self, ptr, shape, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": "<f2", "version": 2}


def _cache_views(cache, cfg, layer):
    """One layer's keys and values, [kv_heads][capacity][128] f16, in place."""
    shape = (cfg.kv_heads, cache.capacity(), HEAD)
    return [torch.as_tensor(_DeviceArray(p, shape, cache), device=DEV) for p in cache.layer(layer)]


class _State:
    pass


def _weights(s, specs, g):
    """Encodes and stores `specs` = [(name, type, k, n)] into s.w, s.enc."""
    if not hasattr(s, "store"):
        s.ctx = E.AmdContext(0)
        s.store = E.AmdWeightStore(s.ctx)
        s.w, s.enc = {}, {}
    for name, t, k, n in specs:
        enc = _encode(t, k, n, g)
        s.enc[name] = (t, k, n, enc)
        s.store.materialize_quantized(name, [k, n], t, enc)
        s.w[name] = s.store.quantized_tensor(name)


def _contexts(case):
    """Cached tokens of each member: the longest has `context`, the others 40-100% of it."""
    rng = np.random.default_rng(case["context"])
    m = case["members"]
    return [case["context"]] + [int(case["context"] * v) for v in rng.uniform(0.4, 1.0, m - 1)]


def _model_specs(case):
    h, f, q, kv = case["hidden"], case["ffn"], case["q_heads"] * HEAD, case["kv_heads"] * HEAD
    specs = [("token_embd", 12, h, case["vocab"]), ("output", 14, h, case["vocab"])]
    for i in range(case["layers"]):
        specs += [(f"{i}.{nm}", t, k, n) for nm, t, k, n in (
            ("attn_q", 12, h, q), ("attn_k", 12, h, kv), ("attn_v", 12, h, kv), ("attn_output", 12, q, h),
            ("ffn_gate", 12, h, f), ("ffn_up", 12, h, f), ("ffn_down", 13, f, h))]
    return specs


def _prepare_model(s, case, seed, g, members):
    _weights(s, _model_specs(case), g)
    h = case["hidden"]
    s.norms = {"output_norm": _gamma(h, g)}
    layers = []
    for i in range(case["layers"]):
        for nm, size in (("attn_norm", h), ("ffn_norm", h), ("attn_q_norm", HEAD), ("attn_k_norm", HEAD)):
            s.norms[f"{i}.{nm}"] = _gamma(size, g)
        layers.append({key[len(f"{i}."):]: v for src in (s.w, s.norms) for key, v in src.items() if key.startswith(f"{i}.")})
    s.cfg = E.AmdQwen3Config(layers=case["layers"], hidden=h, q_heads=case["q_heads"], kv_heads=case["kv_heads"],
                             head_dim=HEAD, ffn=case["ffn"], vocab=case["vocab"], rope_base=ROPE_BASE, epsilon=EPS)
    s.dec = E.AmdQwen3Decode(s.ctx, s.cfg, s.w["token_embd"], s.w["output"], s.norms["output_norm"], layers, members)
    s.rng = np.random.default_rng(seed)


def _filled_cache(s, tokens, capacity, g):
    cache = E.AmdKvCache(s.ctx, s.cfg, capacity)
    for i in range(s.cfg.layers):
        for v in _cache_views(cache, s.cfg, i):
            v.zero_()
            v[:, :tokens].copy_(torch.randn((s.cfg.kv_heads, tokens, HEAD), device=DEV, generator=g).half())
    return cache


def prepare(case, seed):
    s = _State()
    s.case = case
    g = _generator(seed)
    kind = case["kind"]
    if kind == "proj":
        t, k, m = TYPES[case["type"]], case["k"], case["members"]
        rows = [int(n) for n in case["rows"].split(",")]
        _weights(s, [(f"{i}.{j}", t, k, n) for i in range(case["layers"]) for j, n in enumerate(rows)], g)
        s.kern = E.QwenGemvKernel.from_value_type(s.ctx, t)
        s.x = [torch.randn(m * k, device=DEV, generator=g) for _ in range(case["layers"])]
        s.gamma = _gamma(k, g) if case["norm"] else None
        s.y = [[torch.zeros(m * n, device=DEV) for n in rows] for _ in range(case["layers"])]
        s.groups = [[s.w[f"{i}.{j}"] for j in range(len(rows))] for i in range(case["layers"])]
    elif kind == "mlp":
        h, f, m = case["hidden"], case["ffn"], case["members"]
        gu, dn = TYPES[case["type"]], TYPES[case["down"]]
        _weights(s, [(f"{i}.{nm}", t, k, n) for i in range(case["layers"])
                     for nm, t, k, n in (("gate", gu, h, f), ("up", gu, h, f), ("down", dn, f, h))], g)
        s.kern, s.down = (E.QwenGemvKernel.from_value_type(s.ctx, t) for t in (gu, dn))
        s.x = [torch.randn(m * h, device=DEV, generator=g) for _ in range(case["layers"])]
        s.gamma = [_gamma(h, g) for _ in range(case["layers"])]
        s.act = [torch.zeros(m * f, device=DEV) for _ in range(case["layers"])]
        s.y = [torch.zeros(m * h, device=DEV) for _ in range(case["layers"])]
    elif kind in ("attn", "chunk"):
        s.ctx = E.AmdContext(0)
        s.cfg = E.AmdQwen3Config(layers=case.get("layers", 1), hidden=4096, q_heads=case["q_heads"], kv_heads=case["kv_heads"],
                                 head_dim=HEAD, ffn=12288, vocab=1024, rope_base=ROPE_BASE, epsilon=EPS)
        q, kv = case["q_heads"] * HEAD, case["kv_heads"] * HEAD
        if kind == "attn":
            s.contexts = _contexts(case)
            s.caches = [_filled_cache(s, c, c + 8, g) for c in s.contexts]
            s.positions = torch.tensor(s.contexts, dtype=torch.int32, device=DEV)
            m = case["members"]
        else:
            s.caches = [_filled_cache(s, case["position"], case["position"] + case["tokens"], g)]
            m = case["tokens"]
        s.views = [[_cache_views(c, s.cfg, i) for i in range(s.cfg.layers)] for c in s.caches]
        s.io = [[torch.randn(m * n, device=DEV, generator=g) for n in (q, kv, kv)] for _ in range(s.cfg.layers)]
        s.norms = [(_gamma(HEAD, g), _gamma(HEAD, g)) for _ in range(s.cfg.layers)]
        s.y = [torch.zeros(m * q, device=DEV) for _ in range(s.cfg.layers)]
    elif kind == "gemm":
        t, k, n, m = TYPES[case["type"]], case["k"], case["n"], case["members"]
        _weights(s, [("w", t, k, n)], g)
        s.kern = E.QwenGemvKernel.from_value_type(s.ctx, t)
        s.ctx.reserve_prefill(m, k, n)
        s.x = torch.randn(m, k, device=DEV, generator=g)
        s.x = s.x.bfloat16() if case["dtype"] == "bf16" else s.x
        s.gamma = _gamma(k, g) if case["norm"] else None
        s.y = torch.zeros(m * n, device=DEV)
    elif kind == "decode":
        _prepare_model(s, case, seed, g, case["members"])
        s.contexts = _contexts(case)
        s.caches = [_filled_cache(s, c, c + 8, g) for c in s.contexts]
        s.tokens = [int(v) for v in s.rng.integers(0, case["vocab"], case["members"])]
    else:
        _prepare_model(s, case, seed, g, 1)
        s.tokens = [int(v) for v in s.rng.integers(0, case["vocab"], case["tokens"] + 1)]
        s.dec.reserve_prompt(0)
        s.cache = _filled_cache(s, 0, case["tokens"] + 8, g)
        s.views = [_cache_views(s.cache, s.cfg, i) for i in range(s.cfg.layers)]
    return s


# -------------------------------------------------------------------- a pass

def run(s):
    case = s.case
    kind = case["kind"]
    if kind == "proj":
        m = case["members"]
        for ws, x, ys in zip(s.groups, s.x, s.y):
            if len(ws) > 1:
                s.kern.execute_group(ws, x, ys, m, gamma=s.gamma, epsilon=EPS)
            elif s.gamma is not None:
                s.kern.execute_rms_norm(ws[0], x, s.gamma, EPS, ys[0], m)
            elif m == 1:
                s.kern.execute_warp(ws[0], x, ys[0])
            else:
                s.kern.execute_warp_batch(ws[0], x, ys[0], m)
        return s.y
    if kind == "mlp":
        m = case["members"]
        for i in range(case["layers"]):
            s.kern.execute_gate_up_swiglu(s.w[f"{i}.gate"], s.w[f"{i}.up"], s.x[i], s.act[i], m, gamma=s.gamma[i], epsilon=EPS)
            s.down.execute_warp_batch(s.w[f"{i}.down"], s.act[i], s.y[i], m)
        return s.y
    if kind == "attn":
        for i, ((q, k, v), (qn, kn)) in enumerate(zip(s.io, s.norms)):
            E.attention_decode(s.ctx, s.cfg, s.caches, i, q, k, v, qn, kn, s.positions, s.y[i])
        return {"y": s.y, "new": [[t[:, c] for pair in views for t in pair] for views, c in zip(s.views[:2], s.contexts)]}
    if kind == "chunk":
        (q, k, v), (qn, kn) = s.io[0], s.norms[0]
        E.attention_prefill(s.ctx, s.cfg, s.caches[0], 0, q, k, v, qn, kn, case["tokens"], case["position"], s.y[0])
        return {"y": s.y[0], "cache": s.views[0][0]}
    if kind == "gemm":
        s.kern.gemm_prefill(s.w["w"], s.x, s.y, case["members"], gamma=s.gamma, epsilon=EPS)
        return s.y
    if kind == "decode":
        s.dec.decode_step_batch(s.caches, s.tokens, s.contexts)
        return [s.dec.copy_logits(i) for i in range(case["members"])]
    s.dec.prefill_prompt(s.cache, s.tokens[:-1], 0)
    s.dec.decode_step(s.cache, s.tokens[-1], case["tokens"])
    return {"logits": s.dec.copy_logits(0), "cache": s.views}


# ------------------------------------------------------ what a pass must move

def _wbytes(t, k, n):
    return n * (k // 256) * BLOCK[t]


def _attn_work(case, pairs, rows, layers):
    """Attention over `pairs` (token, cached token) pairs and `rows` new tokens."""
    return 4.0 * HEAD * case["q_heads"] * pairs * layers, layers * rows * HEAD * (8.0 * case["q_heads"] + 12.0 * case["kv_heads"])


def work(case):
    kind = case["kind"]
    if kind in ("proj", "mlp"):
        m, n_layers = case["members"], case["layers"]
        if kind == "proj":
            t, k, n = TYPES[case["type"]], case["k"], sum(int(v) for v in case["rows"].split(","))
            b, fl = _wbytes(t, k, n) + 4 * m * (k + n), 2 * m * k * n
        else:
            h, f = case["hidden"], case["ffn"]
            b = _wbytes(TYPES[case["type"]], h, 2 * f) + _wbytes(TYPES[case["down"]], f, h) + 8 * m * h
            fl = 6 * m * h * f
        return {"bytes": float(b * n_layers), "flops": float(fl * n_layers)}
    if kind == "attn":
        cached = sum(_contexts(case))
        fl, b = _attn_work(case, cached + case["members"], case["members"], case["layers"])
        return {"bytes": b + 4.0 * HEAD * case["kv_heads"] * cached * case["layers"], "flops": fl}
    if kind == "chunk":
        n, p = case["tokens"], case["position"]
        fl, b = _attn_work(case, n * p + n * (n + 1) / 2, n, 1)
        return {"bytes": b + 4.0 * HEAD * case["kv_heads"] * p, "flops": fl}
    if kind == "gemm":
        m, k, n = case["members"], case["k"], case["n"]
        xb = 2 if case["dtype"] == "bf16" else 4
        return {"bytes": float(_wbytes(TYPES[case["type"]], k, n) + m * k * xb + 4 * m * n), "flops": 2.0 * m * k * n}
    specs = _model_specs(case)
    layer_bytes = sum(_wbytes(t, k, n) for _, t, k, n in specs[2:])
    layer_mults = sum(k * n for _, _, k, n in specs[2:])
    head_bytes, head_mults = _wbytes(*specs[1][1:]), case["hidden"] * case["vocab"]
    if kind == "decode":
        cached, m = sum(_contexts(case)), case["members"]
        fl, _ = _attn_work(case, cached + m, m, case["layers"])
        return {"bytes": layer_bytes + head_bytes + 4.0 * HEAD * case["kv_heads"] * cached * case["layers"] + 4.0 * m * case["vocab"],
                "flops": fl + 2.0 * m * (layer_mults + head_mults)}
    n = case["tokens"]
    fl, b = _attn_work(case, n * (n + 1) / 2, n, case["layers"] - 1)
    # the prompt's last layer only needs its K and V; the sampling step needs all
    last = 2 * case["hidden"] * case["kv_heads"] * HEAD
    prompt_mults = layer_mults * (case["layers"] - 1) // case["layers"] + last
    return {"bytes": 2.0 * layer_bytes + head_bytes + b + 4.0 * HEAD * case["kv_heads"] * n * case["layers"],
            "flops": fl + 2.0 * (n * prompt_mults + layer_mults + head_mults)}


def tolerance(case):
    """Four times what another order of the sums shows, by the arithmetic of the
    path: f32 sums, f32 attention that appends f16 keys (a rounding flipped here
    and there), f16 matmul operands."""
    kind = case["kind"]
    if kind == "proj":
        return {"rel": 1e-5, "max": 1e-4}
    if kind == "mlp":
        return {"rel": 2e-5, "max": 2e-4}
    if kind == "attn":
        return {"rel": 4e-4, "max": 4e-3}
    if kind == "chunk":
        return {"rel": 2e-4, "max": 5e-3}
    if kind == "gemm":
        return {"rel": 1.2e-3, "max": 2e-2}
    if kind == "decode":
        return {"rel": 2e-4, "max": 4e-3}
    return {"rel": 8e-3, "max": 8e-2}


# ------------------------------------------------------------ 64-bit results

def _six_bit_scales(raw):
    """The eight (scale, min) pairs of the 12 packed bytes of Q4_K / Q5_K blocks."""
    low, mid, high = raw[:, 0:4], raw[:, 4:8], raw[:, 8:12]
    sc = torch.cat((low & 63, (high & 15) | ((low >> 6) << 4)), 1)
    mn = torch.cat((mid & 63, (high >> 4) | ((mid >> 6) << 4)), 1)
    return sc.double(), mn.double()


def _decode(spec, first=0, count=None):
    """Rows first .. first + count - 1 of an encoded weight as an f64 matrix."""
    t, k, n, enc = spec
    count = n - first if count is None else count
    b = enc.view(n, -1)[first:first + count].reshape(-1, BLOCK[t])

    def half(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).double()

    if t == 14:
        ql, qh = b[:, 0:128].view(-1, 2, 64), b[:, 128:192].view(-1, 2, 32)
        lo = torch.stack((ql & 15, ql >> 4), 2).view(-1, 2, 4, 32)
        hi = torch.stack([(qh >> (2 * j)) & 3 for j in range(4)], 2)
        q = (lo | (hi << 4)).double() - 32
        scales = b[:, 192:208].contiguous().view(torch.int8).double()
        w = q.view(-1, 16, 16) * scales[:, :, None] * half(208)[:, :, None]
    else:
        sc, mn = _six_bit_scales(b[:, 4:16])
        qs = b[:, 16:144] if t == 12 else b[:, 48:176]
        qs = qs.reshape(-1, 4, 1, 32)
        q = torch.cat((qs & 15, qs >> 4), 2).view(-1, 8, 32)
        if t == 13:
            qh = b[:, 16:48]
            q = q | (torch.stack([(qh >> j) & 1 for j in range(8)], 1) << 4)
        w = q.double() * (sc * half(0))[:, :, None] - (mn * half(2))[:, :, None]
    return w.reshape(count, k)


def _matmul(x, spec):
    """x W^T in f64, a slab of rows at a time."""
    n, k = spec[2], spec[1]
    step = max(1, (1 << 27) // k)
    return torch.cat([x @ _decode(spec, i, min(step, n - i)).t() for i in range(0, n, step)], 1)


def _rms(x, gamma):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * gamma.double()


def _heads(x, n, gamma, positions):
    """[tokens][n*128] normalised per head and rotated (split halves), [n][tokens][128]."""
    x = _rms(x.view(len(positions), n, HEAD), gamma)
    freq = ROPE_BASE ** (-2.0 * torch.arange(HEAD // 2, dtype=torch.float64, device=DEV) / HEAD)
    ang = positions.double()[:, None, None] * freq
    a, b = x[..., :HEAD // 2], x[..., HEAD // 2:]
    return torch.cat((a * ang.cos() - b * ang.sin(), a * ang.sin() + b * ang.cos()), -1).transpose(0, 1).contiguous()


def _attention(q, keys, values, position):
    """q [q_heads][tokens][128] at position.., keys / values [kv_heads][context][128]: causal, [tokens][q_heads*128]."""
    n, per = q.shape[1], q.shape[0] // keys.shape[0]
    seen = torch.arange(keys.shape[1], device=DEV)[None, :] <= position + torch.arange(n, device=DEV)[:, None]
    out = []
    for i in range(q.shape[0]):
        sc = (q[i] @ keys[i // per].t().contiguous()) / math.sqrt(HEAD)
        out.append(torch.softmax(sc.masked_fill(~seen, -math.inf), -1) @ values[i // per])
    return torch.stack(out, 1).reshape(n, -1)


def _append(keys, values, k, v, gamma, position):
    """The cache's f16 keys and values with the new tokens' in place, as f64."""
    n, kvh = k.shape[0], keys.shape[0]
    keys, values = keys.double().clone(), values.double().clone()
    keys[:, position:position + n] = _heads(k, kvh, gamma, position + torch.arange(n, device=DEV)).half().double()
    values[:, position:position + n] = v.view(n, kvh, HEAD).transpose(0, 1).half().double()
    return keys, values


def _model_exact(s, tokens, position, keys, values):
    """One sequence's tokens from `position` through the model: (logits of the last, keys, values)."""
    case = s.case
    n, at = len(tokens), position + torch.arange(len(tokens), device=DEV)
    x = torch.cat([_decode(s.enc["token_embd"], tok, 1) for tok in tokens])
    for i in range(case["layers"]):
        p = f"{i}."
        h = _rms(x, s.norms[p + "attn_norm"])
        keys[i], values[i] = _append(keys[i], values[i], _matmul(h, s.enc[p + "attn_k"]), _matmul(h, s.enc[p + "attn_v"]),
                                     s.norms[p + "attn_k_norm"], position)
        q = _heads(_matmul(h, s.enc[p + "attn_q"]), case["q_heads"], s.norms[p + "attn_q_norm"], at)
        a = _attention(q, keys[i][:, :position + n], values[i][:, :position + n], position)
        x = x + _matmul(a, s.enc[p + "attn_output"])
        h = _rms(x, s.norms[p + "ffn_norm"])
        x = x + _matmul(torch.nn.functional.silu(_matmul(h, s.enc[p + "ffn_gate"])) * _matmul(h, s.enc[p + "ffn_up"]),
                        s.enc[p + "ffn_down"])
    return _matmul(_rms(x[-1:], s.norms["output_norm"]), s.enc["output"]).view(-1), keys, values


def exact(case, seed):
    kind = case["kind"]
    s = prepare(case, seed)
    if kind == "proj":
        m, k = case["members"], case["k"]
        out = []
        for i, x in enumerate(s.x):
            x = x.double().view(m, k)
            x = x if s.gamma is None else _rms(x, s.gamma)
            out.append([_matmul(x, s.enc[f"{i}.{j}"]).view(-1) for j in range(len(s.groups[i]))])
        return out
    if kind == "mlp":
        out = []
        for i, x in enumerate(s.x):
            h = _rms(x.double().view(case["members"], -1), s.gamma[i])
            act = torch.nn.functional.silu(_matmul(h, s.enc[f"{i}.gate"])) * _matmul(h, s.enc[f"{i}.up"])
            out.append(_matmul(act, s.enc[f"{i}.down"]).view(-1))
        return out
    if kind in ("attn", "chunk"):
        qh, kvh = case["q_heads"], case["kv_heads"]
        ys, new = [], []
        for i, ((q, k, v), (qn, kn)) in enumerate(zip(s.io, s.norms)):
            q, k, v = (t.double().view(-1, n * HEAD) for t, n in ((q, qh), (k, kvh), (v, kvh)))
            rows = []
            for j in range(len(s.caches)):
                at, one = (s.contexts[j], slice(j, j + 1)) if kind == "attn" else (case["position"], slice(None))
                n = len(q[one])
                keys, values = _append(*s.views[j][i], k[one], v[one], kn, at)
                rows.append(_attention(_heads(q[one], qh, qn, at + torch.arange(n, device=DEV)), keys[:, :at + n], values[:, :at + n], at))
                if kind == "chunk":
                    return {"y": rows[0].reshape(-1), "cache": [keys, values]}
                if j < 2:
                    new.append((j, keys[:, at], values[:, at]))
            ys.append(torch.cat(rows).reshape(-1))
        return {"y": ys, "new": [[t for j, a, b in new if j == m for t in (a, b)] for m in range(min(2, case["members"]))]}
    if kind == "gemm":
        x = s.x.double()
        return _matmul(x if s.gamma is None else _rms(x, s.gamma), s.enc["w"]).view(-1)
    if kind == "decode":
        out = []
        for i, (cache, c) in enumerate(zip(s.caches, s.contexts)):
            keys, values = map(list, zip(*(_cache_views(cache, s.cfg, j) for j in range(case["layers"]))))
            out.append(_model_exact(s, [s.tokens[i]], c, keys, values)[0])
        return out
    keys, values = map(list, zip(*s.views))
    _, keys, values = _model_exact(s, s.tokens[:-1], 0, keys, values)
    logits, keys, values = _model_exact(s, s.tokens[-1:], case["tokens"], keys, values)
    return {"logits": logits, "cache": [[a, b] for a, b in zip(keys, values)]}
