"""Prompt prefill on the prefill matmul (ribn_amd_qwen3_prefill_prompt) against
the oracle's serial prefill, through the C ABI.

The path: every projection as a matmul over the chunk's tokens (f16
activations after a per-token power-of-two scale, weights dequantised into
f16, f16 MFMA, f32 accumulation; the ribn_amd_gemm_prefill kernels), then
causal chunk attention on the matrix cores (q and the probabilities as two
f16 pieces each, f16 K/V from the cache, f32 sums). It replaces the
reference's run_prefill_chunk (crates/nvidia/src/decode.rs:2149-2267), whose
projections run through gemv_batch a few tokens at a time.

The attention alone (ribn_amd_attention_prefill) is checked against the
oracle's attention stepped token by token within ATTN_TOL, the appended V
bit for bit and K within 1e-3. The whole prompt path is checked against
oracle/qwen3_oracle.py stepping the same prompt one token at a time
(OracleQwen3.step(..., head=False), the reference's prefill_step):
  * every K/V the prompt wrote to the cache, as f16 values, per token within
    KV_TOL of the layer's largest value (zero-mean weights), or within 4
    times what f16 operands alone do to that token (weights of one sign);
  * after the prompt, one decode step on the prompt's last token: logits and
    final hidden state within LOGIT_TOL normwise, the greedy token equal
    wherever the oracle's top-2 margin exceeds four times the error.
The prefill matmul rounds its operands to f16 (2^-11 relative), so these
bars sit above the f32 decode path's 1e-3 (tests/test_gpu_decode.py).
Shapes: GQA groups 1, 2, 4 and 8 (all four kernel instantiations), chunks
of 16..128 tokens with partial last chunks and a one-token chunk, a prompt
continuing a cache at a non-zero position, the Qwen3-8B layer geometry, and
the entry point's error cases.
"""
import ctypes

import numpy as np
import pytest

from engine_amd import synth
from oracle import kquant_oracle as O
from oracle.qwen3_oracle import OracleQwen3

from .decode_helpers import small_weights
from .gpu_helpers import max_rel_err, to_dev, to_host

pytestmark = pytest.mark.gpu

KV_TOL = 4e-3
LOGIT_TOL = 4e-3
ATTN_TOL = 5e-4

TINY = dict(layers=2, hidden=1024, q_heads=8, kv_heads=2, head_dim=128, ffn=4608, vocab=2048,
            rope_base=1.0e6, epsilon=1.0e-6)
WIDE = dict(layers=1, hidden=4096, q_heads=32, kv_heads=8, head_dim=128, ffn=12288, vocab=4096,
            rope_base=1.0e6, epsilon=1.0e-6)


def case(**kw):
    print("CASE", " ".join(f"{k}={v}" for k, v in kw.items()), flush=True)


class ThreadedOracle(OracleQwen3):
    """The oracle step with its GEMVs split by rows over 16 host threads
    (each row's sequential f32 sum unchanged)."""

    def _gemv(self, name, x):
        t, k, n, enc = self.w[name]
        return O.quant_gemv(t, enc, k, n, x, threads=16)


def f16_activations(x):
    """x as the prefill matmul's activation stage rounds it: scaled by the
    power of two that maps max |x| just below 2^15, rounded to f16 (RNE),
    scaled back (engine_amd/csrc/qgemm.hip act_f16_kernel)."""
    x = np.asarray(x, np.float32)
    amax = float(np.abs(x).max())
    if amax == 0.0:
        return x
    s = np.float32(2.0 ** (15 - int(np.frexp(amax)[1])))
    return ((x * s).astype(np.float16).astype(np.float32) / s).astype(np.float32)


class F16OperandOracle(OracleQwen3):
    """The oracle with the prefill matmul's operand precision: every GEMV input
    rounded as its activation stage rounds it (f16_activations) and every
    dequantised weight rounded to f16 (the kernel dequantises into f16 MFMA
    operands), products summed in f32 by a dense matmul; attention and
    everything else as the oracle. How far f16 operands alone move each cache
    row of a given model."""

    def __init__(self, cfg, weights, capacity):
        super().__init__(cfg, weights, capacity)
        self._dense = {}

    def _gemv(self, name, x):
        if name not in self._dense:
            t, k, n, enc = self.w[name]
            self._dense[name] = O.dequantize_tensor(t, enc).reshape(n, k).astype(np.float16).astype(np.float32)
        return (self._dense[name] @ f16_activations(x)).astype(np.float32)


@pytest.fixture(scope="module")
def env():
    import torch
    import engine_amd as E
    assert torch.cuda.is_available(), "GPU tests need a ROCm device"
    ctx = E.AmdContext(0)
    return {"E": E, "ctx": ctx, "store": E.AmdWeightStore(ctx), "n": [0]}


def build(env, cfg, w):
    E, store = env["E"], env["store"]
    handles = {}
    for name, val in w.items():
        if isinstance(val, tuple):
            t, k, n, enc = val
            env["n"][0] += 1
            key = f"p{env['n'][0]}"
            store.materialize_quantized(key, [k, n], t, enc)
            handles[name] = store.quantized_tensor(key)
        else:
            handles[name] = to_dev(val)
    layers = [{f: handles[f"blk.{l}.{f}"] for f in
               ("attn_q", "attn_k", "attn_v", "attn_output", "ffn_gate", "ffn_up", "ffn_down", "attn_norm",
                "attn_q_norm", "attn_k_norm", "ffn_norm")} for l in range(cfg["layers"])]
    return E.AmdQwen3Decode(env["ctx"], E.AmdQwen3Config(**cfg), handles["token_embd"], handles["output"],
                            handles["output_norm"], layers, 1)


def cache_arrays(env, cache, cfg):
    """[layer][K, V] as [kv_heads][capacity][128] f16 bits."""
    lib, ctx = env["ctx"]._lib, env["ctx"]
    out = []
    for layer in range(cfg["layers"]):
        pair = []
        for ptr in cache.layer(layer):
            full = np.zeros((cfg["kv_heads"], cache.capacity(), 128), np.uint16)
            assert lib.ribn_amd_memcpy_dtoh(ctx.handle, full.ctypes.data_as(ctypes.c_void_p), ctypes.c_void_p(ptr),
                                            full.nbytes) == 0
            pair.append(full)
        out.append(pair)
    return out


def f16_err(a_bits, b_bits):
    a = a_bits.view(np.float16).astype(np.float64)
    b = b_bits.view(np.float16).astype(np.float64)
    return float(np.abs(a - b).max() / np.abs(b).max())


def per_token_err(dev, host, count):
    """Per-token normwise error of [kv_heads][capacity][128] device bits
    against the oracle's [capacity][kv_heads][128] bits over positions < count,
    each token's largest |difference| over the layer's largest |value|."""
    a = dev[:, :count].transpose(1, 0, 2).view(np.float16).astype(np.float64)
    b = host[:count].view(np.float16).astype(np.float64)
    return np.abs(a - b).max(axis=(1, 2)) / np.abs(b).max()


def run_case(env, cfg, seed, prompt_len, chunk, start=0, centered=True):
    """Oracle-serial vs prompt prefill of `prompt_len` tokens (the last one
    then decoded) at positions start.., with `start` earlier tokens fed to
    both serially first.

    centered (zero-mean weights): every cache row within KV_TOL. Otherwise
    (all weights of one sign, as the BASELINE weight distribution: activations
    in the hundreds and sharp softmaxes) a token's rows may move further, up to
    4 times as far as F16OperandOracle's rows move from the exact oracle's on
    the same token, and at least KV_TOL."""
    w = small_weights(cfg, seed, types={"attn_v": 14, "ffn_down": 13, "output": 14}, centered=centered)
    dec = build(env, cfg, w)
    cap = start + prompt_len + 8
    cache = env["E"].AmdKvCache(env["ctx"], env["E"].AmdQwen3Config(**cfg), cap)
    orc = ThreadedOracle(cfg, w, cap)
    rounded = None if centered else F16OperandOracle(cfg, w, cap)
    rng = np.random.default_rng(seed)
    tokens = [int(t) for t in rng.integers(cfg["vocab"], size=start + prompt_len)]
    for p in range(start):
        dec.prefill_step(cache, tokens[p], p)
        orc.step(tokens[p], p, head=False)
        if rounded is not None:
            rounded.step(tokens[p], p, head=False)
    body = tokens[start:-1]
    dec.prefill_prompt(cache, body, start, chunk)
    for i, tok in enumerate(body):
        orc.step(tok, start + i, head=False)
        if rounded is not None:
            rounded.step(tok, start + i, head=False)
    last = start + prompt_len - 1
    sel = dec.decode_step(cache, tokens[-1], last)
    ref = orc.step(tokens[-1], last)
    got = cache_arrays(env, cache, cfg)
    for l in range(cfg["layers"]):
        for name, dev, host, alt in zip("KV", got[l], (orc.keys[l], orc.values[l]),
                                        (None, None) if rounded is None else (rounded.keys[l], rounded.values[l])):
            err = per_token_err(dev, host, last + 1)
            if alt is None:
                bound = np.full_like(err, KV_TOL)
            else:
                a = alt[:last + 1].view(np.float16).astype(np.float64)
                b = host[:last + 1].view(np.float16).astype(np.float64)
                floor = np.abs(a - b).max(axis=(1, 2)) / np.abs(b).max()
                bound = np.maximum(KV_TOL, 4 * floor)
            worst = int(np.argmax(err / bound))
            print(f"layer {l} {name}: max {err.max():.2e}, tokens over {KV_TOL:g}: {int((err > KV_TOL).sum())}; "
                  f"worst vs bound: token {worst} {err[worst]:.2e} <= {bound[worst]:.2e}", flush=True)
            assert (err <= bound).all(), (l, name, worst, err[worst], bound[worst])
    logits = dec.copy_logits(0)
    lerr = max_rel_err(logits, orc.logits)
    herr = max_rel_err(dec.copy_hidden(0), orc.hidden)
    print(f"logits {lerr:.2e} hidden {herr:.2e} token {sel} (oracle {ref})", flush=True)
    assert lerr <= LOGIT_TOL, lerr
    assert herr <= LOGIT_TOL, herr
    top2 = np.sort(orc.logits.astype(np.float64))[-2:]
    if (top2[1] - top2[0]) / np.abs(orc.logits).max() > 4 * max(lerr, 1e-7):
        assert sel == ref, (sel, ref)
    dec.close()


@pytest.mark.parametrize("qh,kvh,p0,T", [(32, 8, 0, 150), (8, 2, 300, 64), (4, 4, 5, 33), (16, 2, 2040, 40),
                                          (4, 2, 0, 1), (8, 2, 64, 17)])
def test_chunk_attention_matches_oracle(env, qh, kvh, p0, T):
    """The prompt attention alone (ribn_amd_attention_prefill) against the
    oracle's attention stepped token by token over the same cache: seeded
    N(0, 1) q / k, V scaled by 4, random f16 cache rows before p0."""
    case(test="chunk_attention", qh=qh, kvh=kvh, p0=p0, T=T)
    E = env["E"]
    cfg = dict(layers=1, hidden=qh * 128, q_heads=qh, kv_heads=kvh, head_dim=128, ffn=256, vocab=1,
               rope_base=1.0e6, epsilon=1.0e-6)
    conf = E.AmdQwen3Config(**cfg)
    cap = p0 + T + 3
    rng = np.random.default_rng(qh * 100 + kvh + p0 + T)
    keys = rng.standard_normal((cap, kvh, 128)).astype(np.float16).view(np.uint16)
    values = rng.standard_normal((cap, kvh, 128)).astype(np.float16).view(np.uint16)
    cache = E.AmdKvCache(env["ctx"], conf, cap)
    if p0:
        lib, ctx = env["ctx"]._lib, env["ctx"]
        for ptr, arr in zip(cache.layer(0), (keys, values)):
            dev = np.zeros((kvh, cap, 128), np.uint16)
            dev[:, :p0] = arr[:p0].transpose(1, 0, 2)
            assert lib.ribn_amd_memcpy_htod(ctx.handle, ctypes.c_void_p(ptr), dev.ctypes.data_as(ctypes.c_void_p),
                                            dev.nbytes) == 0
    q = rng.standard_normal((T, qh * 128)).astype(np.float32)
    k = rng.standard_normal((T, kvh * 128)).astype(np.float32)
    v = (rng.standard_normal((T, kvh * 128)) * 4).astype(np.float32)
    qn = synth.gamma_numpy(128, qh + 11)
    kn = synth.gamma_numpy(128, qh + 12)
    out = to_dev(np.full(T * qh * 128, np.nan, np.float32))
    E.attention_prefill(env["ctx"], conf, cache, 0, to_dev(q.reshape(-1)), to_dev(k.reshape(-1)),
                        to_dev(v.reshape(-1)), to_dev(qn), to_dev(kn), T, p0, out)
    got = to_host(out, env["ctx"]).reshape(T, -1)
    kk = np.ascontiguousarray(keys.reshape(cap, -1))
    vv = np.ascontiguousarray(values.reshape(cap, -1))
    worst = 0.0
    for t in range(T):
        ref = O.qwen3_attention(q[t], k[t], v[t], qn, kn, 1e-6, 1e6, qh, kvh, 128, p0 + t, kk, vv)
        worst = max(worst, max_rel_err(got[t], ref))
    dev_k, dev_v = cache_arrays(env, cache, dict(cfg))[0]
    k_err = f16_err(dev_k[:, p0:p0 + T].transpose(1, 0, 2).reshape(T, -1), kk[p0:p0 + T])
    v_equal = np.array_equal(dev_v[:, p0:p0 + T].transpose(1, 0, 2).reshape(T, -1), vv[p0:p0 + T])
    print(f"attention {worst:.2e}, appended K {k_err:.2e}, V bit-exact {v_equal}", flush=True)
    assert np.isfinite(got).all()
    assert worst <= ATTN_TOL, worst
    # V is f16(v): bit-exact; K passes the norm and the rope (normwise, as the decode test)
    assert v_equal
    assert k_err <= 1e-3, k_err


@pytest.mark.parametrize("chunk", [64, 128])
def test_tiny_prompt_matches_serial_oracle(env, chunk):
    """GQA 4, two layers: 149 prompt tokens in chunks of 64 (64 + 64 + 21) or
    128 (128 + 21)."""
    case(test="prompt_tiny", chunk=chunk)
    run_case(env, TINY, 41, 150, chunk)


def test_one_signed_weights_within_the_f16_operand_floor(env):
    """The same prompt on weights of one sign (the BASELINE distribution):
    layer 1's rows of a few tokens move by up to ~7e-2, as far as f16
    operands alone move them (F16OperandOracle: 7.5e-2 on the same tokens,
    the CPU's f32 sums over f16 inputs and weights), while the next step's
    logits stay within LOGIT_TOL."""
    case(test="prompt_one_signed")
    run_case(env, TINY, 41, 150, 64, centered=False)


@pytest.mark.parametrize("qh,kvh", [(4, 4), (4, 2), (16, 2)])
def test_gqa_groups_match_serial_oracle(env, qh, kvh):
    """GQA 1, 2 and 8 (workgroups of 4 / 2 / 1 token tiles of 16)."""
    case(test="prompt_gqa", qh=qh, kvh=kvh)
    cfg = dict(layers=1, hidden=512, q_heads=qh, kv_heads=kvh, head_dim=128, ffn=768, vocab=300,
               rope_base=1.0e6, epsilon=1.0e-6)
    run_case(env, cfg, 50 + qh + kvh, 71, 32)


def test_prompt_continues_a_cache(env):
    """A prompt at position 37 of a cache the serial path filled (keys before
    the chunk come from the cache, the chunk's own from its append)."""
    case(test="prompt_continues")
    run_case(env, TINY, 43, 90, 16, start=37)


def test_qwen3_8b_layer_geometry(env):
    """One Qwen3-8B-shaped layer (hidden 4096, 32/8 heads, SwiGLU 12288, Q6_K
    v, Q5_K down): 129 prompt tokens in chunks of 128 (128 + a one-token chunk)."""
    case(test="prompt_wide")
    run_case(env, WIDE, 44, 130, 128)


def test_prompt_errors(env):
    case(test="prompt_errors")
    E = env["E"]
    w = small_weights(TINY, 45)
    dec = build(env, TINY, w)
    cache = E.AmdKvCache(env["ctx"], E.AmdQwen3Config(**TINY), 32)
    with pytest.raises(E.AmdModelKernelError) as e:
        dec.prefill_prompt(cache, [1, 2, 3], 0, 8)
    assert e.value.kind == "InvalidArgument"
    with pytest.raises(E.AmdModelKernelError) as e:
        dec.prefill_prompt(cache, list(range(30)), 5, 16)
    assert e.value.kind == "PositionOverflow"
    with pytest.raises(E.AmdModelKernelError) as e:
        dec.prefill_prompt(cache, [1, TINY["vocab"]], 0, 16)
    assert e.value.kind == "InvalidPlan"
    with pytest.raises(E.AmdModelKernelError) as e:
        dec.prefill_prompt(cache, [], 0, 16)
    assert e.value.kind == "InputLength"
    dec.reserve_prompt(64)
    dec.prefill_prompt(cache, list(range(20)), 0, 16)  # still usable after the errors
    env["ctx"].synchronize()
    dec.close()


@pytest.mark.parametrize("qh,kvh,p0,T", [(128, 128, 0, 33), (128, 128, 70, 129), (128, 64, 5, 139), (128, 32, 0, 163),
                                         (128, 32, 61, 192), (128, 16, 3, 487), (32, 8, 0, 705), (32, 8, 1000, 768)])
def test_wide_chunk_attention(env, qh, kvh, p0, T):
    """The many-token form of the chunk attention (32 tokens a wave, two key halves): every GQA
    width, ragged last tiles, chunks that continue a cache, against an f64 attention over the f16
    keys and values the call left in the cache (the bound of the narrow form's test)."""
    import torch
    case(test="wide_chunk_attention", qh=qh, kvh=kvh, p0=p0, T=T)
    E = env["E"]
    cfg = dict(layers=1, hidden=4096, q_heads=qh, kv_heads=kvh, head_dim=128, ffn=256, vocab=1, rope_base=1.0e6,
               epsilon=1.0e-6)
    conf = E.AmdQwen3Config(**cfg)
    cap = p0 + T + 3
    rng = np.random.default_rng(qh + kvh + p0 + T)
    cache = E.AmdKvCache(env["ctx"], conf, cap)
    for ptr in cache.layer(0):
        dev = rng.standard_normal((kvh, cap, 128)).astype(np.float16)
        assert env["ctx"]._lib.ribn_amd_memcpy_htod(env["ctx"].handle, ctypes.c_void_p(ptr),
                                                    dev.ctypes.data_as(ctypes.c_void_p), dev.nbytes) == 0
    q = rng.standard_normal((T, qh * 128)).astype(np.float32)
    k = rng.standard_normal((T, kvh * 128)).astype(np.float32)
    v = (rng.standard_normal((T, kvh * 128)) * 4).astype(np.float32)
    qn, kn = synth.gamma_numpy(128, 1), synth.gamma_numpy(128, 2)
    out = to_dev(np.full(T * qh * 128, np.nan, np.float32))
    E.attention_prefill(env["ctx"], conf, cache, 0, to_dev(q.reshape(-1)), to_dev(k.reshape(-1)), to_dev(v.reshape(-1)),
                        to_dev(qn), to_dev(kn), T, p0, out)
    got = to_host(out, env["ctx"]).reshape(T, qh, 128)
    dev_k, dev_v = (torch.from_numpy(np.ascontiguousarray(a)).view(torch.float16).cuda().double()
                    for a in cache_arrays(env, cache, cfg)[0])
    qd = torch.from_numpy(q).cuda().double().view(T, qh, 128)
    qd = qd * torch.rsqrt((qd * qd).mean(-1, keepdim=True) + 1e-6) * torch.from_numpy(qn).cuda().double()
    pos = p0 + torch.arange(T, device="cuda:0")
    ang = pos.double()[:, None] * 1.0e6 ** (-torch.arange(64, device="cuda:0").double() / 64)
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]
    qd = torch.cat((qd[..., :64] * cos - qd[..., 64:] * sin, qd[..., :64] * sin + qd[..., 64:] * cos), -1)
    seen = torch.arange(p0 + T, device="cuda:0")[None] <= pos[:, None]
    for h in range(qh):
        kh, vh = dev_k[h // (qh // kvh), :p0 + T], dev_v[h // (qh // kvh), :p0 + T]
        sc = (qd[:, h] @ kh.t().contiguous()) / 128 ** 0.5
        ref = (torch.softmax(sc.masked_fill(~seen, -np.inf), -1) @ vh).cpu().numpy()
        assert max_rel_err(got[:, h], ref) <= ATTN_TOL, h


@pytest.mark.parametrize("t,kvh,T", [(12, 8, 300), (13, 8, 333), (14, 16, 257), (12, 8, 129)])
def test_prompt_kv_pair(env, t, kvh, T):
    """k and v of a prompt chunk in one paired matmul (and, at 129 tokens, the split it cannot fill):
    the appended keys and values of a one-layer decoder against f64 products of the dequantised
    weights, normwise within the f16 product's 1e-3 and the f16 cache's half unit, 2^-11."""
    import torch
    case(test="prompt_kv_pair", t=t, kvh=kvh, T=T)
    E, ctx = env["E"], env["ctx"]
    h, vocab, nkv = 2048, 320, kvh * 128
    cfg = dict(layers=1, hidden=h, q_heads=16, kv_heads=kvh, head_dim=128, ffn=256, vocab=vocab, rope_base=1.0e6,
               epsilon=1.0e-6)
    store = E.AmdWeightStore(ctx)
    enc, w = {}, {}
    for i, (nm, ty, k, n) in enumerate((("token_embd", 12, h, vocab), ("output", 14, h, vocab), ("attn_q", 12, h, h),
                                        ("attn_k", t, h, nkv), ("attn_v", t, h, nkv), ("attn_output", 12, h, h),
                                        ("ffn_gate", 12, h, 256), ("ffn_up", 12, h, 256), ("ffn_down", 13, 256, h))):
        enc[nm] = synth.kquant_numpy(ty, k, n, seed=900 + i + t, centered=True)
        store.materialize_quantized(nm, [k, n], ty, enc[nm])
        w[nm] = store.quantized_tensor(nm)
    norms = {nm: synth.gamma_numpy(n, seed=950 + i) for i, (nm, n) in enumerate(
        (("output_norm", h), ("attn_norm", h), ("ffn_norm", h), ("attn_q_norm", 128), ("attn_k_norm", 128)))}
    dev = {nm: to_dev(v) for nm, v in norms.items()}
    layer = {nm: w[nm] for nm in ("attn_q", "attn_k", "attn_v", "attn_output", "ffn_gate", "ffn_up", "ffn_down")}
    layer.update({nm: dev[nm] for nm in ("attn_norm", "ffn_norm", "attn_q_norm", "attn_k_norm")})
    conf = E.AmdQwen3Config(**cfg)
    dec = E.AmdQwen3Decode(ctx, conf, w["token_embd"], w["output"], dev["output_norm"], [layer], 1)
    cache = E.AmdKvCache(ctx, conf, T)
    tokens = np.random.default_rng(T).integers(0, vocab, T)
    dec.prefill_prompt(cache, tokens, 0)
    ctx.synchronize()
    got_k, got_v = (a.view(np.float16).astype(np.float64) for a in cache_arrays(env, cache, cfg)[0])

    def rms(x, g):
        return x / np.sqrt((x * x).mean(-1, keepdims=True) + 1e-6) * g.astype(np.float64)

    x = O.dequantize_tensor(12, enc["token_embd"]).reshape(vocab, h)[tokens].astype(np.float64)
    x = rms(x, norms["attn_norm"])
    k, v = (x @ O.dequantize_tensor(t, enc[nm]).reshape(nkv, h).T.astype(np.float64) for nm in ("attn_k", "attn_v"))
    k = rms(k.reshape(T, kvh, 128), norms["attn_k_norm"])
    ang = np.arange(T)[:, None] * 1.0e6 ** (-np.arange(64) / 64.0)
    c, s = np.cos(ang)[:, None], np.sin(ang)[:, None]
    k = np.concatenate((k[..., :64] * c - k[..., 64:] * s, k[..., :64] * s + k[..., 64:] * c), -1)
    for got, ref in ((got_k, k), (got_v, v.reshape(T, kvh, 128))):
        assert max_rel_err(got.transpose(1, 0, 2), ref) <= 1e-3 + 2.0 ** -11
    dec.close()


@pytest.mark.parametrize("qh,kvh,p0,T", [(8, 8, 0, 70), (16, 8, 5, 70), (32, 8, 61, 50), (64, 8, 0, 40),
                                         (128, 128, 70, 129), (128, 64, 5, 139), (128, 32, 61, 192), (128, 16, 3, 487)])
@pytest.mark.parametrize("what,value", [("v", np.inf), ("v", -7e4), ("v", np.nan), ("k", np.nan)])
def test_chunk_attention_non_finite(env, qh, kvh, p0, T, what, value):
    """A value (or key) that is not finite in the f16 cache reaches the tokens that attend it and no
    other: in both forms of the chunk attention and every GQA width, tokens before it, other heads and
    (for a value) other dims give the bits they give without it; -7e4 rounds to an f16 infinity."""
    case(test="chunk_attention_non_finite", qh=qh, kvh=kvh, p0=p0, T=T, what=what, value=value)
    E, per = env["E"], qh // kvh
    cfg = dict(layers=1, hidden=4096, q_heads=qh, kv_heads=kvh, head_dim=128, ffn=256, vocab=1, rope_base=1.0e6,
               epsilon=1.0e-6)
    conf = E.AmdQwen3Config(**cfg)
    cap = p0 + T
    rng = np.random.default_rng(qh + kvh + p0 + T)
    old = [rng.standard_normal((kvh, cap, 128)).astype(np.float16) for _ in range(2)]
    q = rng.standard_normal((T, qh * 128)).astype(np.float32)
    kv = {nm: rng.standard_normal((T, kvh * 128)).astype(np.float32) for nm in "kv"}
    qn, kn = to_dev(synth.gamma_numpy(128, 1)), to_dev(synth.gamma_numpy(128, 2))

    def run(k, v):
        cache = E.AmdKvCache(env["ctx"], conf, cap)
        for ptr, dev in zip(cache.layer(0), old):
            assert env["ctx"]._lib.ribn_amd_memcpy_htod(env["ctx"].handle, ctypes.c_void_p(ptr),
                                                        dev.ctypes.data_as(ctypes.c_void_p), dev.nbytes) == 0
        out = to_dev(np.zeros(T * qh * 128, np.float32))
        E.attention_prefill(env["ctx"], conf, cache, 0, to_dev(q.reshape(-1)), to_dev(k.reshape(-1)), to_dev(v.reshape(-1)),
                            qn, kn, T, p0, out)
        return to_host(out, env["ctx"]).reshape(T, kvh, per, 128)

    want = run(kv["k"], kv["v"])
    assert np.all(np.isfinite(want))
    for at in (T // 2 + 3, T - 2):
        head, dim = at % kvh, (37 * at) % 128
        bad = {nm: a.copy() for nm, a in kv.items()}
        bad[what][at, head * 128 + dim] = value
        got = run(bad["k"], bad["v"])
        reached = got[at:, head, :, dim] if what == "v" else got[at:, head]
        assert not np.any(np.isfinite(reached)), at
        reached[...] = (want[at:, head, :, dim] if what == "v" else want[at:, head])
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), at
