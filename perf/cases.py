"""Performance cases of leankv_amd: what a program that decodes with this library has it do.

Every case goes through a public entry point at the sizes of the decoder shape that the tests and bench.py use
(hidden 4096, ffn 14336, 32 query heads over 8 kv heads of 128 dims, vocabulary 32768) or at other generic ones.

  kind      entry points                                      what it stands for
  proj      sparse_qkv + sparse_gemv / batched_qkv + ...      the attention projections of one decode step (q, k, v, o)
  mlp       sparse_gateup_swiglu + sparse_gemv / batched_*    the MLP of one decode step
  quantize  TurboQuantMSE.quantize                            quantizing the K and V of a prompt
  readback  TurboQuantCache.__getitem__                       the K / V that the cache hands to any attention (its default mode)
  prefill   TurboQuantCache.update + prefill_attention        one layer of a prompt, whole or in chunks
  attn      kernels.tq_decode_attn                            decode attention over the packed cache
  paged     PagedTurboQuantCache.decode_attention             the same over pages, sequences of different lengths
  step      LeanKVEngine / BatchedEngine                      a whole graph-replayed decode step of a shallow decoder
"""

from __future__ import annotations

import functools
import math

import numpy as np
import torch

D = 128  # head size
KINDS = ("proj", "mlp", "quantize", "readback", "prefill", "attn", "paged", "step")

# Lloyd-Max centroids of a coordinate of a random unit vector in 128 dimensions (the upper half; the lower mirrors it)
_HALF = {
    1: (0.07066157273809426,),
    2: (0.039990945215356365, 0.1330401982533685),
    3: (0.021602468667239208, 0.06658059531595685, 0.11813298369899362, 0.188390613802078),
    4: (0.011296498142743886, 0.03413402823112085, 0.05774453560525709, 0.0827925666730958, 0.11024706538276369,
        0.14176165429673318, 0.18079372947217437, 0.23762718673095365),
}


def listed():
    return [
        # one token through q, k, v and o at 40 % sparsity: the smallest launches of a decode step
        dict(name="proj_1row", kind="proj", rows=1, hidden=4096, heads=32, kv=8, sparsity=0.4),
        # one token through the MLP at 40 % sparsity: most of a decode step's bytes
        dict(name="mlp_1row", kind="mlp", rows=1, hidden=4096, ffn=14336, sparsity=0.4),
        # sixteen sequences' tokens through the MLP (dense, as the projections are dispatched for several rows)
        dict(name="mlp_16rows", kind="mlp", rows=16, hidden=4096, ffn=14336, sparsity=0.0),
        # K and V of a 4096-token prompt, 3 bits
        dict(name="quantize_kv", kind="quantize", vectors=8 * 4096, bits=3, half=True),
        # the whole K / V of a 4096-token sequence read back for another attention implementation
        dict(name="readback_4096", kind="readback", batch=1, kv=8, length=4096, hot=64, bits=3),
        # one layer of a 4096-token prompt
        dict(name="prefill_4096", kind="prefill", batch=1, heads=32, kv=8, length=4096, chunks=1, hot=64, bits=3),
        # four prompts of a ragged length in chunks, 4 bits, a longer window
        dict(name="prefill_chunks", kind="prefill", batch=4, heads=32, kv=8, length=1201, chunks=3, hot=128, bits=4),
        # decode attention of sixteen sequences at context 4096, 3 bits
        dict(name="attn_16x4096", kind="attn", batch=16, heads=32, kv=8, length=4096, hot=64, bits=3),
        # one long sequence, 2 bits
        dict(name="attn_1x32768", kind="attn", batch=1, heads=32, kv=8, length=32768, hot=64, bits=2),
        # sixteen sequences of mixed lengths in pages
        dict(name="paged_16_mixed", kind="paged", batch=16, heads=32, kv=8, length=4096, hot=64, bits=3, page=16),
        # a decode step of one sequence at context 4096 on the sparse projections and a packed cache.  The sparsity is
        # low because a whole step at 40 % cannot be compared: a value that rounding moves over its threshold changes
        # the next projection by a per cent, which moves others (the products at 40 % are proj_1row and mlp_1row)
        dict(name="step_1row", kind="step", rows=1, layers=4, length=4096, hot=64, bits=3, sparsity=0.03),
        # a decode step of sixteen sequences (dense projections, as several rows are dispatched)
        dict(name="step_16rows", kind="step", rows=16, layers=2, length=1024, hot=64, bits=3, sparsity=0.03),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(KINDS)
    bits = rng.choice((1, 2, 3, 3, 4))
    hot = rng.choice((16, 48, 64, 64, 100, 128, 256))
    kv = rng.choice((1, 2, 4, 8, 8))
    heads = kv * rng.choice((1, 2, 4, 4, 8) if kv < 8 else (1, 2, 4, 4))
    sparsity = rng.choice((0.0, round(rng.uniform(0.3, 0.5), 3), round(rng.uniform(0.3, 0.5), 3)))
    if kind == "proj":
        return dict(kind=kind, rows=_log_int(rng, 1, 32), hidden=8 * _log_int(rng, 64, 512), heads=heads, kv=kv,
                    sparsity=sparsity)
    if kind == "mlp":
        hidden = 8 * _log_int(rng, 64, 512)
        return dict(kind=kind, rows=_log_int(rng, 1, 32), hidden=hidden, ffn=8 * int(hidden * rng.uniform(2, 3.5) / 8),
                    sparsity=sparsity)
    if kind == "quantize":
        return dict(kind=kind, vectors=_log_int(rng, 1, 65536), bits=bits, half=rng.random() < 0.5)
    if kind == "readback":
        length = _log_int(rng, 20, 16384)
        return dict(kind=kind, batch=rng.randint(1, max(1, min(16, 32768 // length))), kv=kv, length=length, hot=hot,
                    bits=bits)
    if kind == "prefill":
        length = _log_int(rng, 33, 4000)
        return dict(kind=kind, batch=rng.randint(1, max(1, min(4, 4000 // length))), heads=heads, kv=kv, length=length,
                    chunks=rng.randint(1, 3), hot=hot, bits=bits)
    if kind == "attn":
        length = _log_int(rng, 20, 32768)
        return dict(kind=kind, batch=rng.randint(1, max(1, min(32, 65536 // length))), heads=heads, kv=kv,
                    length=length, hot=hot, bits=bits)
    if kind == "paged":
        length = _log_int(rng, 64, 8192)
        return dict(kind=kind, batch=rng.randint(1, max(1, min(16, 65536 // length))), heads=heads, kv=kv,
                    length=length, hot=hot, bits=bits, page=rng.choice((16, 32, 64, 128)))
    rows = rng.choice((1, 1, rng.randint(2, 8), rng.randint(9, 32)))
    return dict(kind=kind, rows=rows, layers=rng.randint(1, 2), length=_log_int(rng, 33, 8192 // min(rows, 8)),
                hot=rng.choice((48, 64, 128)), bits=bits, sparsity=round(rng.uniform(0.01, 0.04), 3))


# ------------------------------------------------------------------------------------------------------------ inputs
def _gen(seed, tag):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + tag) % (1 << 62))
    return g


def _randn(shape, seed, tag, scale=1.0, dtype=torch.float16):
    return (torch.randn(shape, generator=_gen(seed, tag), device="cuda") * scale).to(dtype)


def _weight(n, z, seed, tag):
    """An fp16 [n, z] weight stored column-major, as prepare_weight_for_sparse_gemv leaves it."""
    return _randn((z, n), seed, tag, 0.02).t()


def _kv(shape, seed, tag):
    """Keys or values: normal coordinates, four of the 128 channels ten times as large."""
    x = _randn(shape, seed, tag)
    x[..., [5, 37, 70, 101]] *= 10
    return x


def _abs_quantile(p):
    """|N(0, 1)| below this with probability p."""
    return float(torch.special.ndtri(torch.tensor(0.5 + p / 2, dtype=torch.float64))) if p > 0 else 0.0


@functools.lru_cache(maxsize=None)
def _swiglu_quantile(p, std):
    """The p-quantile of |silu(g) u| for normal g and u of this deviation."""
    if p <= 0:
        return 0.0
    z = np.random.RandomState(0).randn(2, 1 << 20) * std
    return float(np.quantile(np.abs(z[0] / (1 + np.exp(-z[0])) * z[1]), p))


def _centroids(bits):
    half = _HALF[bits]
    return torch.tensor([-c for c in reversed(half)] + list(half), dtype=torch.float64)


def _rotation(seed):
    """The orthogonal matrix of a rotation seed: QR of a seeded normal matrix, the diagonal of R positive."""
    g = torch.Generator(device="cpu")
    g.manual_seed(seed)
    q, r = torch.linalg.qr(torch.randn(D, D, generator=g, dtype=torch.float32))
    return (q * torch.sign(torch.diag(r)).unsqueeze(0)).contiguous()


def _codes(x, pi, bits):
    """(codes, norms) of x [..., 128] in x's own precision: the bucket of each rotated unit coordinate."""
    c = _centroids(bits)
    b = ((c[1:] + c[:-1]) / 2).float().to(x.device, x.dtype)  # the decision boundaries are fp32 midpoints
    n = x.norm(dim=-1)
    y = (x / (n + 1e-10).unsqueeze(-1)) @ pi.to(x.device, x.dtype).t()
    return torch.bucketize(y, b), n


def _pack(codes, bits):
    width = {1: 1, 2: 2, 3: 4, 4: 4}[bits]
    per = 8 // width
    r = codes.to(torch.uint8).reshape(*codes.shape[:-1], -1, per)
    sh = torch.arange(per, device=codes.device, dtype=torch.uint8) * width
    return (r << sh).sum(dim=-1, dtype=torch.uint8)


def _cold64(x, pi, bits):
    """What the packed store holds of x (fp16), in 64 bits: centroids rotated back and scaled by the norm."""
    codes, n = _codes(x.double(), pi.double(), bits)
    c = _centroids(bits).float().double().to(x.device)
    return (c[codes] @ pi.double().to(x.device)) * n.unsqueeze(-1)


def _stored64(x, pi, bits, hot, length=None):
    """K or V [..., length, 128] as the cache holds it: all but the newest `hot` tokens through the packed store."""
    length = x.shape[-2] if length is None else length
    cold = max(0, length - hot)
    x = x[..., :length, :]
    return torch.cat([_cold64(x[..., :cold, :], pi, bits), x[..., cold:, :].double()], dim=-2)


def _attend64(q, k, v, first):
    """Causal attention in 64 bits: q [H, S, 128] (query i sees keys 0 .. first + i) over k, v [kv, T, 128]."""
    g = q.shape[0] // k.shape[0]
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    T = k.shape[1]
    for h in range(q.shape[0]):
        for s0 in range(0, q.shape[1], 1024):
            s = (q[h, s0:s0 + 1024].double() @ k[h // g].t().contiguous()) / math.sqrt(D)
            i = torch.arange(s0, s0 + s.shape[0], device=q.device).unsqueeze(1)
            s.masked_fill_(torch.arange(T, device=q.device).unsqueeze(0) > first + i, -math.inf)
            out[h, s0:s0 + 1024] = torch.softmax(s, dim=-1) @ v[h // g]
    return out


def _sparse64(x, w, t):
    """rows of x through w [n, z], coordinates with |x| <= t dropped."""
    x = x.double()
    return torch.where(x.abs() > t, x, torch.zeros_like(x)) @ w.double().t().contiguous()


def _silu64(x):
    return x * torch.sigmoid(x)


# -------------------------------------------------------------------------------------------------- the decoder's step
_HIDDEN, _FFN, _HEADS, _KV, _VOCAB, _EPS, _THETA = 4096, 14336, 32, 8, 32768, 1e-5, 10000.0
_SHAPES = dict(q_proj=(_HEADS * D, _HIDDEN), k_proj=(_KV * D, _HIDDEN), v_proj=(_KV * D, _HIDDEN),
               o_proj=(_HIDDEN, _HEADS * D), gate_proj=(_FFN, _HIDDEN), up_proj=(_FFN, _HIDDEN),
               down_proj=(_HIDDEN, _FFN))


def _decoder(case, seed):
    """name -> fp16 tensor of a shallow decoder, [out, in] weights as a checkpoint holds them."""
    w = {"model.embed_tokens.weight": _randn((_VOCAB, _HIDDEN), seed, 1, 0.02),
         "lm_head.weight": _randn((_VOCAB, _HIDDEN), seed, 2, 0.02),
         "model.norm.weight": 1 + _randn((_HIDDEN,), seed, 3, 0.1)}
    for i in range(case["layers"]):
        p = "model.layers.%d." % i
        for j, (name, shape) in enumerate(_SHAPES.items()):
            part = "mlp." if name in ("gate_proj", "up_proj", "down_proj") else "self_attn."
            w[p + part + name + ".weight"] = _randn(shape, seed, 100 * (i + 1) + j, 0.02)
        for j, name in enumerate(("input_layernorm", "post_attention_layernorm")):
            w[p + name + ".weight"] = 1 + _randn((_HIDDEN,), seed, 100 * (i + 1) + 20 + j, 0.1)
    return w


def _thresholds(case):
    """About the case's share of each projection's inputs lies below these."""
    p, std = case["sparsity"], 0.02 * math.sqrt(_HIDDEN)
    x = _abs_quantile(p)
    spread = std * min(1.0, math.sqrt(math.exp(std ** 4) / case["length"]))  # of an attention output over random values
    return dict(q_proj=x, k_proj=x, v_proj=x, o_proj=x * spread, gate_proj=x, up_proj=x,
                down_proj=_swiglu_quantile(p, 0.97 * std))


def _context(case, seed, layer):
    shape = (case["rows"], _KV, case["length"], D)
    return _randn(shape, seed, 5000 + 2 * layer, 1.28), _randn(shape, seed, 5001 + 2 * layer, 1.28)


def _tokens(case, seed):
    return torch.randint(0, _VOCAB, (case["rows"],), generator=_gen(seed, 9), device="cuda")


_STEPS = 64  # positions a state's passes walk before they start again at the context


def _prepare_step(case, seed):
    from transformers import MistralConfig, MistralForCausalLM
    from transformers.models.mistral.modeling_mistral import MistralRotaryEmbedding

    from leankv_amd.engine import BatchedEngine, LeanKVEngine
    from leankv_amd.teal.patching import apply_teal
    from leankv_amd.turboquant.cache import TurboQuantCache

    cfg = MistralConfig(vocab_size=_VOCAB, hidden_size=_HIDDEN, intermediate_size=_FFN,
                        num_hidden_layers=case["layers"], num_attention_heads=_HEADS, num_key_value_heads=_KV,
                        head_dim=D, rms_norm_eps=_EPS, rope_theta=_THETA, max_position_embeddings=32768,
                        sliding_window=None, tie_word_embeddings=False)
    with torch.device("meta"):
        model = MistralForCausalLM(cfg)
    model.load_state_dict(_decoder(case, seed), assign=True)
    model.model.rotary_emb = MistralRotaryEmbedding(cfg, device="cuda")
    model.eval().requires_grad_(False)
    th = _thresholds(case)
    apply_teal(model, thresholds={i: th for i in range(case["layers"])}, use_triton=True)
    rows, length = case["rows"], case["length"]
    cache = TurboQuantCache(bits=case["bits"], num_layers=case["layers"], hot_buffer_size=case["hot"], device="cuda",
                            max_seq_len=length + _STEPS)
    for i in range(case["layers"]):
        cache.update(*_context(case, seed, i), i)
    names = ("_k_codes", "_v_codes", "_k_norms", "_v_norms", "_k_hot", "_v_hot")
    kept = [[t.clone() for t in getattr(cache, n)] for n in names]
    tok = _tokens(case, seed)
    # the first step runs eagerly and the step is captured; the cache then goes back to the context
    if rows == 1:
        eng = LeanKVEngine(model, cache, length + _STEPS)
        eng.start(tok, length)
        eng.step()
        eng.capture()
    else:
        eng = BatchedEngine(model, cache, rows)
        eng.set_position(length)
        eng.tok.copy_(tok)
        eng.step()
    for n, saved in zip(names, kept):
        for t, s in zip(getattr(cache, n), saved):
            t.copy_(s)
    return dict(kind="step", eng=eng, tok=tok, at=0, length=length, rows=rows)


def _run_step(s):
    """A decode step of given tokens: each pass feeds the next position."""
    eng, pos = s["eng"], s["length"] + s["at"] % _STEPS
    s["at"] += 1
    if s["rows"] == 1:
        eng.start(s["tok"], pos)
    else:
        eng.set_position(pos)
        eng.tok.copy_(s["tok"])
    eng.step()
    return eng.logits


def _exact_step(case, seed):
    w, tok, rows, length = _decoder(case, seed), _tokens(case, seed), case["rows"], case["length"]
    th = _thresholds(case) if rows == 1 else dict.fromkeys(_SHAPES, 0.0)
    inv = 1.0 / _THETA ** (torch.arange(0, D, 2, device="cuda", dtype=torch.float64) / D)
    ang = torch.cat([length * inv, length * inv])
    cos, sin = ang.cos(), ang.sin()

    def norm(x, name):
        return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + _EPS) * w[name].double()

    def rope(x):
        half = torch.cat([-x[..., D // 2:], x[..., :D // 2]], dim=-1)
        return x * cos + half * sin

    x = w["model.embed_tokens.weight"][tok].double()
    for i in range(case["layers"]):
        p = "model.layers.%d." % i

        def lin(x, name, part):
            return _sparse64(x, w[p + part + name + ".weight"], th[name])

        h = norm(x, p + "input_layernorm.weight")
        q = rope(lin(h, "q_proj", "self_attn.").view(rows, _HEADS, D))
        k = rope(lin(h, "k_proj", "self_attn.").view(rows, _KV, D))
        v = lin(h, "v_proj", "self_attn.").view(rows, _KV, D)
        ck, cv = _context(case, seed, i)
        pk, pv = _rotation(42 + 2 * i), _rotation(43 + 2 * i)
        cold = max(0, length + 1 - case["hot"])
        o = torch.empty(rows, _HEADS * D, dtype=torch.float64, device="cuda")
        for b in range(rows):
            kk = torch.cat([_cold64(ck[b, :, :cold], pk, case["bits"]), ck[b, :, cold:].double(), k[b].unsqueeze(1)], 1)
            vv = torch.cat([_cold64(cv[b, :, :cold], pv, case["bits"]), cv[b, :, cold:].double(), v[b].unsqueeze(1)], 1)
            o[b] = _attend64(q[b].unsqueeze(1), kk, vv, length).reshape(-1)
        x = x + lin(o, "o_proj", "self_attn.")
        h = norm(x, p + "post_attention_layernorm.weight")
        a = _silu64(lin(h, "gate_proj", "mlp.")) * lin(h, "up_proj", "mlp.")
        x = x + lin(a, "down_proj", "mlp.")
    logits = norm(x, "model.norm.weight") @ w["lm_head.weight"].double().t().contiguous()
    return logits.view(-1) if rows == 1 else logits.view(rows, 1, _VOCAB)


# ------------------------------------------------------------------------------------------------------------ prepare
def _x_rows(case, seed, n, tag, scale=1.0):
    return _randn((case["rows"], n), seed, tag, scale)


def _proj_inputs(case, seed):
    nq, nkv, z = case["heads"] * D, case["kv"] * D, case["hidden"]
    t = _abs_quantile(case["sparsity"]) if case["rows"] == 1 else 0.0
    return dict(x=_x_rows(case, seed, z, 1), a=_x_rows(case, seed, nq, 2, 0.08), wq=_weight(nq, z, seed, 3),
                wk=_weight(nkv, z, seed, 4), wv=_weight(nkv, z, seed, 5), wo=_weight(z, nq, seed, 6), t=t, ta=0.08 * t)


def _mlp_inputs(case, seed):
    f, z = case["ffn"], case["hidden"]
    one = case["rows"] == 1
    return dict(x=_x_rows(case, seed, z, 1), wg=_weight(f, z, seed, 2), wu=_weight(f, z, seed, 3),
                wd=_weight(z, f, seed, 4), t=_abs_quantile(case["sparsity"]) if one else 0.0,
                ta=_swiglu_quantile(case["sparsity"], 0.97 * 0.02 * math.sqrt(z)) if one else 0.0)


def _chunk_ends(case):
    n, k = case["length"], case["chunks"]
    return [n * (i + 1) // k for i in range(k)]


def _paged_lengths(case, seed):
    """Lengths from an eighth of the longest up; the longest is the case's."""
    r = np.random.RandomState(seed % (1 << 31))
    n = case["length"]
    return [n] + [int(v) for v in r.randint(max(1, n // 8), n + 1, case["batch"] - 1)]


def _paged_kv(case, seed, b, n):
    return _kv((case["kv"], n, D), seed, 10 + 2 * b), _kv((case["kv"], n, D), seed, 11 + 2 * b)


def _attn_cold(case, seed):
    """Packed codes and norms of every cold token (plain torch), rotations and the hot tokens."""
    B, kv, n, hot, bits = case["batch"], case["kv"], case["length"], case["hot"], case["bits"]
    cold = max(0, n - hot)
    out = dict(cold=cold)
    for j, nm in enumerate("kv"):
        x = _kv((B, kv, n, D), seed, 10 + j)
        pi = _rotation(42 + j)
        codes, norms = _codes(x[:, :, :cold].float(), pi, bits)
        out[nm] = dict(codes=codes, norms=norms, pi=pi, hot=x[:, :, cold:])
    return out


def prepare(case, seed):
    kind = case["kind"]
    if kind == "step":
        return _prepare_step(case, seed)
    if kind in ("proj", "mlp"):
        return dict(case, **(_proj_inputs if kind == "proj" else _mlp_inputs)(case, seed))
    if kind == "quantize":
        from leankv_amd.turboquant.quantizer import TurboQuantMSE

        dt = torch.float16 if case["half"] else torch.float32
        k, v = (_kv((case["vectors"], D), seed, j).to(dt) for j in (1, 2))
        return dict(kind=kind, k=k, v=v, qk=TurboQuantMSE(D, bits=case["bits"], device="cuda", seed=42),
                    qv=TurboQuantMSE(D, bits=case["bits"], device="cuda", seed=43))
    if kind in ("readback", "prefill"):
        from leankv_amd.turboquant.cache import TurboQuantCache

        fused = kind == "prefill"
        cache = TurboQuantCache(bits=case["bits"], num_layers=1, hot_buffer_size=case["hot"], device="cuda",
                                max_seq_len=case["length"] + 128, fused_attention=fused)
        shape = (case["batch"], case["kv"], case["length"], D)
        k, v = _kv(shape, seed, 1), _kv(shape, seed, 2)
        if not fused:
            cache.update(k, v, 0)
            return dict(kind=kind, cache=cache)
        ends = _chunk_ends(case)
        parts, at = [], 0
        for i, e in enumerate(ends):
            q = _randn((case["batch"], case["heads"], e - at, D), seed, 20 + i)
            parts.append((k[:, :, at:e].contiguous(), v[:, :, at:e].contiguous(), q))
            at = e
        return dict(kind=kind, cache=cache, parts=parts, cold=max(0, case["length"] - case["hot"]))
    if kind == "attn":
        c = _attn_cold(case, seed)
        B, kv, n, hot, cap = case["batch"], case["kv"], case["length"], case["hot"], case["length"] + 128
        slots = torch.arange(c["cold"], n, device="cuda") % hot
        s = dict(kind=kind, bits=case["bits"], cent=_centroids(case["bits"]).float().cuda(), max_len=cap + hot,
                 q=_randn((B, case["heads"], D), seed, 3), len=torch.tensor([n], dtype=torch.int32, device="cuda"))
        for nm in "kv":
            packed = _pack(c[nm]["codes"], case["bits"])
            codes = torch.zeros(B, kv, cap, packed.shape[-1], dtype=torch.uint8, device="cuda")
            codes[:, :, :c["cold"]] = packed
            norms = torch.zeros(B, kv, cap, device="cuda")
            norms[:, :, :c["cold"]] = c[nm]["norms"]
            ring = torch.zeros(B, kv, hot, D, dtype=torch.float16, device="cuda")
            ring[:, :, slots] = c[nm]["hot"]
            s.update({nm + "_codes": codes, nm + "_norms": norms, nm + "_hot": ring, "Pi" + nm.upper(): c[nm]["pi"].cuda()})
        return s
    from leankv_amd.turboquant.paged_tq_cache import PagedTurboQuantCache

    lens, page = _paged_lengths(case, seed), case["page"]
    pages = sum(-(-n // page) for n in lens)
    cache = PagedTurboQuantCache(num_layers=1, num_kv_heads=case["kv"], num_q_heads=case["heads"], bits=case["bits"],
                                 hot_buffer_size=case["hot"], page_size=page, max_pages=pages + 8,
                                 max_batch_size=len(lens), device="cuda")
    for b, n in enumerate(lens):
        cache.append(0, b, *_paged_kv(case, seed, b, n))
    return dict(kind=kind, cache=cache, q=_randn((len(lens), case["heads"], D), seed, 3))


# ---------------------------------------------------------------------------------------------------------------- run
def run(s):
    kind = s["kind"]
    if kind == "step":
        return _run_step(s)
    if kind == "proj":
        from leankv_amd.teal.kernels.sparse_gemv import batched_qkv, batched_sparse_gemm, sparse_gemv, sparse_qkv

        if s["rows"] == 1:
            q, k, v = sparse_qkv(s["x"], s["wq"], s["wk"], s["wv"], s["t"], s["t"], s["t"])
            return q, k, v, sparse_gemv(s["a"].view(1, 1, -1), s["wo"], s["ta"])
        q, k, v = batched_qkv(s["x"], s["wq"], s["wk"], s["wv"])
        return q, k, v, batched_sparse_gemm(s["a"], s["wo"], 0.0)
    if kind == "mlp":
        from leankv_amd.teal.kernels.sparse_gemv import (batched_gateup_swiglu, batched_sparse_gemm,
                                                         sparse_gateup_swiglu, sparse_gemv)

        if s["rows"] == 1:
            h = sparse_gateup_swiglu(s["x"], s["wg"], s["wu"], s["t"], s["t"])
            return h, sparse_gemv(h, s["wd"], s["ta"])
        h = batched_gateup_swiglu(s["x"], s["wg"], s["wu"])
        return h, batched_sparse_gemm(h, s["wd"], 0.0)
    if kind == "quantize":
        a, b = s["qk"].quantize(s["k"]), s["qv"].quantize(s["v"])
        return a.indices, a.norms, b.indices, b.norms
    if kind == "readback":
        return s["cache"][0]
    if kind == "prefill":
        c, n = s["cache"], s["cold"]
        c.reset()
        outs = []
        for k, v, q in s["parts"]:
            c.update(k, v, 0)
            outs.append(c.prefill_attention(0, q))
        return outs, [c._k_codes[0][:, :, :n], c._v_codes[0][:, :, :n], c._k_norms[0][:, :, :n],
                      c._v_norms[0][:, :, :n], c._k_hot[0], c._v_hot[0]]
    if kind == "attn":
        from leankv_amd import kernels

        return kernels.tq_decode_attn(s["q"], s["k_codes"], s["k_norms"], s["v_codes"], s["v_norms"], s["k_hot"],
                                      s["v_hot"], s["PiK"], s["PiV"], s["cent"], s["bits"], s["len"], s["max_len"])
    return s["cache"].decode_attention(0, s["q"])


# ------------------------------------------------------------------------------------------------ work and tolerance
def _row_bytes(bits):
    return {1: 16, 2: 32, 3: 64, 4: 64}[bits]


def work(case):
    kind = case["kind"]
    if kind in ("proj", "mlp"):
        z, rows = case["hidden"], case["rows"]
        shapes = ([(case["heads"] * D, z), (case["kv"] * D, z), (case["kv"] * D, z), (z, case["heads"] * D)]
                  if kind == "proj" else [(case["ffn"], z), (case["ffn"], z), (z, case["ffn"])])
        keep = 1 - case["sparsity"] if rows == 1 else 1.0
        w = sum(n * zz for n, zz in shapes) * keep
        io = sum(n + zz for n, zz in shapes) * rows
        return {"bytes": 2 * w + 2 * io, "flops": 2 * w * rows}
    if kind == "quantize":
        m, e = 2 * case["vectors"], 2 if case["half"] else 4
        return {"bytes": m * (D * e + _row_bytes(case["bits"]) + e), "flops": m * 2 * D * D}
    if kind == "step":
        rows, keep = case["rows"], 1 - case["sparsity"] if case["rows"] == 1 else 1.0
        w = case["layers"] * sum(n * z for n, z in _SHAPES.values()) * keep + _VOCAB * _HIDDEN
        kvb = case["layers"] * rows * _KV * 2 * (max(0, case["length"] - case["hot"]) * (_row_bytes(case["bits"]) + 4)
                                                 + min(case["length"], case["hot"]) * 2 * D)
        att = case["layers"] * rows * _HEADS * case["length"] * 4 * D
        return {"bytes": 2 * w + kvb + 2 * rows * (_VOCAB + _HIDDEN), "flops": 2 * w * rows + att}
    B, kv, n, hot, rb = case["batch"], case["kv"], case["length"], case["hot"], _row_bytes(case["bits"])
    cold = max(0, n - hot)
    store = 2 * B * kv * (cold * (rb + 4) + min(n, hot) * 2 * D)
    if kind == "readback":
        return {"bytes": store + 2 * B * kv * n * D * 2, "flops": 2 * B * kv * cold * 2 * D * D}
    heads = case["heads"]
    if kind == "prefill":
        pairs = B * heads * n * (n + 1) // 2
        return {"bytes": 2 * B * kv * n * D * 2 + store + 2 * B * heads * n * D * 2,
                "flops": pairs * 4 * D + 2 * B * kv * cold * 2 * D * D}
    if kind == "paged":  # lengths spread from an eighth to the whole
        n = n * (1 + (B - 1) * 0.5625) / B
        store = 2 * B * kv * (max(0.0, n - hot) * (rb + 4) + min(n, hot) * 2 * D)
    return {"bytes": store + 2 * B * heads * D * 2, "flops": B * heads * n * 4 * D}


def tolerance(case):
    """About four times the distance of today's fp16 results from 64 bits; codes and copies are whole and equal.
    A step adds what its layers pass on, and the sparse rows what one value over or under its threshold changes."""
    kind = case["kind"]
    if kind == "step":
        return {"rel": 0.02}
    if kind == "mlp" and case["rows"] == 1:
        return {"rel": 8e-3}
    return {"rel": {"proj": 1e-3, "quantize": 1e-3, "readback": 1.5e-3, "mlp": 2e-3}.get(kind, 5e-3)}


# -------------------------------------------------------------------------------------------------------------- exact
def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        return _exact_step(case, seed)
    if kind == "proj":
        i = _proj_inputs(case, seed)
        outs = [_sparse64(i["x"], i[w], i["t"]) for w in ("wq", "wk", "wv")] + [_sparse64(i["a"], i["wo"], i["ta"])]
        return outs if case["rows"] > 1 else [o.view(-1) for o in outs[:3]] + [outs[3].view(1, 1, -1)]
    if kind == "mlp":
        i = _mlp_inputs(case, seed)
        h = _silu64(_sparse64(i["x"], i["wg"], i["t"])) * _sparse64(i["x"], i["wu"], i["t"])
        y = _sparse64(h, i["wd"], i["ta"])
        return (h, y) if case["rows"] > 1 else (h.view(1, 1, -1), y.view(1, 1, -1))
    if kind == "quantize":
        dt = torch.float16 if case["half"] else torch.float32
        k, v = (_kv((case["vectors"], D), seed, j).to(dt).double() for j in (1, 2))
        return None, k.norm(dim=-1), None, v.norm(dim=-1)
    hot, bits = case["hot"], case["bits"]
    if kind in ("readback", "prefill"):
        shape = (case["batch"], case["kv"], case["length"], D)
        k, v = _kv(shape, seed, 1), _kv(shape, seed, 2)
        pk, pv = _rotation(42), _rotation(43)
        if kind == "readback":
            return _stored64(k, pk, bits, hot), _stored64(v, pv, bits, hot)
        outs, at = [], 0
        for i, e in enumerate(_chunk_ends(case)):
            q = _randn((case["batch"], case["heads"], e - at, D), seed, 20 + i)
            kk, vv = _stored64(k, pk, bits, hot, e), _stored64(v, pv, bits, hot, e)
            outs.append(torch.stack([_attend64(q[b], kk[b], vv[b], at) for b in range(case["batch"])]))
            at = e
        cold = max(0, case["length"] - hot)
        kn, vn = k[:, :, :cold].double().norm(dim=-1), v[:, :, :cold].double().norm(dim=-1)
        return outs, [None, None, kn, vn, None, None]
    if kind == "attn":
        c = _attn_cold(case, seed)
        q = _randn((case["batch"], case["heads"], D), seed, 3)
        cent = _centroids(bits).float().double().cuda()
        kk, vv = (torch.cat([(cent[c[nm]["codes"]] @ c[nm]["pi"].double().cuda()) * c[nm]["norms"].double().unsqueeze(-1),
                             c[nm]["hot"].double()], dim=2) for nm in "kv")
        n = case["length"]
        return torch.stack([_attend64(q[b].unsqueeze(1), kk[b], vv[b], n).squeeze(1) for b in range(case["batch"])])
    lens = _paged_lengths(case, seed)
    q = _randn((len(lens), case["heads"], D), seed, 3)
    pk, pv = _rotation(42), _rotation(43)
    outs = []
    for b, n in enumerate(lens):
        k, v = _paged_kv(case, seed, b, n)
        outs.append(_attend64(q[b].unsqueeze(1), _stored64(k, pk, bits, hot), _stored64(v, pv, bits, hot), n).squeeze(1))
    return torch.stack(outs)
