"""The performance cases of this framework: what a program that uses it asks of it, at the sizes it meets.

A case is a dict with a "kind" and the sizes of one call:

  oil8       mth.oil8_gemv          one OIL8 projection of `batch` FP32 token rows (decode, small serving batches, prompts)
  oil4       mth.oil4_gemv          one OIL4 projection (codebooks per 128 or 64 weights, or one per tensor)
  prefill    mth.oil4_gemm_prefill  one OIL4 projection of a bf16 prompt
  ternary    mth.i2s_gemv_f32       one I2_S projection of FP32 token rows, quantised to int8 per token
  ternary_i8 mth.i2s_gemv           the same on activations that are int8 already
  i2s_gemm   mth.i2s_gemm           the ternary matrix product on FP32 activations (no quantisation)
  attention  mth.attention_decode   one decode step's attention over an FP32 KV cache
  decode     Decoder.step           teacher-forced decode steps of a whole decoder, then the logits
  prompt     Decoder.prefill        a prompt as one forward pass of a whole decoder, then the logits

The decoder has the widths of the 32-layer configuration (synth.DECODER_CONFIG5) and fewer layers, so that its weights can
be made from a seed in about a second.  Its steps are teacher-forced (the prompt is the sequence), so that a near tie of two
logits cannot change what the next step reads; its down projections' scale is divided by a power of two, as the decoder
tests do it, so that one int8 activation that rounds the other way stays below the differences of FP32 summation order
(divided by 128, such a step moves the logits by 3e-6).
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mythos.cpp_amd"))

import decoder  # noqa: E402
import mythos_oil as mth  # noqa: E402
import synth  # noqa: E402

DEV = "cuda"
DOWN_DIV = 512.0


def listed():
    return [
        # the smallest call: one attention projection of one token (hidden 4096)
        dict(name="oil8_4096_b1", kind="oil8", M=4096, K=4096, batch=1),
        # a down projection kept in OIL8: rows longer than the hidden size (ffn 11008)
        dict(name="oil8_down_b1", kind="oil8", M=4096, K=11008, batch=1),
        # continuous batching: more tokens than one decode group, fewer than a prompt, rows not a multiple of a tile
        dict(name="oil8_b40_ragged", kind="oil8", M=4000, K=4096, batch=40),
        # an MLP up projection of one token
        dict(name="oil4_up_b1", kind="oil4", M=11008, K=4096, batch=1, cb_block=128),
        # gate and up of a full decode group
        dict(name="oil4_gate_up_b16", kind="oil4", M=22016, K=4096, batch=16, cb_block=128),
        # prompt processing in bf16, compute-bound
        dict(name="oil4_prefill_512", kind="prefill", M=512, N=14336, K=4096, cb_block=128),
        # the ternary down projection of a full decode group, from FP32 activations
        dict(name="ternary_down_b16", kind="ternary", M=4096, K=11008, batch=16),
        # the ternary matrix product on FP32 activations, an odd number of tokens
        dict(name="i2s_gemm_300", kind="i2s_gemm", M=4096, N=300, K=4096),
        # decode attention over a long context, grouped-query heads
        dict(name="attention_6000", kind="attention", batch=2, heads=32, kv_heads=8, head_dim=128, ctx=6000, max_seq=8192),
        # one user's decode, a full group's decode, and a long prompt
        dict(name="decode_b1", kind="decode", hidden=4096, heads=32, kv_heads=32, head_dim=128, ffn=11008, layers=4,
             batch=1, length=256, kv="f32"),
        dict(name="decode_b16", kind="decode", hidden=4096, heads=32, kv_heads=32, head_dim=128, ffn=11008, layers=4,
             batch=16, length=128, kv="bf16"),
        dict(name="prompt_1500", kind="prompt", hidden=4096, heads=32, kv_heads=32, head_dim=128, ffn=11008, layers=4,
             batch=1, length=1500, kv="f32"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _dim(rng, lo, hi, steps):
    """A size between lo and hi (spread over its logarithm), a multiple of one of `steps`."""
    s = rng.choice(steps)
    return max(s, _log(rng, lo, hi) // s * s)


def _batch(rng, most=512):
    """One token, a decode group, or a serving batch / prompt of any size."""
    return rng.choice([1, rng.randint(2, 16), _log(rng, 17, most)])


def draw(rng):
    kind = rng.choice(["oil8", "oil8", "oil4", "oil4", "prefill", "ternary", "ternary_i8", "i2s_gemm", "attention",
                       "attention", "decode", "prompt"])
    if kind == "oil8":
        return dict(kind=kind, M=_dim(rng, 512, 32000, [64, 16, 1]), K=_dim(rng, 512, 14336, [256, 128, 16]),
                    batch=_batch(rng))
    if kind == "oil4":
        cb = rng.choice([128, 128, 128, 64, 0])
        return dict(kind=kind, M=_dim(rng, 512, 28672, [64, 16, 1]), K=_dim(rng, 512, 14336, [512, 256, 128]),
                    batch=_batch(rng), cb_block=cb)
    if kind == "prefill":
        return dict(kind=kind, M=_log(rng, 100, 2048), N=_dim(rng, 1024, 28672, [128, 64, 16]),
                    K=_dim(rng, 1024, 14336, [512, 256, 128]), cb_block=128)
    if kind in ("ternary", "ternary_i8"):
        return dict(kind=kind, M=_dim(rng, 512, 14336, [64, 16, 1]), K=_dim(rng, 512, 14336, [256, 64, 4]),
                    batch=_batch(rng))
    if kind == "i2s_gemm":
        return dict(kind=kind, M=_dim(rng, 512, 11008, [64, 16, 1]), N=_log(rng, 1, 512),
                    K=_dim(rng, 512, 11008, [256, 64, 4]))
    if kind == "attention":
        heads = rng.choice([8, 16, 32, 40])
        ctx = _log(rng, 16, 12000)
        D = rng.choice([64, 128, 128, 256])
        batch = rng.choice([1, 1, rng.randint(2, 16)])
        kvh = heads // rng.choice([1, 2, 4, 8])
        while batch > 1 and batch * kvh * ctx * D * 8 > (1 << 30):  # a cache of at most 1 GiB
            batch //= 2
        return dict(kind=kind, batch=batch, heads=heads, kv_heads=kvh, head_dim=D, ctx=ctx,
                    max_seq=min(16384, ctx + rng.randint(0, ctx)))
    hidden = rng.choice([1024, 2048, 4096])
    D = rng.choice([64, 128])
    heads = hidden // D
    batch = rng.choice([1, rng.randint(2, 16)])
    most = 400 if kind == "decode" else 2000 // batch if batch <= 16 else 100
    return dict(kind=kind, hidden=hidden, heads=heads, kv_heads=heads // rng.choice([1, 4]), head_dim=D,
                ffn=_dim(rng, 2 * hidden, 11008, [256, 64]), layers=rng.choice([2, 3]), batch=batch,
                length=_log(rng, 24, max(25, most)), kv=rng.choice(["f32", "bf16"]))


# ---- inputs ------------------------------------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) + 0x5EED)


def _bytes(g, rows, cols):
    return torch.randint(0, 256, (rows, cols), generator=g, device=DEV, dtype=torch.uint8)


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32) * std


def _codebook8(g):
    return torch.sort(_normal(g, 256, std=0.02)).values


def _codebooks4(g, n):
    """n codebooks of 16 FP16 entries, as bits."""
    return _normal(g, n * 16, std=0.02).half().view(torch.int16)


def _ternary(g, rows, cols):
    """[rows][cols / 4] packed codes t + 1, t uniform in {-1, 0, 1}."""
    c = torch.randint(0, 3, (rows, cols // 4, 4), generator=g, device=DEV, dtype=torch.uint8)
    return c[..., 0] | (c[..., 1] << 2) | (c[..., 2] << 4) | (c[..., 3] << 6)


def _model(case, g):
    """A decoder's weights in synth.decoder_model's layout, drawn on the GPU."""
    cfg = synth.decoder_config(hidden=case["hidden"], heads=case["heads"], kv_heads=case["kv_heads"],
                               head_dim=case["head_dim"], ffn=case["ffn"], layers=case["layers"],
                               max_seq=case["length"] + 8)
    H, F, V, B = cfg["hidden"], cfg["ffn"], cfg["vocab"], cfg["cb_block"]
    QD, KD = cfg["heads"] * cfg["head_dim"], cfg["kv_heads"] * cfg["head_dim"]

    def host(t):
        return t.cpu().numpy()

    model = {"emb": host(_normal(g, V, H)), "layers": []}
    for _ in range(cfg["layers"]):
        ly = {"attn_norm": host(1 + _normal(g, H, std=0.1)), "ffn_norm": host(1 + _normal(g, H, std=0.1))}
        for name, rows, cols in (("q", QD, H), ("k", KD, H), ("v", KD, H), ("o", H, QD)):
            ly["w" + name], ly["cb" + name] = host(_bytes(g, rows, cols)), host(_codebook8(g))
        ly["wgate_up"] = host(_bytes(g, 2 * F, H // 2))
        ly["cbgate_up"] = host(_codebooks4(g, 2 * F * (H // B))).view(np.uint16)
        ly["wdown"] = host(_ternary(g, H, F))
        ly["down_scale"] = np.float32(synth.W_SCALE_TERNARY / DOWN_DIV)
        model["layers"].append(ly)
    model["final_norm"] = host(1 + _normal(g, H, std=0.1))
    model["lm_idx"], model["lm_cb"] = host(_bytes(g, V, H)), host(_codebook8(g))
    prompts = torch.randint(0, V, (case["batch"], case["length"]), generator=g, device=DEV, dtype=torch.int32)
    return cfg, model, host(prompts)


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    s = {"case": case}
    if kind in ("oil8", "oil4", "ternary", "ternary_i8"):
        M, K, b = case["M"], case["K"], case["batch"]
        s["y"] = torch.empty(b, M, device=DEV)
        if kind == "oil8":
            s["w"], s["cb"], s["x"] = _bytes(g, M, K), _codebook8(g), _normal(g, b, K)
        elif kind == "oil4":
            blk = case["cb_block"]
            s["w"], s["cb"] = _bytes(g, M, K // 2), _codebooks4(g, M * (K // blk) if blk else 1)
            s["x"] = _normal(g, b, K)
        elif kind == "ternary":
            s["w"], s["x"] = _ternary(g, M, K), _normal(g, b, K)
        else:
            s["w"] = _ternary(g, M, K)
            s["x"] = torch.randint(-127, 128, (b, K), generator=g, device=DEV, dtype=torch.int8)
            s["scale"] = 0.02 + 0.01 * torch.rand(b, generator=g, device=DEV)
    elif kind == "prefill":
        M, N, K, blk = case["M"], case["N"], case["K"], case["cb_block"]
        s["x"] = _normal(g, M, K).bfloat16()
        s["w"], s["cb"] = _bytes(g, N, K // 2), _codebooks4(g, N * (K // blk))
        s["y"] = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
    elif kind == "i2s_gemm":
        M, N, K = case["M"], case["N"], case["K"]
        s["w"], s["x"], s["y"] = _ternary(g, M, K), _normal(g, N, K), torch.empty(M, N, device=DEV)
    elif kind == "attention":
        b, h, kvh, D, S = (case[k] for k in ("batch", "heads", "kv_heads", "head_dim", "max_seq"))
        s["q"], s["k"], s["v"] = _normal(g, b, h, D), _normal(g, b, kvh, S, D), _normal(g, b, kvh, S, D)
        s["y"] = torch.empty(b, h, D, device=DEV)
    else:
        cfg, model, s["prompts"] = _model(case, g)
        s["dec"] = decoder.Decoder(cfg, max_batch=case["batch"], kv_dtype=case["kv"])
        s["dec"].load(model)
    return s


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "oil8":
        mth.oil8_gemv(s["w"], s["cb"], s["x"], s["y"], c["M"], c["K"], c["batch"])
    elif kind == "oil4":
        mth.oil4_gemv(s["w"], s["cb"], c["cb_block"], s["x"], s["y"], c["M"], c["K"], c["batch"])
    elif kind == "prefill":
        mth.oil4_gemm_prefill(s["x"], s["w"], s["cb"], c["cb_block"], s["y"], c["M"], c["N"], c["K"])
    elif kind == "ternary":
        mth.i2s_gemv_f32(s["w"], synth.W_SCALE_TERNARY, s["x"], s["y"], c["M"], c["K"], c["batch"])
    elif kind == "ternary_i8":
        mth.i2s_gemv(s["w"], synth.W_SCALE_TERNARY, s["x"], s["scale"], s["y"], c["M"], c["K"], c["batch"])
    elif kind == "i2s_gemm":
        mth.i2s_gemm(s["w"], s["x"], s["y"], c["M"], c["N"], c["K"])
    elif kind == "attention":
        mth.attention_decode(s["q"], s["k"], s["v"], s["y"], c["batch"], c["heads"], c["kv_heads"], c["head_dim"],
                             c["ctx"], c["max_seq"])
    else:
        dec = s["dec"]
        dec.start(s["prompts"])
        if kind == "decode":
            dec.step(c["length"])
        else:
            dec.prefill()
        return dec.logits()
    return s["y"]


# ---- what a pass cannot do without -------------------------------------------------------------------------------------
def work(case):
    c, kind = case, case["kind"]
    if kind == "oil8":
        M, K, b = c["M"], c["K"], c["batch"]
        return dict(bytes=M * K + 1024 + 4 * b * (K + M), flops=2 * M * K * b)
    if kind == "oil4":
        M, K, b = c["M"], c["K"], c["batch"]
        cb = 32 * (M * (K // c["cb_block"]) if c["cb_block"] else 1)
        return dict(bytes=M * K // 2 + cb + 4 * b * (K + M), flops=2 * M * K * b)
    if kind == "prefill":
        M, N, K = c["M"], c["N"], c["K"]
        return dict(bytes=2 * M * (K + N) + N * K // 2 + 32 * N * (K // c["cb_block"]), flops=2 * M * N * K)
    if kind in ("ternary", "ternary_i8"):
        M, K, b = c["M"], c["K"], c["batch"]
        act = 4 * K if kind == "ternary" else K + 4
        return dict(bytes=M * K // 4 + b * (act + 4 * M), flops=2 * M * K * b)
    if kind == "i2s_gemm":
        M, N, K = c["M"], c["N"], c["K"]
        return dict(bytes=M * K // 4 + 4 * N * (K + M), flops=2 * M * N * K)
    if kind == "attention":
        b, h, kvh, D, ctx = (c[k] for k in ("batch", "heads", "kv_heads", "head_dim", "ctx"))
        return dict(bytes=8 * b * kvh * ctx * D + 8 * b * h * D, flops=4 * b * h * ctx * D)
    H, F, V, L, b, n = c["hidden"], c["ffn"], 32000, c["layers"], c["batch"], c["length"]
    QD, KD = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    layer = H * (QD + 2 * KD) + QD * H + 2 * F * H // 2 + 2 * F * (H // 128) * 32 + H * F // 4 + 8 * H + 4096
    weights, params = L * layer + V * H, L * (2 * H * QD + 2 * H * KD + 3 * F * H)
    e = 2 if c["kv"] == "bf16" else 4
    rows = n * (n + 1) // 2  # positions attended to by one sequence
    attn = 4 * L * b * rows * QD
    if kind == "decode":
        return dict(bytes=n * weights + 2 * L * b * KD * e * rows + 4 * b * V,
                    flops=2 * b * n * (params + V * H) + attn)
    return dict(bytes=weights + 4 * b * n * H + 2 * L * b * KD * e * n + 4 * b * V,
                flops=2 * b * n * params + 2 * b * V * H + attn)


def tolerance(case):
    kind = case["kind"]
    if kind in ("ternary", "ternary_i8"):
        return "exact"  # integer sums, one rounding order in the epilogue
    if kind == "prefill":
        return {"rel": 7e-3}  # bf16 outputs: 1.7e-3 from 64 bits
    if kind == "attention":
        return {"rel": 1.2e-6}  # up to 2.8e-7 from 64 bits
    if kind in ("decode", "prompt"):
        # FP32 throughout (up to 5e-5 from 64 bits: the softmax of large scores widens the sums' rounding); with a bf16
        # cache, K and V elements that round the other way (the prompt as one pass against its steps: up to 9e-4)
        return {"rel": 1e-4 if case["kv"] == "f32" else 4e-3}
    return {"rel": 2e-6}  # FP32 sums in another order: up to 4.2e-7 from 64 bits


# ---- the same in 64 bits -----------------------------------------------------------------------------------------------
def _w4(w, cb, rows, K, blk):
    """[rows][K] float64 weights of OIL4 nibbles and codebooks."""
    nib = torch.stack([w & 0xF, w >> 4], -1).reshape(rows, K).long()
    t = cb.view(torch.float16).double()
    if not blk:
        return t[nib]
    first = torch.arange(rows, device=DEV)[:, None] * (K // blk) + torch.arange(K, device=DEV)[None, :] // blk
    return t[first * 16 + nib]


def _w2(w, rows, K):
    """[rows][K] float64 ternary weights."""
    c = torch.stack([(w >> (2 * i)) & 3 for i in range(4)], -1).reshape(rows, K)
    return c.clamp(max=2).double() - 1


def _by_rows(rows, K, fn):
    """fn(first, last) over groups of weight rows whose float64 copies stay below 1 GiB, joined along dim 1."""
    n = max(1, (1 << 27) // K)
    return torch.cat([fn(i, min(rows, i + n)) for i in range(0, rows, n)], 1)


def _quant(x):
    """quantize_per_token: the int8 values (as float64) and 1 / scale, with the FP32 scale that defines them."""
    mx = x.abs().amax(-1, keepdim=True).float().clamp(min=1e-10)
    v = (x.float() * (127.0 / mx)).double()
    return torch.sign(v) * torch.floor(v.abs() + 0.5), mx.double() / 127.0


def _norm(x, gamma, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * gamma


def _attend(q, k, v, heads, kv_heads):
    """Causal attention of [n][heads][D] over [n][kv_heads][D]: head h reads kv head h % kv_heads."""
    n, D = q.shape[0], q.shape[2]
    out = torch.empty_like(q)
    mask = torch.ones(n, n, device=DEV, dtype=torch.bool).triu(1)
    for h in range(heads):
        s = (q[:, h] @ k[:, h % kv_heads].T.contiguous()) / math.sqrt(D)
        out[:, h] = torch.softmax(s.masked_fill(mask, -math.inf), -1) @ v[:, h % kv_heads]
    return out


def _forward(case, seed):
    """Logits of every sequence's last position, every position at once in float64."""
    cfg, model, prompts = _model(case, _gen(seed))
    H, F, D, heads, kvh = cfg["hidden"], cfg["ffn"], cfg["head_dim"], cfg["heads"], cfg["kv_heads"]

    def dev(a):
        return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)

    cos, sin = (dev(t[:case["length"]]).double() for t in mth.rope_tables(D, cfg["max_seq"], cfg["theta"]))

    def rope(x):
        a, b = x[..., :D // 2], x[..., D // 2:]
        return torch.cat([a * cos[:, None] - b * sin[:, None], a * sin[:, None] + b * cos[:, None]], -1)

    seqs = [dev(model["emb"])[dev(prompts[i]).long()].double() for i in range(case["batch"])]
    for ly in model["layers"]:
        w = {n: dev(ly["cb" + n]).double()[dev(ly["w" + n]).long()] for n in "qkvo"}
        gu = _w4(dev(ly["wgate_up"]), dev(ly["cbgate_up"].view(np.int16)), 2 * F, H, cfg["cb_block"])
        down = _w2(dev(ly["wdown"]), H, F)
        for i, x in enumerate(seqs):
            h = _norm(x, dev(ly["attn_norm"]).double(), cfg["eps"])
            q, k, v = ((h @ w[n].T.contiguous()).view(len(h), -1, D) for n in "qkv")
            x = x + _attend(rope(q), rope(k), v, heads, kvh).reshape(len(h), -1) @ w["o"].T.contiguous()
            h = _norm(x, dev(ly["ffn_norm"]).double(), cfg["eps"])
            y = h @ gu.T.contiguous()
            g, u = y[:, :F], y[:, F:]
            a, inv = _quant(g / (1 + torch.exp(-g)) * u)
            seqs[i] = x + a @ down.T.contiguous() * float(ly["down_scale"]) * inv
    last = torch.stack([x[-1] for x in seqs])
    h = _norm(last, dev(model["final_norm"]).double(), cfg["eps"])
    idx, cb = dev(model["lm_idx"]), dev(model["lm_cb"]).double()
    return _by_rows(cfg["vocab"], H, lambda i, j: h @ cb[idx[i:j].long()].T.contiguous())


def exact(case, seed):
    kind = case["kind"]
    if kind in ("decode", "prompt"):
        # a bf16 cache rounds K and V between the layers: the FP32 sums, not 64 bits, say which way a near tie goes
        return _forward(case, seed).cpu().numpy() if case["kv"] == "f32" else None
    s = prepare(case, seed)
    if kind == "attention":
        b, h, kvh, D, ctx = (case[k] for k in ("batch", "heads", "kv_heads", "head_dim", "ctx"))
        out = torch.empty(b, h, D, device=DEV, dtype=torch.float64)
        for i in range(b):
            for j in range(h):
                k, v = (s[n][i, j % kvh, :ctx].double() for n in "kv")
                out[i, j] = torch.softmax(k @ s["q"][i, j].double() / math.sqrt(D), 0) @ v
        return out
    if kind == "i2s_gemm":
        x = s["x"].double()
        return _by_rows(case["M"], case["K"],
                        lambda i, j: x @ _w2(s["w"][i:j], j - i, case["K"]).T.contiguous()).T.contiguous()
    if kind in ("ternary", "ternary_i8"):
        q, inv = _quant(s["x"]) if kind == "ternary" else (s["x"].double(), s["scale"].double()[:, None])
        ws = float(np.float32(synth.W_SCALE_TERNARY))
        return _by_rows(case["M"], case["K"],
                        lambda i, j: q @ _w2(s["w"][i:j], j - i, case["K"]).T.contiguous()) * ws * inv
    x = s["x"].double()
    if kind == "oil8":
        cb = s["cb"].double()
        return _by_rows(case["M"], case["K"], lambda i, j: x @ cb[s["w"][i:j].long()].T.contiguous())
    rows, blk = case["N"] if kind == "prefill" else case["M"], case["cb_block"]
    per = 16 * (case["K"] // blk) if blk else 0
    return _by_rows(rows, case["K"], lambda i, j: x @ _w4(s["w"][i:j], s["cb"][per * i:per * j] if blk else s["cb"],
                                                        j - i, case["K"], blk).T.contiguous())
