"""GPU parity of the prompt rows' attention (launch_attention_rows: the rows of
a chunk at positions p0 .., each attending causally to cache rows 0 .. its own)
against float64.

Sizes sit at the edges of its tiles: 64 query rows by 64 positions in halves of
32, both head dimensions, grouped KV heads, chunks that start inside a tile, and
values that the matrix-core path hands to its FP32 path (Inf, NaN, values that
round to Inf as bf16).
"""
import ctypes as C
import math

import pytest

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


def rows_attention(mth, q, k, v, np_, p0):
    """launch_attention_rows over q [B * np, H, D] and caches [B, KVH, S, D]."""
    import torch
    f = mth.lib._ZN3mth21launch_attention_rowsEPKfPKvS3_bPfliiiiiiP12ihipStream_t
    f.argtypes = [C.c_void_p] * 3 + [C.c_bool, C.c_void_p, C.c_int64] + [C.c_int] * 6 + [C.c_void_p]
    f.restype = C.c_int
    rows, H, D = q.shape
    B, KVH, S, _ = k.shape
    assert rows == B * np_ and p0 + np_ <= S and v.shape == k.shape
    out = torch.full_like(q, float("nan"))
    assert f(q.data_ptr(), k.data_ptr(), v.data_ptr(), k.dtype == torch.bfloat16, out.data_ptr(), rows, np_, p0, H,
             KVH, D, S, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    return out


def reference(q, k, v, np_, p0):
    """(attention in float64, bound).  A score is a sum of D products, whose
    parts below 2^-24 of each are left out and whose FP32 sums round some 24
    times: off by less than 32 EPS sum |q k| scale, which moves a probability by
    twice that (numerator and sum); exp, the weighted sums of a tile and the
    rescaling of earlier tiles round some 32 and 4 times more per tile."""
    import torch
    rows, H, D = q.shape
    ctx, KVH = p0 + np_, k.shape[1]
    o = torch.empty(rows, H, D, dtype=torch.float64)
    tol = torch.empty_like(o)
    mask = torch.ones(np_, ctx, dtype=torch.bool).triu(p0 + 1)
    for b in range(k.shape[0]):
        for h in range(H):
            qq, kk, vv = q[b * np_:(b + 1) * np_, h].double(), k[b, h % KVH, :ctx].double(), v[b, h % KVH, :ctx].double()
            p = torch.softmax((qq @ kk.T / math.sqrt(D)).masked_fill(mask, -math.inf), -1)
            o[b * np_:(b + 1) * np_, h] = p @ vv
            s = (qq.abs() @ kk.abs().T / math.sqrt(D)).amax(-1, keepdim=True)
            tol[b * np_:(b + 1) * np_, h] = (p @ vv.abs()) * EPS * (64 * s + 32 + 4 * math.ceil(ctx / 64))
    return o, tol


def inputs(B, np_, p0, H, KVH, D, kv, seed):
    import torch
    g = torch.Generator().manual_seed(seed)
    S = p0 + np_ + 3
    q = torch.randn(B * np_, H, D, generator=g) * 2.0
    k, v = (torch.randn(B, KVH, S, D, generator=g) for _ in range(2))
    k, v = k * 1.5, v * torch.exp2(torch.randint(-20, 20, (1, 1, 1, D), generator=g).float())
    if kv == "bf16":
        k, v = k.bfloat16(), v.bfloat16()
    k[:, :, p0 + np_:] = math.nan  # past the chunk: never read into a result
    v[:, :, p0 + np_:] = math.nan
    return q, k, v


@pytest.mark.parametrize("B,np_,p0,H,KVH,D,kv", [
    (1, 16, 0, 2, 2, 128, "f32"), (2, 17, 5, 4, 2, 64, "f32"), (3, 31, 1, 2, 1, 128, "bf16"),
    (1, 33, 31, 3, 3, 64, "bf16"), (1, 64, 64, 2, 2, 128, "f32"), (2, 65, 63, 4, 2, 128, "bf16"),
    (1, 127, 33, 2, 2, 64, "f32"), (1, 129, 500, 2, 1, 128, "f32"), (2, 200, 0, 4, 4, 128, "f32"),
])
def test_prompt_attention(B, np_, p0, H, KVH, D, kv, mth, dev):
    print(f"prompt attention B={B} np={np_} p0={p0} H={H} KVH={KVH} D={D} {kv}", flush=True)
    q, k, v = inputs(B, np_, p0, H, KVH, D, kv, np_ + p0)
    want, tol = reference(q, k, v, np_, p0)
    got = rows_attention(mth, q.to(dev), k.to(dev), v.to(dev), np_, p0).cpu().double()
    assert bool(((got - want).abs() <= tol).all()), ((got - want).abs() / tol).max().item()


@pytest.mark.parametrize("D,kv", [(128, "f32"), (64, "bf16")])
@pytest.mark.parametrize("value", [math.inf, math.nan, 3.4e38])
def test_prompt_attention_unsplittable(value, D, kv, mth, dev):
    """One such value of V at position 70 of 100: the rows before it are what
    they are without it; from it on its column is Inf, NaN or (the largest FP32
    values, which round to Inf as bf16) what float64 gives."""
    import torch
    print(f"prompt attention value={value} D={D} {kv}", flush=True)
    q, k, v = inputs(1, 100, 0, 2, 2, D, kv, 9)
    v[:, :, 70, 3] = value
    got = rows_attention(mth, q.to(dev), k.to(dev), v.to(dev), 100, 0).cpu().double()
    clean = v.clone()
    clean[:, :, 70, 3] = 0.0
    want, tol = reference(q, k, clean, 100, 0)
    rest = torch.ones_like(want, dtype=torch.bool)
    rest[70:, :, 3] = False
    assert bool(((got - want).abs() <= tol)[rest].all())
    if kv == "f32" and value == 3.4e38:
        want, tol = reference(q, k, v, 100, 0)
        assert bool(((got - want).abs() <= tol)[70:, :, 3].all())
    else:
        assert not bool(torch.isfinite(got[70:, :, 3]).any())
