"""GPU parity of the token-batch routes that take any row length and row
count: activations converted once per call into the stream's workspace, then
a matrix-core kernel whose edges are padding.

Sizes sit where they can go wrong: one past and one short of a tile of rows or
tokens, row lengths with a partial last chunk, code rows that are not whole
16-byte pieces, K split over workgroups and not, the smallest of each range.
"""
import numpy as np
import pytest

import synth
from test_gpu_gemv import empty, to_dev

pytestmark = pytest.mark.gpu

WS = float(synth.W_SCALE_TERNARY)


def offset(t, shift):
    """t's bytes at an address `shift` bytes past an aligned one."""
    import torch
    raw = torch.empty(t.numel() * t.element_size() + 64, dtype=torch.uint8, device=t.device)
    part = raw[shift:shift + t.numel() * t.element_size()].view(t.dtype)
    return part.copy_(t.reshape(-1))


# ---------------------------------------------------------------- ternary --
@pytest.mark.parametrize("M,K,batch,shift", [
    (1, 64, 2, 0), (130, 256, 17, 0),          # smallest row; one chunk, one row tile + 2, one token group + 1
    (127, 1024, 64, 0), (129, 4416, 65, 0),    # token tile edges; 17.25 chunks, K split over workgroups
    (200, 2564, 16, 0), (64, 260, 5, 0),       # codes of 641 / 65 bytes per row: rows at every alignment
    (300, 1100, 40, 0), (65, 68, 33, 0),       # the same on the GEMM; one partial chunk
    (128, 512, 20, 4), (128, 512, 3, 4),       # codes and activations 4 bytes past an aligned address
    (96, 17000, 18, 0),                        # longer than the quantisation keeps in registers
])
def test_ternary_rows_bit_exact(M, K, batch, shift, oracle, mth, dev):
    """mth_i2s_gemv_f32 and mth_i2s_gemv: bit for bit the oracle's
    quantize_per_token + i2s_gemv per token (integer sums, one rounding order),
    rows of very different magnitudes and an all-zero row among them."""
    import torch
    print(f"ternary rows M={M} K={K} batch={batch} shift={shift}", flush=True)
    g = np.random.default_rng(M + K + batch)
    packed = g.integers(0, 256, (M, K // 4), dtype=np.uint8)      # all four codes
    x = (g.normal(0, 1, (batch, K)) * np.exp2(g.integers(-40, 40, batch))[:, None]).astype(np.float32)
    x[batch // 2] = 0.0
    p, xd = offset(to_dev(packed, dev), shift), offset(to_dev(x, dev), shift)
    y = empty(batch * M, torch.float32, dev)
    mth.i2s_gemv_f32(p, WS, xd, y, M, K, batch)
    torch.cuda.synchronize()
    assert np.array_equal(y.cpu().numpy().reshape(batch, M),
                          oracle.i2s_gemv_f32(packed.ravel(), WS, x, M, K, batch, threads=8))
    q = g.integers(-128, 128, (batch, K), dtype=np.int8)
    inv = g.uniform(0.001, 2.0, batch).astype(np.float32)
    mth.i2s_gemv(p, WS, offset(to_dev(q, dev), shift), to_dev(inv, dev), y, M, K, batch)
    torch.cuda.synchronize()
    got = y.cpu().numpy().reshape(batch, M)
    for t in range(batch):
        assert np.array_equal(got[t], oracle.i2s_gemv_rows(packed.ravel(), WS, q[t], inv[t], M, K, threads=8)), t


def test_ternary_rows_under_capture(oracle, mth, dev):
    """A capture on a stream that holds no workspace: the call takes the route
    that needs none, and every replay gives the oracle's bits."""
    import torch
    M, K, batch = 130, 1024, 20
    g = np.random.default_rng(3)
    packed = g.integers(0, 256, (M, K // 4), dtype=np.uint8)
    x = g.normal(0, 1, (batch, K)).astype(np.float32)
    p, xd, y = to_dev(packed, dev), to_dev(x, dev), empty(batch * M, torch.float32, dev)
    want = oracle.i2s_gemv_f32(packed.ravel(), WS, x, M, K, batch, threads=8)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    gr = torch.cuda.CUDAGraph()
    with torch.cuda.graph(gr, stream=s):
        mth.i2s_gemv_f32(p, WS, xd, y, M, K, batch)
    for rep in range(3):
        y.fill_(float("nan"))
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            gr.replay()
        torch.cuda.synchronize()
        assert np.array_equal(y.cpu().numpy().reshape(batch, M), want), rep


# -------------------------------------------------------------- attention --
@pytest.mark.parametrize("B,H,KVH,D,ctx,S", [
    (1, 8, 8, 128, 329, 400),        # shortest split context of 128, one head per workgroup, a slice of 9 rows
    (2, 32, 8, 128, 1025, 1500),     # 4 heads per workgroup, a slice of one row
    (1, 40, 5, 64, 2000, 2000),      # 8 heads per workgroup
    (3, 12, 4, 64, 777, 1024),       # a group of 3: one head per workgroup
    (2, 16, 1, 256, 400, 512),       # 16 heads of one kv head, two workgroup rows; D = 256
    (1, 4, 2, 64, 16384, 16384),     # the longest context: slices at their limit
    (16, 32, 2, 64, 1300, 1300),     # many workgroups, 16 rows per lane
])
def test_attention_split(B, H, KVH, D, ctx, S, mth, dev):
    """The context split over workgroups against float64: scores of a spread
    that leaves whole slices without weight, one row whose maximum sits in the
    last slice.  FP32 sums of ctx products: a few 1e-7 of the output's norm."""
    import torch
    print(f"attention split B={B} H={H} KVH={KVH} D={D} ctx={ctx}", flush=True)
    g = torch.Generator(device=dev).manual_seed(ctx + D)
    q = torch.randn(B, H, D, generator=g, device=dev) * 2
    kc, vc = (torch.randn(B, KVH, S, D, generator=g, device=dev) for _ in range(2))
    kc[0, 0, ctx - 1] = q[0, 0] * 0.5
    kc[:, :, ctx:], vc[:, :, ctx:] = float("nan"), float("nan")      # rows past the context are never used
    out = torch.full((B, H, D), float("nan"), device=dev)
    mth.attention_decode(q, kc, vc, out, B, H, KVH, D, ctx, S)
    torch.cuda.synchronize()
    want = torch.empty(B, H, D, dtype=torch.float64, device=dev)
    for b in range(B):
        for h in range(H):
            k, v = kc[b, h % KVH, :ctx].double(), vc[b, h % KVH, :ctx].double()
            p = torch.softmax((k @ q[b, h].double()) / D ** 0.5, 0)
            want[b, h] = p @ v
    rel = ((out.double() - want).norm(dim=-1) / want.norm(dim=-1)).max().item()
    assert rel <= 4e-6, rel


def test_attention_split_specials(mth, dev):
    """A slice whose scores are all -inf has no weight; a NaN in V reaches the
    output (0 * NaN), as in the undivided sum."""
    import torch
    B, H, D, ctx = 1, 8, 128, 2000
    g = torch.Generator(device=dev).manual_seed(5)
    q = torch.rand(B, H, D, generator=g, device=dev) + 0.1
    kc, vc = (torch.randn(B, H, ctx, D, generator=g, device=dev) for _ in range(2))
    kc[:, :, 256:1400] = float("-inf")
    vc[0, 3, 700, 5] = float("nan")
    out = torch.empty(B, H, D, device=dev)
    mth.attention_decode(q, kc, vc, out, B, H, H, D, ctx, ctx)
    keep = [i for i in range(ctx) if not 256 <= i < 1400]
    for h in range(H):
        p = torch.softmax((kc[0, h, keep].double() @ q[0, h].double()) / D ** 0.5, 0)
        want = p @ vc[0, h, keep].double()
        got = out[0, h].double()
        if h == 3:
            assert torch.isnan(got[5]) and torch.isnan(got).sum() == 1
            got[5] = want[5]
        assert ((got - want).norm() / want.norm()).item() <= 4e-6
