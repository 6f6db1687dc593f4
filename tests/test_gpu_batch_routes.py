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


def test_attention_on_per_thread_streams(mth, dev):
    """hipStreamPerThread is one handle for a stream per thread: long-context
    attention of four threads at once on it, each on its own queries."""
    import threading
    import types
    import torch
    B, H, KVH, D, ctx, n, reps = 2, 32, 8, 128, 1500, 4, 20
    print("attention on per-thread streams", flush=True)
    g = torch.Generator(device=dev).manual_seed(9)
    q = torch.randn(n, B, H, D, generator=g, device=dev)
    kc, vc = (torch.randn(B, KVH, ctx, D, generator=g, device=dev) for _ in range(2))
    out = torch.full((n, reps, B, H, D), float("nan"), device=dev)
    torch.cuda.synchronize()
    errors = []

    def work(i):
        try:
            for r in range(reps):
                mth.attention_decode(q[i], kc, vc, out[i, r], B, H, KVH, D, ctx, ctx,
                                     stream=types.SimpleNamespace(cuda_stream=2))
        except Exception as e:
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(n)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors, errors
    k, v = (x.double()[:, torch.arange(H, device=dev) % KVH] for x in (kc, vc))
    for i in range(n):
        p = torch.softmax((k * q[i].double()[:, :, None, :]).sum(-1) / D ** 0.5, -1)
        want = (p[..., None] * v).sum(-2)
        assert bool(((out[i].double() - want).norm(dim=(-1, -2)) <= 4e-6 * want.norm(dim=(-1, -2))).all()), i


@pytest.mark.parametrize("what", ["attention", "i2s_gemm"])
def test_captured_calls_without_workspace(what, mth, dev):
    """Captured on a stream that already holds a workspace, these run on the kernels that use none: every replay, with
    eager calls of the workspace route on the same stream between them, gives the same bits."""
    import torch
    print(f"captured {what}", flush=True)
    g = torch.Generator(device=dev).manual_seed(4)
    s = torch.cuda.Stream()
    if what == "attention":
        B, H, KVH, D, ctx = 2, 32, 8, 128, 1500
        q = torch.randn(B, H, D, generator=g, device=dev)
        kc, vc = (torch.randn(B, KVH, ctx, D, generator=g, device=dev) for _ in range(2))
        eager, out = torch.empty(B, H, D, device=dev), torch.empty(B, H, D, device=dev)
        call = lambda o: mth.attention_decode(q, kc, vc, o, B, H, KVH, D, ctx, ctx)
    else:
        M, N, K = 300, 40, 4096
        w = torch.randint(0, 256, (M, K // 4), generator=g, device=dev, dtype=torch.uint8)
        x = torch.randn(N, K, generator=g, device=dev)
        eager, out = torch.empty(M, N, device=dev), torch.empty(M, N, device=dev)
        call = lambda o: mth.i2s_gemm(w, x, o, M, N, K)
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        call(eager)
    gr = torch.cuda.CUDAGraph()
    with torch.cuda.graph(gr, stream=s):
        call(out)
    first = None
    for rep in range(3):
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            call(eager)
            gr.replay()
            call(eager)
        torch.cuda.synchronize()
        assert float((out - eager).norm() / eager.norm()) <= 2e-6, rep
        first = out.clone() if first is None else first
        assert torch.equal(out, first), rep


# ----------------------------------------------------- token rows on MFMA --
def w64(kind, w, cb, M, K, blk, dev):
    """[M][K] float64 weights."""
    import torch
    w = torch.from_numpy(w).to(dev)
    if kind == "oil8":
        return torch.from_numpy(cb).to(dev).double()[w.long()]
    if kind == "oil4":
        t = torch.from_numpy(synth.dequant_oil4(w.cpu().numpy(), cb, M, K, blk)).to(dev)
        return t.double()
    return torch.from_numpy(synth.dequant_ternary(w.cpu().numpy(), M, K, 1.0)).to(dev).double()


def rows_inputs(kind, M, K, blk, g):
    if kind == "oil8":
        return g.integers(0, 256, (M, K), dtype=np.uint8), np.sort(g.normal(0, 0.02, 256)).astype(np.float32)
    if kind == "oil4":
        n = M * (K // blk) if blk else 1
        return g.integers(0, 256, (M, K // 2), dtype=np.uint8), g.normal(0, 0.02, n * 16).astype(np.float16).view(np.uint16)
    return g.integers(0, 256, (M, K // 4), dtype=np.uint8), None


def rows_call(kind, mth, w, cb, x, M, K, batch, blk, dev, shift=0):
    import torch
    y = empty(batch * M, torch.float32, dev)
    xd = offset(to_dev(x, dev), shift)
    if kind == "oil8":
        mth.oil8_gemv(to_dev(w, dev), to_dev(cb, dev), xd, y, M, K, batch)
    elif kind == "oil4":
        mth.oil4_gemv(to_dev(w, dev), to_dev(cb, dev), blk, xd, y, M, K, batch)
    else:
        mth.i2s_gemm(offset(to_dev(w, dev), shift), xd, y, M, batch, K)
    torch.cuda.synchronize()
    return y.reshape(batch, M) if kind != "tern" else y.reshape(M, batch).T.contiguous()


@pytest.mark.parametrize("kind,M,K,batch,blk,shift", [
    ("oil8", 5, 4112, 1, 0, 0),          # one token, one piece past 4096 columns (2 per lane), a row group of 1
    ("oil8", 130, 11008, 1, 0, 0),       # 3 pieces per lane, the last partial
    ("oil8", 64, 16384, 1, 0, 0),        # 4 pieces per lane, full
    ("oil8", 3, 16400, 1, 0, 0),         # one token, a row longer than that kernel takes
    ("oil4", 17, 640, 1, 128, 0),        # one token: 2 waves of 512 columns, the second a quarter full
    ("oil4", 33, 4224, 1, 128, 0),       # 9 waves
    ("oil4", 40, 8192, 1, 0, 0),         # 16 full waves of 2 phases, one codebook
    ("oil4", 31, 9088, 1, 128, 0),       # 9 waves of 4 phases, the last nearly full
    ("oil4", 16, 16384, 1, 128, 0),      # 16 waves of 4 phases
    ("oil8", 129, 2064, 17, 0, 0),       # 2 row tiles, 16.1 steps: a last step of one 16-byte piece
    ("oil8", 4000, 4096, 48, 0, 0),      # 3 token groups, K split 8 ways
    ("oil8", 127, 1280, 65, 0, 0),       # 2 token tiles of 48
    ("oil8", 300, 528, 40, 0, 4),        # x not 16-byte aligned
    ("oil8", 640, 17024, 20, 0, 0),      # rows longer than the conversion keeps in registers
    ("oil4", 100, 5120, 1, 64, 0),       # one token, codebooks per 64
    ("oil4", 130, 1120, 33, 32, 0),      # codebooks per 32, a last step of 96 columns
    ("oil4", 257, 3968, 64, 128, 0),
    ("oil4", 255, 9088, 18, 0, 0),       # one codebook per tensor, two steps past 8192
    ("oil4", 64, 640, 200, 64, 8),
    ("tern", 33, 4100, 1, 0, 0),         # rows of 1025 code bytes
    ("tern", 129, 1028, 40, 0, 0),
    ("tern", 4096, 512, 300, 0, 0),
    ("tern", 200, 2052, 64, 0, 4),
])
def test_token_rows(kind, M, K, batch, blk, shift, mth, dev):
    """Token rows of magnitudes 2^-40 .. 2^40 and an all-zero row against
    float64.  Bound: FP32 sums of K products in chunks of 32, so 1e-5 of
    sum |w x| per element and 1e-6 of the row's norm."""
    import torch
    print(f"token rows {kind} M={M} K={K} batch={batch} blk={blk} shift={shift}", flush=True)
    g = np.random.default_rng(M + K + batch)
    w, cb = rows_inputs(kind, M, K, blk, g)
    x = (g.normal(0, 1, (batch, K)) * np.exp2(g.integers(-40, 40, batch))[:, None]).astype(np.float32)
    if batch > 2:
        x[batch // 2] = 0.0
    got = rows_call(kind, mth, w, cb, x, M, K, batch, blk, dev, shift).double()
    W, X = w64(kind, w, cb, M, K, blk, dev), torch.from_numpy(x).to(dev).double()
    want, absw = X @ W.T.contiguous(), X.abs() @ W.abs().T.contiguous()
    assert bool(((got - want).abs() <= 1e-5 * absw + 1e-30).all())
    nrm = want.norm(dim=1)
    assert bool(((got - want).norm(dim=1) <= 1e-6 * nrm + 1e-30).all())


# whole rows in one slice, the longest chains of sums: 4080 .. 8192 columns, each token tile width
@pytest.mark.parametrize("kind,M,K,batch,blk", [("oil8", 12000, 4080, 200, 0), ("oil8", 33000, 6000, 16, 0),
                                                ("oil4", 12000, 4224, 200, 64), ("oil4", 12016, 2688, 140, 128),
                                                ("oil4", 33000, 8192, 17, 64), ("oil4", 16500, 4224, 96, 64),
                                                ("tern", 8000, 4096, 300, 0)])
def test_token_rows_error(kind, M, K, batch, blk, mth, dev):
    """The sums' error against float64, of normal values: FP32 FMAs in 64 lanes (the kernels that take these sizes one
    token after another) are 1.1e-7 .. 2.2e-7 of the norm off, one chain of all products 2.7e-7 .. 6e-7.  2^-22: a part
    pair's own rounding."""
    import torch
    print(f"token rows error {kind} M={M} K={K} batch={batch}", flush=True)
    g = np.random.default_rng(M + K)
    w, cb = rows_inputs(kind, M, K, blk, g)
    x = g.normal(0, 1, (batch, K)).astype(np.float32)
    got = rows_call(kind, mth, w, cb, x, M, K, batch, blk, dev).double()
    err = ref = 0.0
    X = torch.from_numpy(x).to(dev).double()
    step = 3000
    for i in range(0, M, step):
        n = min(M, i + step) - i
        c = cb if kind != "oil4" else cb[16 * (K // blk) * i:16 * (K // blk) * (i + n)]
        want = X @ w64(kind, w[i:i + n], c, n, K, blk, dev).T.contiguous()
        err += float((got[:, i:i + n] - want).square().sum())
        ref += float(want.square().sum())
    assert (err / ref) ** 0.5 <= 2.0 ** -22, (err / ref) ** 0.5


@pytest.mark.parametrize("kind", ["oil8", "oil4", "tern"])
@pytest.mark.parametrize("M,K,batch", [(300, 4096, 40), (40, 4736, 1)])
@pytest.mark.parametrize("what", ["x_inf", "x_nan", "codebook_inf"])
def test_token_rows_non_finite(kind, M, K, batch, what, mth, dev):
    """Inf and NaN reach the outputs the reference's products give them: a
    token's non-finite value its own outputs only, an infinite codebook entry
    the rows that use it; a ternary weight of 0 skips its activation."""
    import torch
    if kind == "tern" and what == "codebook_inf":
        pytest.skip("ternary weights have no codebook")
    blk = 128
    g = np.random.default_rng(11)
    w, cb = rows_inputs(kind, M, K, blk, g)
    x = g.normal(0, 1, (batch, K)).astype(np.float32)
    if what == "codebook_inf":
        if kind == "oil8":
            cb[7] = np.inf
            w[w == 7] = 8
            w[5, 100] = 7
        else:
            cb.reshape(M, K // blk, 16)[5, 3, 9] = 0x7C00
    else:
        x[batch // 2, 77] = np.inf if what == "x_inf" else np.nan
    got = rows_call(kind, mth, w, cb, x, M, K, batch, blk, dev).cpu().numpy()
    W = w64(kind, w, cb, M, K, blk, dev).cpu().numpy()
    with np.errstate(invalid="ignore"):
        prod = x[:, None, :].astype(np.float64) * W[None] if kind != "tern" else np.where(
            W[None] == 0, 0.0, x[:, None, :].astype(np.float64) * W[None])
        want = prod.sum(-1)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    assert np.array_equal(np.isinf(got), inf) and np.array_equal(got[inf], want[inf])
    fin = np.isfinite(want)
    if fin.any():
        assert np.abs(got[fin] - want[fin]).max() <= 1e-5 * np.abs(prod).sum(-1)[fin].max()


# one, two and four token groups; K split over workgroups and not; more than one token tile; a K remainder
@pytest.mark.parametrize("kind,M,K,batch,blk", [("oil8", 300, 1040, 12, 0), ("oil8", 200, 6448, 70, 0),
                                                ("oil4", 130, 1120, 33, 32), ("oil4", 1616, 1920, 200, 128),
                                                ("oil4", 500, 9088, 20, 64), ("tern", 300, 4100, 9, 0),
                                                ("tern", 4096, 1024, 130, 0), ("oil4", 500, 1664, 1, 128),
                                                ("oil4", 500, 9088, 1, 0)])
@pytest.mark.parametrize("span", [2.0 ** 20, 2.0 ** 27, 2.0 ** 40])
def test_token_rows_wide_range(kind, M, K, batch, blk, span, mth, dev):
    """Values far above the rest of their row that meet weights of 0 in half of the outputs: those keep the precision
    of the rest, as FP32 products do.  Other tokens of the tile are as without them, bit for bit."""
    import torch
    print(f"token rows wide range {kind} M={M} K={K} batch={batch} span={span}", flush=True)
    g = np.random.default_rng(M + K)
    w, cb = rows_inputs(kind, M, K, blk, g)
    per = {"oil8": 1, "oil4": 2, "tern": 4}[kind]
    cols, zero = np.array([0, K // 2, K - 1]), M // 2
    if kind == "oil8":
        cb[7] = 0.0
        w[:zero, cols] = 7
    elif kind == "oil4":
        cb.reshape(-1, 16)[:, 5] = 0
        for c in cols:
            w[:zero, c // 2] = (w[:zero, c // 2] & (0xF0 if c % 2 == 0 else 0x0F)) | (5 << (4 * (c % 2)))
    else:
        for c in cols:
            w[:zero, c // 4] = (w[:zero, c // 4] & ~np.uint8(3 << (2 * (c % 4)))) | (1 << (2 * (c % 4)))
    x = (1 + g.random((batch, K))).astype(np.float32) * g.choice([-1, 1], (batch, K)).astype(np.float32)
    plain = rows_call(kind, mth, w, cb, x, M, K, batch, blk, dev)
    wide = sorted({0, batch // 2, batch - 1})
    for t in wide:
        x[t, cols] *= span
    got = rows_call(kind, mth, w, cb, x, M, K, batch, blk, dev)
    rest = [t for t in range(batch) if t not in wide]
    assert torch.equal(got[rest], plain[rest])
    W, X = w64(kind, w, cb, M, K, blk, dev), torch.from_numpy(x).to(dev).double()
    want, absw = X @ W.T.contiguous(), X.abs() @ W.abs().T.contiguous()
    got = got.double()
    assert bool(((got - want).abs() <= 1e-5 * absw + 1e-30).all())
    err = (got - want)[wide][:, :zero].norm(dim=1) / want[wide][:, :zero].norm(dim=1)
    assert bool((err <= 1e-6).all()), err


@pytest.mark.parametrize("kind,M,K,batch,blk", [("oil8", 4000, 4080, 64, 0), ("oil8", 200, 6448, 70, 0),
                                                ("oil4", 12000, 4224, 200, 64), ("oil4", 500, 9088, 20, 64),
                                                ("tern", 4096, 4096, 100, 0)])
def test_token_rows_wide_range_elsewhere(kind, M, K, batch, blk, mth, dev):
    """Every token spans 40 binades, its small values beside large ones in every output: as close to float64 as without
    them (2^-22, test_token_rows_error), none of it summed in one chain."""
    import torch
    print(f"token rows wide range elsewhere {kind} M={M} K={K} batch={batch}", flush=True)
    g = np.random.default_rng(M + K)
    w, cb = rows_inputs(kind, M, K, blk, g)
    x = g.normal(0, 1, (batch, K)).astype(np.float32)
    x[:, ::7] *= np.float32(2.0 ** -40)
    got = rows_call(kind, mth, w, cb, x, M, K, batch, blk, dev).double()
    want = torch.from_numpy(x).to(dev).double() @ w64(kind, w, cb, M, K, blk, dev).T.contiguous()
    err = float((got - want).norm() / want.norm())
    assert err <= 2.0 ** -22, err


@pytest.mark.parametrize("M,K,batch", [(300, 1040, 12), (129, 6448, 70), (4000, 272, 40)])
def test_token_rows_wide_codebook(M, K, batch, mth, dev):
    """OIL8 codebook entries 2^-36 of the others: rows that hold those alone keep the precision of FP32 products."""
    import torch
    print(f"token rows wide codebook M={M} K={K} batch={batch}", flush=True)
    g = np.random.default_rng(K)
    w, cb = rows_inputs("oil8", M, K, 0, g)
    cb[:16] = (g.normal(0, 1, 16) * 2.0 ** -42).astype(np.float32)
    w[: M // 2] %= 16
    w[M // 2:] = np.maximum(w[M // 2:], 16)
    x = g.normal(0, 1, (batch, K)).astype(np.float32)
    got = rows_call("oil8", mth, w, cb, x, M, K, batch, 0, dev).double()
    want = torch.from_numpy(x).to(dev).double() @ w64("oil8", w, cb, M, K, 0, dev).T.contiguous()
    for rows in (slice(0, M // 2), slice(M // 2, M)):
        assert float((got[:, rows] - want[:, rows]).norm() / want[:, rows].norm()) <= 2.0 ** -22, rows


# one slice and several (two to eight), token tiles of 16 to 48, an odd row count
@pytest.mark.parametrize("M,K,batch", [(4000, 528, 18), (3001, 944, 49), (12000, 2064, 200), (4000, 4080, 64),
                                       (8000, 4080, 10)])
def test_token_rows_oil8_short_error(M, K, batch, mth, dev):
    """OIL8 rows of up to 4096 columns off the batched GEMV's shapes: no further from float64 than the kernel that takes
    one token after another in FP32 (0.96e-7 .. 1.1e-7 of the norm)."""
    import torch
    print(f"token rows OIL8 error M={M} K={K} batch={batch}", flush=True)
    g = np.random.default_rng(M + K)
    w, cb = rows_inputs("oil8", M, K, 0, g)
    x = g.normal(0, 1, (batch, K)).astype(np.float32)
    got = rows_call("oil8", mth, w, cb, x, M, K, batch, 0, dev).double()
    want = torch.from_numpy(x).to(dev).double() @ w64("oil8", w, cb, M, K, 0, dev).T.contiguous()
    err = float((got - want).norm() / want.norm())
    assert err <= 1.03e-7, err


@pytest.mark.parametrize("K,blk", [(640, 128), (1152, 128), (1664, 0), (3968, 128), (9088, 128)])
def test_one_token_error(K, blk, mth, dev):
    """One token's sums against float64: FP32 products in 64 lanes are 1.2e-7 (640 .. 1664 columns) .. 2.3e-7 (9088) of
    the norm off; parts of 22 bits (4e-8) in short sums stay below that."""
    import torch
    M = 8000
    print(f"one token error K={K} blk={blk}", flush=True)
    g = np.random.default_rng(K)
    w, cb = rows_inputs("oil4", M, K, blk, g)
    x = g.normal(0, 1, (1, K)).astype(np.float32)
    got = rows_call("oil4", mth, w, cb, x, M, K, 1, blk, dev).double()
    want = torch.from_numpy(x).to(dev).double() @ w64("oil4", w, cb, M, K, blk, dev).T.contiguous()
    assert float((got - want).norm() / want.norm()) <= 1.3e-7


@pytest.mark.parametrize("M,K,batch", [(4096, 4096, 512), (12288, 4096, 1024), (8192, 1024, 300)])
def test_prompt_gemm_oil8_error(M, K, batch, mth, dev):
    """The OIL8 prompt GEMM's sums against float64, tiles of 128 and of 256 rows.  An MFMA rounds its accumulator once
    per 8 columns, by 2.5e-8 of its size in the mean square, at sizes that grow to the full (half of it in the mean
    square); the parts' own rounding is 8e-8.  A tenth more for the sample."""
    import torch
    print(f"prompt GEMM error M={M} K={K} batch={batch}", flush=True)
    g = np.random.default_rng(K)
    w, cb = rows_inputs("oil8", M, K, 0, g)
    x = g.normal(0, 1, (batch, K)).astype(np.float32)
    got = rows_call("oil8", mth, w, cb, x, M, K, batch, 0, dev).double()
    want = torch.from_numpy(x).to(dev).double() @ w64("oil8", w, cb, M, K, 0, dev).T.contiguous()
    err = float((got - want).norm() / want.norm())
    assert err <= 1.1 * (K / 16 * 2.5e-8 ** 2 + 8e-8 ** 2) ** 0.5, err


# ------------------------------------------------ the row kernels by themselves --
# Sizes at their edges that the entry points' estimates give to other kernels: the launches called directly, in a
# workspace of exactly the size they ask for, with guards behind it and behind the output.
SYMS = {
    "ws": ("_ZN3mth25rows_mfma_workspace_bytesEllli", "llli"),
    "ws_bf16": ("_ZN3mth25rows_bf16_workspace_bytesElll", "lll"),
    "ws_i2s": ("_ZN3mth24i2s_rows_workspace_bytesElll", "lll"),
    "oil8": ("_ZN3mth16launch_oil8_rowsEPKNS_7Oil8SegEiPKfllbPvP12ihipStream_tb", "pipllbppb"),
    "oil4": ("_ZN3mth16launch_oil4_rowsEPKhPKtlPKfPflllbPvP12ihipStream_tb", "pplpplllbppb"),
    "oil4_bf16": ("_ZN3mth21launch_oil4_rows_bf16EPKhPKtlS3_PtlllPvP12ihipStream_t", "pplpplllpp"),
    "tern": ("_ZN3mth16launch_tern_rowsEPKhPKfPflllPvP12ihipStream_t", "ppplllpp"),
    "i2s": ("_ZN3mth15launch_i2s_rowsEPKhfPKfPKaS3_PflllPvP12ihipStream_t", "pfpppplllpp"),
}


def direct(mth, name, *args):
    import ctypes as C
    sym, sig = SYMS[name]
    f = getattr(mth.lib, sym)
    f.argtypes = [{"p": C.c_void_p, "l": C.c_int64, "i": C.c_int, "b": C.c_bool, "f": C.c_float}[c] for c in sig]
    f.restype = C.c_size_t if name.startswith("ws") else C.c_int
    return f(*args)


class Guarded:
    """Workspace and outputs with untouched bytes behind them (`ok`), on the current stream."""
    def __init__(self, dev, ws_bytes):
        import torch
        self.bufs = [(torch.full((ws_bytes + 1024,), 0xA5, dtype=torch.uint8, device=dev), ws_bytes)]
        self.ws, self.stream = self.bufs[0][0].data_ptr(), torch.cuda.current_stream().cuda_stream

    def out(self, n, dtype, dev):
        import torch
        size = n * torch.empty(0, dtype=dtype).element_size()
        t = torch.full((size + 1024,), 0xA5, dtype=torch.uint8, device=dev)
        self.bufs.append((t, size))
        return t[:size].view(dtype)

    def ok(self):
        import torch
        torch.cuda.synchronize()
        return all(bool((t[n:] == 0xA5).all()) for t, n in self.bufs)


def rows_close(got, want, absw):
    assert bool(((got.double() - want).abs() <= 1e-5 * absw + 1e-30).all())
    assert bool(((got.double() - want).norm(dim=1) <= 1e-6 * want.norm(dim=1) + 1e-30).all())


@pytest.mark.parametrize("kind,M,K,batch,blk,shift", [
    ("oil8", 1, 32, 1, 0, 0), ("oil8", 129, 2064, 17, 0, 0), ("oil8", 127, 144, 33, 0, 4),
    ("oil8", 257, 4096, 48, 0, 0), ("oil8", 256, 4080, 49, 0, 0), ("oil8", 130, 4112, 64, 0, 0),
    ("oil8", 33000, 272, 5, 0, 0),
    ("oil4", 1, 32, 1, 32, 0), ("oil4", 129, 544, 17, 32, 4), ("oil4", 130, 2080, 65, 0, 0),
    ("tern", 1, 32, 1, 0, 0), ("tern", 129, 1028, 40, 0, 0), ("tern", 33, 100, 17, 0, 4), ("tern", 200, 2052, 64, 0, 4),
])
def test_row_kernels_by_themselves(kind, M, K, batch, blk, shift, mth, dev):
    """As test_token_rows, on the row kernel whatever the estimates say; with and without the FP32 guard (for OIL8 rows
    of up to 4096 columns: its FINE kernels) and with a K split and without where the call chooses."""
    import torch
    g = np.random.default_rng(M + K + batch)
    w, cb = rows_inputs(kind, M, K, blk, g)
    x = (g.normal(0, 1, (batch, K)) * np.exp2(g.integers(-40, 40, batch))[:, None]).astype(np.float32)
    if batch > 2:
        x[batch // 2] = 0.0
    W, X = w64(kind, w, cb, M, K, blk, dev), torch.from_numpy(x).to(dev).double()
    want, absw = X @ W.T.contiguous(), X.abs() @ W.abs().T.contiguous()
    wd, xd = offset(to_dev(w, dev), shift if kind == "tern" else 0), offset(to_dev(x, dev), shift)
    cd = to_dev(cb, dev) if cb is not None else None
    for fp32 in ((False, True) if kind != "tern" else (True,)):
        for alone in ((False, True) if kind != "tern" else (False,)):
            print(f"row kernel {kind} M={M} K={K} batch={batch} blk={blk} fp32={fp32} alone={alone}", flush=True)
            b = Guarded(dev, direct(mth, "ws", M, K, batch, 1))
            y = b.out(batch * M, torch.float32, dev)
            if kind == "oil8":
                seg = np.array([wd.data_ptr(), cd.data_ptr(), y.data_ptr(), M], dtype=np.int64)
                rc = direct(mth, kind, seg.ctypes.data, 1, xd.data_ptr(), K, batch, fp32, b.ws, b.stream, alone)
            elif kind == "oil4":
                rc = direct(mth, kind, wd.data_ptr(), cd.data_ptr(), blk, xd.data_ptr(), y.data_ptr(), M, K, batch, fp32,
                            b.ws, b.stream, alone)
            else:
                rc = direct(mth, kind, wd.data_ptr(), xd.data_ptr(), y.data_ptr(), M, K, batch, b.ws, b.stream)
            assert rc == 0 and b.ok()
            rows_close(y.reshape(batch, M) if kind != "tern" else y.reshape(M, batch).T, want, absw)


# a K split and none, the FINE kernels and the others; an odd matrix (scalar stores and reduction) between even ones
@pytest.mark.parametrize("K,batch,fp32", [(1040, 20, True), (1040, 20, False), (4112, 33, True), (288, 50, True)])
def test_row_kernel_three_matrices(K, batch, fp32, mth, dev):
    import torch
    Ms = (5, 129, 256)
    print(f"row kernel, three matrices, K={K} batch={batch} fp32={fp32}", flush=True)
    g = np.random.default_rng(K)
    x = g.normal(0, 1, (batch, K)).astype(np.float32)
    x[0, :3] *= 2.0 ** 40
    xd = to_dev(x, dev)
    mats = [rows_inputs("oil8", M, K, 0, g) for M in Ms]
    on = [(to_dev(w, dev), to_dev(cb, dev)) for w, cb in mats]
    b = Guarded(dev, direct(mth, "ws", sum(Ms), K, batch, 3))
    ys = [b.out(batch * M, torch.float32, dev) for M in Ms]
    seg = np.array([[w.data_ptr(), cb.data_ptr(), y.data_ptr(), M] for (w, cb), y, M in zip(on, ys, Ms)], dtype=np.int64)
    assert direct(mth, "oil8", seg.ctypes.data, 3, xd.data_ptr(), K, batch, fp32, b.ws, b.stream, False) == 0 and b.ok()
    X = torch.from_numpy(x).to(dev).double()
    for (w, cb), y, M in zip(mats, ys, Ms):
        W = w64("oil8", w, cb, M, K, 0, dev)
        rows_close(y.reshape(batch, M), X @ W.T.contiguous(), X.abs() @ W.abs().T.contiguous())


# stores of whole pairs, of single values (odd rows) and of both (rows not a multiple of 4) in one slice, many
# workgroups; K split with an odd and an even count of outputs
@pytest.mark.parametrize("M,N,K,block", [(1, 1, 32, 32), (15, 127, 96, 32), (17, 129, 256, 128), (33, 130, 384, 128),
                                         (200, 4225, 992, 32), (3, 127, 512, 64), (200, 9000, 160, 32), (5, 132, 1056, 32)])
def test_row_kernel_bf16_by_itself(M, N, K, block, mth, dev):
    """As test_prefill_rows, on the row kernel whatever the estimates say."""
    import torch
    from test_gpu_prefill import check
    print(f"row kernel bf16 M={M} N={N} K={K} block={block}", flush=True)
    a, packed, cbs = synth.prefill(M, N, K, block)
    A = torch.from_numpy(synth.bf16_to_f32(a).reshape(M, K)) * torch.exp2(torch.arange(M) % 41 - 20.0)[:, None]
    x, w, cb = A.bfloat16().to(dev), to_dev(packed, dev), to_dev(cbs, dev)
    b = Guarded(dev, direct(mth, "ws_bf16", N, K, M))
    c = b.out(M * N, torch.bfloat16, dev)
    assert direct(mth, "oil4_bf16", w.data_ptr(), cb.data_ptr(), block, x.data_ptr(), c.data_ptr(), N, K, M, b.ws,
                  b.stream) == 0 and b.ok()
    W = synth.dequant_oil4(packed, cbs, N, K, block).astype(np.float64)
    A = A.bfloat16().double().numpy()
    check(c.view(torch.int16).cpu().numpy().view(np.uint16).reshape(M, N), A @ W.T, np.abs(A) @ np.abs(W).T, "rows")


@pytest.mark.parametrize("M,K,batch,shift", [(1, 64, 2, 0), (64, 260, 5, 0), (128, 512, 3, 4), (129, 1028, 16, 4),
                                             (33, 68, 17, 4)])
def test_ternary_rows_by_themselves(M, K, batch, shift, oracle, mth, dev):
    """As test_ternary_rows_bit_exact, on the padded rows whatever the estimates say."""
    import torch
    print(f"ternary rows by themselves M={M} K={K} batch={batch} shift={shift}", flush=True)
    g = np.random.default_rng(M + K + batch)
    packed = g.integers(0, 256, (M, K // 4), dtype=np.uint8)
    x = (g.normal(0, 1, (batch, K)) * np.exp2(g.integers(-40, 40, batch))[:, None]).astype(np.float32)
    q, inv = g.integers(-128, 128, (batch, K), dtype=np.int8), g.uniform(0.001, 2.0, batch).astype(np.float32)
    p, xd, qd = (offset(to_dev(t, dev), shift) for t in (packed, x, q))
    sc = to_dev(inv, dev)
    for f32 in (True, False):
        b = Guarded(dev, direct(mth, "ws_i2s", M, K, batch))
        y = b.out(batch * M, torch.float32, dev)
        assert direct(mth, "i2s", p.data_ptr(), WS, xd.data_ptr() if f32 else None, None if f32 else qd.data_ptr(),
                      None if f32 else sc.data_ptr(), y.data_ptr(), M, K, batch, b.ws, b.stream) == 0 and b.ok()
        want = (oracle.i2s_gemv_f32(packed.ravel(), WS, x, M, K, batch, threads=8) if f32 else
                np.stack([oracle.i2s_gemv_rows(packed.ravel(), WS, q[t], inv[t], M, K, threads=8) for t in range(batch)]))
        assert np.array_equal(y.cpu().numpy().reshape(batch, M), want), f32


# ----------------------------------------------------------------- argmax --
@pytest.mark.parametrize("rows,n", [(15, 2048), (16, 2049), (17, 5000), (33, 140001)])
def test_argmax_rows(rows, n, oracle, mth, dev):
    """A wave per row: one short of, exactly and one past a workgroup's 16 rows, and more partials than lanes."""
    import torch
    print(f"argmax rows={rows} n={n}", flush=True)
    g = np.random.default_rng(rows)
    x = g.integers(-50, 50, (rows, n)).astype(np.float32)   # many ties: the first index wins
    x[1] = -np.inf
    x[2] = np.nan
    x[3, n - 1] = 99.0
    ids = torch.full((rows,), -1, dtype=torch.int32, device=dev)
    mth.argmax(to_dev(x, dev), ids, rows, n)
    torch.cuda.synchronize()
    assert ids.cpu().tolist() == [oracle.argmax(r) for r in x]


# ---------------------------------------------------------- bf16 prompts --
# one token and one row; one past and one short of a 128 x 64 tile; odd row counts (2-byte aligned output rows); a last
# step of 32 and of 96 columns, codebooks per 32; K split over workgroups and not
@pytest.mark.parametrize("M,N,K,block", [(1, 1, 32, 32), (15, 127, 96, 32), (17, 129, 256, 64), (64, 128, 1120, 32),
                                         (65, 130, 4192, 32), (130, 60, 640, 128), (200, 9000, 160, 32)])
def test_prefill_rows(M, N, K, block, mth, dev):
    """mth_oil4_gemm_prefill at sizes of the row kernel and around them, rows of very different magnitudes: the bars of
    test_gpu_prefill."""
    import torch
    from test_gpu_prefill import check
    print(f"prefill rows M={M} N={N} K={K} block={block}", flush=True)
    a, packed, cbs = synth.prefill(M, N, K, block)
    A = torch.from_numpy(synth.bf16_to_f32(a).reshape(M, K)) * torch.exp2(torch.arange(M) % 41 - 20.0)[:, None]
    c = torch.zeros(M * N, dtype=torch.bfloat16, device=dev)
    mth.oil4_gemm_prefill(A.bfloat16().to(dev), to_dev(packed, dev), to_dev(cbs, dev), block, c, M, N, K)
    torch.cuda.synchronize()
    W = synth.dequant_oil4(packed, cbs, N, K, block).astype(np.float64)
    A = A.bfloat16().double().numpy()
    check(c.view(torch.int16).cpu().numpy().view(np.uint16).reshape(M, N), A @ W.T, np.abs(A) @ np.abs(W).T, "rows")


# 16 tokens; row counts that pick every tile width with a last tile of 16 columns and more: 64 (1616), 96 (24016),
# 112 (28016, 128 where K % 256 != 0), 128 (32016); K of two steps, of whole rounds of four and two past them
@pytest.mark.parametrize("x32", [False, True])
@pytest.mark.parametrize("M,N,K", [(16, 1616, 128), (300, 1616, 640), (16, 24016, 256), (16, 24016, 384),
                                   (16, 28016, 512), (16, 28016, 384), (16, 32016, 256), (16, 32016, 384),
                                   (1100, 4096, 384)])
def test_prefill_tile_edges(M, N, K, x32, mth, dev):
    """bf16 rows on the tiled prompt kernels where the last tile or the last round of steps is partial; FP32 rows of the
    same shapes: the parts keep 2^-22 of a product and the sums round less than K / 16 times."""
    import ctypes as C
    import torch
    from test_gpu_prefill import check
    print(f"prefill tile edges M={M} N={N} K={K} x32={x32}", flush=True)
    a, packed, cbs = synth.prefill(M, N, K, 128)
    A = torch.from_numpy(synth.bf16_to_f32(a).reshape(M, K).copy())
    if x32:
        A = A * (1.0 + torch.rand(M, K, generator=torch.Generator().manual_seed(K)))
    x = A.to(dev) if x32 else A.bfloat16().to(dev)
    w, cb = to_dev(packed, dev), to_dev(cbs, dev)
    c = torch.full((M * N + 64,), float("nan"), dtype=torch.float32 if x32 else torch.bfloat16, device=dev)
    if x32:
        mth.oil4_gemv(w, cb, 128, x, c[:M * N], N, K, M)
    else:
        L, P = mth.lib, C.c_void_p
        size = {}
        for name, sym, n in (("ws", "_ZN3mth28oil4_prefill_workspace_bytesEllll", 4),
                             ("shift", "_ZN3mth24oil4_prefill_shift_bytesEl", 1)):
            f = getattr(L, sym)
            f.argtypes, f.restype = [C.c_int64] * n, C.c_size_t
            size[name] = f
        f = L._ZN3mth28launch_oil4_gemm_prefill_a16EPKtPKhS1_lPtlllPvP12ihipStream_t
        f.argtypes, f.restype = [P, P, P, C.c_int64, P, C.c_int64, C.c_int64, C.c_int64, P, P], C.c_int
        assert size["ws"](M, N, K, 128) > 0
        ws = torch.zeros(size["shift"](M) + size["ws"](M, N, K, 128), dtype=torch.uint8, device=dev)
        assert f(x.data_ptr(), w.data_ptr(), cb.data_ptr(), 128, c.data_ptr(), M, N, K, ws.data_ptr(),
                 torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    assert bool(torch.isnan(c[M * N:]).all())
    W = torch.from_numpy(synth.dequant_oil4(packed, cbs, N, K, 128)).to(dev).double()
    xd = x.double()
    ref, absw = (xd @ W.T.contiguous()).cpu().numpy(), (xd.abs() @ W.abs().T.contiguous()).cpu().numpy()
    got = c[:M * N].cpu().reshape(M, N)
    if x32:
        assert bool((np.abs(got.double().numpy() - ref) <= (K / 16 + 8) * 2.0 ** -24 * absw).all())
    else:
        check(got.view(torch.int16).numpy().view(np.uint16), ref, absw, "tile edges")


@pytest.mark.parametrize("entry", ["prefill", "gemv"])
def test_partial_tiles_under_capture(entry, mth, dev):
    """A capture on a stream whose workspace holds the row shifts alone: partial tiles take the kernels that need no
    more, and every replay gives the same values."""
    import torch
    from test_gpu_prefill import check
    M, N, K = 300, 7056, 384
    print(f"partial tiles under capture {entry}", flush=True)
    a, packed, cbs = synth.prefill(M, N, K, 128)
    w, cb = to_dev(packed, dev), to_dev(cbs, dev)
    A = torch.from_numpy(synth.bf16_to_f32(a).reshape(M, K).copy()).to(dev)
    x = A.bfloat16() if entry == "prefill" else A
    c = torch.zeros(M * N, dtype=x.dtype, device=dev)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    mth.workspace_reserve((4 * M + 255) // 256 * 256, stream=s)
    gr = torch.cuda.CUDAGraph()
    with torch.cuda.graph(gr, stream=s):
        if entry == "prefill":
            mth.oil4_gemm_prefill(x, w, cb, 128, c, M, N, K)
        else:
            mth.oil4_gemv(w, cb, 128, x, c, N, K, M)
    W = torch.from_numpy(synth.dequant_oil4(packed, cbs, N, K, 128)).to(dev).double()
    ref = (A.double() @ W.T.contiguous()).cpu().numpy()
    absw = (A.double().abs() @ W.abs().T.contiguous()).cpu().numpy()
    for rep in range(3):
        c.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            gr.replay()
        torch.cuda.synchronize()
        got = c.cpu().reshape(M, N)
        if entry == "prefill":
            check(got.view(torch.int16).numpy().view(np.uint16), ref, absw, f"replay {rep}")
        else:
            assert bool((np.abs(got.double().numpy() - ref) <= (K / 16 + 8) * 2.0 ** -24 * absw).all()), rep


# a few rows of no whole tile; token counts of a prompt with rows and columns that are no whole tiles of its kernels
@pytest.mark.parametrize("M,K,batch,blk", [(130, 1120, 20, 0), (1616, 1280, 200, 128), (1616, 1280, 500, 128),
                                           (208, 1152, 300, 128), (1616, 1408, 500, 128)])
def test_token_rows_oil4_infinite_entry(M, K, batch, blk, mth, dev):
    """An infinite codebook entry times values 2^-60 below their row's largest (0 in both FP16 parts): +-Inf, as one
    FP32 product gives, and NaN where entries of both signs meet."""
    import torch
    print(f"token rows OIL4 infinite entry M={M} K={K} batch={batch}", flush=True)
    g = np.random.default_rng(8)
    nib = g.integers(2, 16, (M, K), dtype=np.uint8)          # entries 0 (+Inf) and 1 (-Inf) only where placed
    nib[3, 100] = nib[129, 1119] = nib[5, 40] = 0
    nib[7, 64] = nib[5, 1000] = 1
    cb = g.normal(0, 0.02, 16).astype(np.float16)
    cb[0], cb[1] = np.inf, -np.inf
    x = (1.0 + g.random((batch, K))).astype(np.float32)
    x[:, [100, 1119, 40, 64, 1000]] = 2.0 ** -60
    y = empty(batch * M, torch.float32, dev)
    cbs = np.tile(cb.view(np.uint16), M * (K // blk) if blk else 1)
    mth.oil4_gemv(to_dev(nib[:, 0::2] | (nib[:, 1::2] << 4), dev), to_dev(cbs, dev), blk, to_dev(x, dev), y, M, K, batch)
    torch.cuda.synchronize()
    got = y.cpu().numpy().reshape(batch, M)
    assert (got[:, [3, 129]] == np.inf).all() and (got[:, 7] == -np.inf).all() and np.isnan(got[:, 5]).all()
    rest = [m for m in range(M) if m not in (3, 5, 7, 129)]
    assert np.isfinite(got[:, rest]).all()
