"""Which kernels a call launches and what it keeps in the workspace, with the
HIP runtime replaced by a recorder (recorded.py): no GPU.
"""
import itertools
import os
import textwrap

import recorded

W, CB, X, Y, Z = (0x100000000000 * (i + 1) for i in range(5))   # 16-byte aligned device addresses, never touched
ROWS = ("rows_split", "rows_half", "rows_mfma", "rows_reduce")
PER_THREAD = 2                                                   # hipStreamPerThread
stream = itertools.count(0x10000, 0x100)                         # a fresh stream: no workspace yet


def oil8(M, K, b, s, x=X):
    return {"fn": "mth_oil8_gemv", "args": [W, CB, x, Y, M, K, b, s]}


def oil4(M, K, b, s, blk=128):
    return {"fn": "mth_oil4_gemv", "args": [W, CB, blk, X, Y, M, K, b, s]}


def i2s(M, K, b, s):
    return {"fn": "mth_i2s_gemv", "args": [W, 1.0, X, CB, Y, M, K, b, s]}


def i2s_f32(M, K, b, s):
    return {"fn": "mth_i2s_gemv_f32", "args": [W, 1.0, X, Y, M, K, b, s]}


def i2s_gemm(M, N, K, s):
    return {"fn": "mth_i2s_gemm", "args": [W, X, Y, M, N, K, s]}


def attention(b, h, kvh, D, ctx, s):
    return {"fn": "mth_attention_decode", "args": [X, W, CB, Y, b, h, kvh, D, ctx, ctx, s]}


def kernels(r):
    assert r["rc"] == 0, r["error"]
    return [n for n, _ in r["kernels"]]


def on(r, *names):
    """Whether one of the call's kernels has one of these names in its own."""
    return any(n in k for k in kernels(r) for n in names)


# one call of each entry point whose other route keeps nothing in the workspace, and its workspace kernels
def without_workspace(s):
    return [(attention(2, 32, 8, 128, 6000, s), "attn_split_k"), (i2s_gemm(4096, 300, 4096, s), "rows_mfma_k"),
            (i2s_f32(4096, 11008, 16, s), "i2s_quant_rows_k"), (oil8(64, 17024, 1, s), "rows_mfma_k"),
            (oil4(7529, 10240, 1, s, 64), "rows_mfma_k")]


def test_per_thread_stream_shares_no_workspace():
    """hipStreamPerThread is one handle for a stream of its own in every
    thread: calls that can do without the workspace, which is kept by handle,
    do so there."""
    calls = without_workspace(PER_THREAD)
    for (c, name), r in zip(calls, recorded.run([c for c, _ in calls])):
        assert not on(r, name) and r["mallocs"] == 0, (c, kernels(r))
    calls = without_workspace(next(stream))                      # an ordinary stream: the route with workspace
    for (c, name), r in zip(calls, recorded.run([c for c, _ in calls])):
        assert on(r, name), (c, kernels(r))


def test_partial_tiles_of_fp32_rows():
    """FP32 token rows whose columns or K steps are no whole tiles of the
    prompt GEMM keep off it (an infinite codebook entry would meet a part that
    is 0 there); whole tiles run on it."""
    calls = [oil4(M, K, b, next(stream)) for M in (1616, 8016, 14352, 24016) for K in (384, 640, 768, 1280, 1920)
             for b in (128, 200, 500)]
    for c, r in zip(calls, recorded.run(calls)):
        assert not on(r, "oil4_prefill_ws"), (c, kernels(r))
    r = recorded.run([oil4(22016, 4096, 512, next(stream))])[0]
    assert on(r, "oil4_prefill_ws"), kernels(r)


def test_token_rows_take_no_more_launches():
    """17 .. 127 tokens at shapes the batched GEMVs take (16 tokens per launch,
    with a reduction where K is split): the route taken has no more launches."""
    calls, most = [], []
    for K in (512, 1024, 2048, 4096):
        for M in (256, 2048, 8192, 16384, 32000):
            for b in (17, 32, 33, 48, 64, 127):
                calls += [oil8(M, K, b, next(stream)), oil4(M, K, b, next(stream)), oil4(M, K, b, next(stream), 0)]
                most += 3 * [(b + 15) // 16 * (1 if K == 512 else 2)]
    for c, n, r in zip(calls, most, recorded.run(calls)):
        assert len(kernels(r)) <= n, (c, kernels(r))


def test_few_int8_ternary_tokens_take_the_faster_route():
    """A few int8 tokens at shapes where the walk over the tokens and the token
    rows (two launches, three with a K split) were timed: the faster of the two."""
    walk = [(1024, 832, 13), (4096, 320, 12), (512, 260, 12), (1024, 260, 14), (4096, 1984, 9), (8192, 1984, 6),
            (4096, 2052, 2), (1024, 9152, 6), (4096, 3136, 7), (8192, 832, 8)]      # 9.4 .. 12.6 us; rows 12 .. 16.9
    rows = [(512, 192, 14), (4096, 832, 16), (4096, 4096, 8), (8192, 9152, 3), (1024, 9152, 10), (4096, 388, 12),
            (8192, 5188, 2), (1024, 260, 17), (64, 64, 17)]                         # 12 .. 15.7 us; the walk 12.5 .. 36
    calls = [i2s(M, K, b, next(stream)) for M, K, b in walk + rows]
    for i, (c, r) in enumerate(zip(calls, recorded.run(calls))):
        assert (len(kernels(r)) > 1) == (i >= len(walk)), (c, kernels(r))


def test_attention_of_64_columns_splits_where_it_pays():
    """Few heads of 64 columns over a cache of more than 1024 positions: one
    launch to 1374 positions (at 1260: 10.9 .. 11.4 us against 11.4 .. 12.1),
    two from 1375 (at 1400: 12.0 .. 12.9 against 11.0 .. 12.2)."""
    calls = [attention(1, 32, 8, 64, ctx, next(stream)) for ctx in (1260, 1306, 1374, 1375, 1400, 6000)]
    assert [len(kernels(r)) for r in recorded.run(calls)] == [1, 1, 1, 2, 2, 2]


def test_noalloc_runs_the_same_kernels():
    """mth_oil4_gemv_noalloc's results are mth_oil4_gemv's bit for bit at these
    sizes because both launch the same kernels."""
    sizes = [(b, K) for b, Ks in ((1, (32, 544, 4096, 4224, 11008, 16384)), (2, (512, 7680, 8192)), (16, (512, 4096)))
             for K in Ks]
    calls = [oil4(M, K, b, next(stream), blk) for b, K in sizes for M in (1, 700, 5000) for blk in (0, 128)
             if blk == 0 or K % blk == 0]
    calls += [oil4(700, K, 1, next(stream), 32) for K in (32, 1056, 4096)]
    for c, a, b in zip(calls, recorded.run(calls), recorded.run([dict(c, fn="mth_oil4_gemv_noalloc") for c in calls])):
        assert a["kernels"] == b["kernels"] and b["mallocs"] == 0 and kernels(b), c


def test_graphs_hold_no_workspace_of_calls_without():
    """Captured on a stream that holds a large workspace: calls whose other
    route keeps nothing there record no address of it, calls that need it do."""
    st = next(stream)
    calls = [{"fn": "mth_workspace_reserve", "args": [1 << 30, st]}]
    calls += [c for c, _ in without_workspace(st)]
    calls += [oil8(300, 1040, 40, st), oil8(512, 512, 40, st), oil8(300, 4112, 2, st), oil4(500, 1024, 40, st, 64),
              oil4(500, 640, 40, st), oil4(512, 512, 40, st), oil4(1616, 384, 200, st), i2s(130, 1028, 20, st),
              i2s(64, 260, 300, st), i2s(512, 256, 40, st)]
    needs = len(calls)
    calls += [oil8(4096, 4096, 40, st), oil4(4096, 4096, 40, st), i2s(4096, 4096, 40, st)]
    for c in calls[1:]:
        c["capture"] = st
    out = recorded.run(calls)
    for i, (c, r) in enumerate(zip(calls, out)):
        used = on(r, *ROWS, "i2s_pad_rows_k", "i2s_quant_rows_k", "i2s_gemm_mfma", "attn_combine", "reduce")
        assert used == (i >= needs) and (i == 0 or r["mallocs"] == 0), (c, kernels(r))


def threads(body):
    """A child with the recorder and the library loaded; body's `call(id, fn,
    args)` makes a call in a thread of its own."""
    head = """
        import sys, threading, time
        sys.path.insert(0, %r)
        import recorded, test_routes as t
        rec, lib = recorded.library()
        def call(i, c):
            def work():
                rec.rec_thread_id(i)
                assert getattr(lib, c["fn"])(*c["args"]) == 0
            th = threading.Thread(target=work, daemon=True)
            th.start()
            return th
        def until_waiting():
            end = time.time() + 20
            while not rec.rec_waiting():
                assert time.time() < end
                time.sleep(0.01)
        A, B = 0x10000000, 0x10000000 + (1 << 40)
    """ % os.path.dirname(os.path.abspath(__file__))
    recorded.child(["-c", textwrap.dedent(head) + textwrap.dedent(body)])


def test_a_full_queue_holds_up_no_other_stream():
    """While one thread waits for room in its stream's queue, calls on other
    streams go on, whether they use the workspace or not."""
    threads("""
        rec.rec_hold(A)
        first = call(1, t.oil8(4096, 4096, 1, A))       # one launch, no workspace
        until_waiting()
        rest = [call(2, c) for c in (t.oil8(4096, 4096, 1, B), t.oil4(11008, 4096, 1, B), t.i2s_gemm(4096, 300, 4096, B),
                                     t.attention(2, 32, 8, 128, 6000, B), t.oil8(4096, 4096, 40, B))]
        for th in rest:
            th.join(20)
            assert not th.is_alive()
        assert first.is_alive()
        rec.rec_release()
        first.join(20)
        rec.rec_hold(A)
        first = call(1, t.i2s_gemm(4096, 300, 4096, A))  # three launches through the workspace
        until_waiting()
        rest = [call(2, c) for c in (t.i2s_gemm(4096, 300, 4096, B), t.oil8(4096, 4096, 40, B))]
        for th in rest:
            th.join(20)
            assert not th.is_alive()
        rec.rec_release()
        first.join(20)
        assert not first.is_alive()
    """)


def test_threads_that_share_a_stream_enqueue_in_turn():
    """Calls that hand data on through a stream's workspace: no other call's
    launches come between theirs."""
    threads("""
        calls = [t.i2s_gemm(4096, 300, 4096, A), t.attention(2, 32, 8, 128, 6000, A), t.oil8(4096, 4096, 40, A),
                 t.oil4(1616, 1920, 200, A), t.i2s_f32(4096, 11008, 16, A), t.oil4(4096, 4096, 8, A)]
        for rep in range(20):
            rec.rec_reset()
            rec.rec_hold(A)
            all_ = [call(1, calls[rep % len(calls)])]
            until_waiting()
            all_ += [call(2 + i, c) for i, c in enumerate(calls)]
            time.sleep(0.05)
            assert rec.rec_launches() == 1
            rec.rec_release()
            for th in all_:
                th.join(20)
                assert not th.is_alive()
            ids = [rec.rec_thread(i) for i in range(rec.rec_launches())]
            runs = [i for k, i in enumerate(ids) if k == 0 or ids[k - 1] != i]
            assert len(runs) == len(set(runs)) == 1 + len(calls), ids
    """)


def test_workspace_grows_in_relaxed_capture_mode():
    """An allocation in the default mode invalidates a capture that another
    thread has open; the mode is the thread's own again afterwards."""
    threads("""
        import ctypes as C
        for c in (t.attention(2, 32, 8, 128, 6000, A), {"fn": "mth_workspace_reserve", "args": [1 << 28, B]}):
            rec.rec_reset()
            assert getattr(lib, c["fn"])(*c["args"]) == 0
            assert rec.rec_mallocs() == 1 and rec.rec_malloc_mode() == 2   # hipStreamCaptureModeRelaxed
            mode = C.c_int(0)
            assert rec.hipThreadExchangeStreamCaptureMode(C.byref(mode)) == 0 and mode.value == 0
    """)
