"""si_attention over batches of queries: the whole-row kernel (8 queries or
more, 1, 2 or 4 KV groups, 10 MiB of cache rows or more) against 64 bits at the
edges of its chunks and steps, with cache rows past each context poisoned, in
contiguous and paged caches, and the per-group kernel where the caches or the
workspace are smaller.

Bound: fp16 hi + lo weights (2^-22), 32-bit sums over up to 2100 positions and
the scores' rounding through the exponential, 1e-5 of a row's largest output."""
import ctypes

import numpy as np
import pytest

import si_amd
from tests.gpu_helpers import empty, host

pytestmark = pytest.mark.gpu

CASES = [  # qheads, kvheads, hdim, contexts (the longest is max_ctx)
    (28, 4, 128, [1, 2, 15, 16, 17, 63, 64, 65, 127, 128, 700, 2100]),
    (14, 2, 64, [0, 1, 31, 32, 33, 128, 129, 999]),
    (14, 2, 64, [5] * 8),
    (12, 2, 128, [300, 1, 299, 0, 64, 65, 128, 300, 17]),
    (5, 1, 32, [64, 63, 65, 1, 256, 257, 255, 0, 511]),
    (16, 1, 96, [70, 1, 2, 3, 64, 65, 66, 100]),
    (8, 4, 64, [40 + 7 * i for i in range(40)]),
    (5, 1, 32, [200, 1, 17, 64, 0, 199, 128, 2, 65]),
    # past ROWS_CACHE, contexts about the chunks' ends
    (28, 4, 128, [1, 63, 64, 65, 127, 129, 700, 0]),        # 11 chunks of 64
    (14, 2, 64, [0, 1, 127, 128, 129, 256, 257, 31, 2304]),  # 18 of 128
    (12, 2, 128, [1200, 1, 0, 127, 128, 129, 160, 31, 1199]),
    (5, 1, 32, [9300, 1, 303, 304, 305, 63, 64, 65, 0]),  # an odd count of partial states
    (16, 1, 96, [3500, 1, 255, 256, 257, 64, 65, 2]),
]
ROWS_CACHE = 10 << 20  # bytes of K and V rows from which the whole-row kernel runs


def _want(q, k, v, ctx, per):
    import torch
    out = torch.zeros(q.shape, dtype=torch.float64, device="cuda")
    for i, n in enumerate(ctx):
        if n:
            for h in range(q.shape[1]):
                kg, vg = (t[i, :n, h // per].double() for t in (k, v))
                p = (kg @ q[i, h].double() / q.shape[2] ** 0.5).softmax(0)
                out[i, h] = p @ vg
    return out


def _check(out, want, ctx):
    for i, n in enumerate(ctx):
        if n == 0:
            assert bool((out[i] == 0).all()), f"query {i}: empty context"
            continue
        err = (out[i].double() - want[i]).abs().amax(1) / want[i].abs().amax(1)
        assert err.max().item() < 1e-5, (i, n, err.max().item())


@pytest.mark.parametrize("qh,kv,d,ctx", CASES)
def test_attention_rows_edges(qh, kv, d, ctx):
    import torch
    n, most = len(ctx), max(ctx)
    g = torch.Generator(device="cuda").manual_seed(most)
    q = torch.randn(n, qh, d, generator=g, device="cuda")
    k, v = (torch.randn(n, most, kv, d, generator=g, device="cuda").half() for _ in range(2))
    for i, c in enumerate(ctx):  # rows no context reaches
        k[i, c:], v[i, c:] = float("nan"), float("inf")
    want = _want(q, k, v, ctx, qh // kv)
    s = si_amd.make_shape(32, qh, kv, d)
    cd = torch.tensor(ctx, dtype=torch.int32, device="cuda")
    full = si_amd.lib().si_attention_workspace(ctypes.byref(s), n, most)
    per_group = max(1, min((512 + kv * n - 1) // (kv * n), (most + 63) // 64))
    least = n * qh * max(per_group, 2) * (d + 2) * 4
    for need in {full, min(full, least)}:
        ws = torch.full((need // 4,), float("nan"), device="cuda")
        out, qs = empty((n, qh, d), torch.float32), empty((n, qh * d), torch.int8)
        sc = empty((n, qh * d // 32), torch.int16)
        ran = si_amd.kernel_times_ms("k_", lambda: si_amd.call(
            "si_attention", ctypes.byref(s), si_amd.ptr(q), n, si_amd.ptr(k), si_amd.ptr(v),
            k.stride(0), si_amd.ptr(cd), 0, 0, most, si_amd.ptr(out), si_amd.ptr(qs),
            si_amd.ptr(sc), None, si_amd.ptr(ws), need, si_amd.stream_handle()))
        rows = need == full and n * most * kv * d * 4 >= ROWS_CACHE
        assert ran[0][0].startswith("k_dec_attn_rows" if rows else "k_attn_decode_mfma"), ran
        _check(out, want, ctx)
    # the same rows through shuffled pages: the same bits as the contiguous call
    page = 16
    each = (most + page - 1) // page
    table = torch.randperm(n * each, generator=g, device="cuda").to(torch.int32).view(n, each)
    kp, vp = (torch.full((n * each, page, kv, d), float("nan"), device="cuda").half()
              for _ in range(2))
    pad = torch.full((n, each * page, kv, d), float("nan"), device="cuda").half()
    for pool, t in ((kp, k), (vp, v)):
        pad[:, :most] = t
        pool[table.long().view(-1)] = pad.view(n * each, page, kv, d)
    ws = torch.full((full // 4,), float("nan"), device="cuda")
    out = empty((n, qh, d), torch.float32)
    si_amd.call("si_attention_paged", ctypes.byref(s), si_amd.ptr(q), n, si_amd.ptr(kp),
                si_amd.ptr(vp), n * each, page, si_amd.ptr(table), each, si_amd.ptr(cd), most,
                si_amd.ptr(out), None, None, None, si_amd.ptr(ws), full, si_amd.stream_handle())
    ws = torch.full((full // 4,), float("nan"), device="cuda")
    flat = empty((n, qh, d), torch.float32)
    si_amd.call("si_attention", ctypes.byref(s), si_amd.ptr(q), n, si_amd.ptr(k), si_amd.ptr(v),
                k.stride(0), si_amd.ptr(cd), 0, 0, most, si_amd.ptr(flat), None, None, None,
                si_amd.ptr(ws), full, si_amd.stream_handle())
    assert np.array_equal(host(out), host(flat))


def test_attention_rows_host_contexts():
    """Contexts from the host (ctx0 + i * step, one cache per sequence)."""
    import torch
    qh, kv, d, n, ctx0, step = 14, 2, 64, 9, 30, 11
    ctx = [ctx0 + step * i for i in range(n)]
    g = torch.Generator(device="cuda").manual_seed(5)
    q = torch.randn(n, qh, d, generator=g, device="cuda")
    k, v = (torch.randn(n, ctx[-1], kv, d, generator=g, device="cuda").half() for _ in range(2))
    s = si_amd.make_shape(32, qh, kv, d)
    need = si_amd.lib().si_attention_workspace(ctypes.byref(s), n, ctx[-1])
    ws, out = empty((need,), torch.uint8), empty((n, qh, d), torch.float32)
    si_amd.call("si_attention", ctypes.byref(s), si_amd.ptr(q), n, si_amd.ptr(k), si_amd.ptr(v),
                k.stride(0), None, ctx0, step, ctx[-1], si_amd.ptr(out), None, None, None,
                si_amd.ptr(ws), need, si_amd.stream_handle())
    _check(out, _want(q, k, v, ctx, qh // kv), ctx)


@pytest.mark.parametrize("qh,kv,d,cap,ctx", [
    (28, 4, 128, 4096, [300, 1, 0, 32, 33, 299, 16, 17, 64, 65, 128, 200]),
    (28, 4, 128, 700, [100 + i for i in range(80)]),  # more queries than lanes, the longest last
    (14, 2, 64, 9000, [1000, 64, 65, 1, 0, 999, 500, 130]),
    (5, 1, 32, 20000, [0] * 8 + [5]),
    (16, 1, 96, 6000, [700, 1, 255, 256, 257, 128, 129, 2]),
    (12, 2, 128, 4096, [0] * 9),
])
@pytest.mark.parametrize("on_host", [False, True])
def test_attention_rows_short_contexts(qh, kv, d, cap, ctx, on_host):
    """Contexts far below max_ctx: the longest one's chunks are its share of the
    grid (max_ctx's share would leave it to one workgroup), seen in the partial
    states (outputs, then maxima: -inf for an empty chunk)."""
    import torch
    n = len(ctx)
    if on_host:
        ctx = [10 + 3 * i for i in range(n)]
    g = torch.Generator(device="cuda").manual_seed(cap)
    q = torch.randn(n, qh, d, generator=g, device="cuda")
    k, v = (torch.full((n, cap, kv, d), float("nan"), dtype=torch.float16, device="cuda")
            for _ in range(2))
    for i, c in enumerate(ctx):
        for t in (k, v):
            t[i, :c] = torch.randn(c, kv, d, generator=g, device="cuda").half()
    s = si_amd.make_shape(32, qh, kv, d)
    cd = None if on_host else torch.tensor(ctx, dtype=torch.int32, device="cuda")
    need = si_amd.lib().si_attention_workspace(ctypes.byref(s), n, cap)
    ws = torch.full((need // 4,), float("nan"), device="cuda")
    out = empty((n, qh, d), torch.float32)
    ran = si_amd.kernel_times_ms("k_", lambda: si_amd.call(
        "si_attention", ctypes.byref(s), si_amd.ptr(q), n, si_amd.ptr(k), si_amd.ptr(v),
        k.stride(0), si_amd.ptr(cd), 10, 3, cap, si_amd.ptr(out), None, None, None,
        si_amd.ptr(ws), need, si_amd.stream_handle()))
    assert ran[0][0].startswith("k_dec_attn_rows"), ran
    _check(out, _want(q, k, v, ctx, qh // kv), ctx)
    step = 16 * (4 // kv)
    ns = min(-(-cap // (4 * step)), -(-512 // n), 31)
    top = ws[n * qh * ns * d:][:n * qh * ns].view(n, qh, ns)
    up16 = lambda c: (c + 15) // 16 * 16
    chunk = min(up16(-(-cap // ns)), max(2 * step, up16(-(-max(ctx) // ns))))
    for i, c in enumerate(ctx):
        assert bool((torch.isfinite(top[i]).sum(1) == -(-c // chunk)).all()), (i, c, chunk)
