"""Causal prefill attention at the edges of its tiling: group sizes that do and
do not divide the 32-row tiles, one token to several tiles, prefixes that end
inside a K/V tile, and each workgroup shape (by the number of row tiles:
many KV groups reach the larger ones with few tokens), against 64 bits.

A row's error is bounded by the fp16 hi + lo halves of its weights (2^-22 of
each, so of the row's largest |v|), the 32-bit sums over up to 2000 positions
and the scores' own rounding through the exponential: 1e-5 of the row's
largest output covers them with a margin of about ten."""
import ctypes

import numpy as np
import pytest

import si_amd
from tests.gpu_helpers import dev, empty, host

pytestmark = pytest.mark.gpu

CASES = [  # qheads, kvheads, hdim, tokens, prefix
    (14, 2, 64, 2, 0), (14, 2, 64, 33, 0), (28, 4, 128, 37, 91), (12, 2, 128, 5, 31),
    (3, 1, 96, 43, 64), (16, 1, 32, 70, 33), (5, 5, 32, 32, 32), (8, 8, 96, 65, 1),
    (64, 64, 32, 530, 7),     # 2 row tiles per workgroup
    (32, 32, 64, 1030, 0), (64, 32, 96, 300, 3), (40, 8, 128, 420, 29),
    (32, 32, 128, 1300, 0),   # 4 row tiles per workgroup
    (64, 64, 96, 650, 130),
]


@pytest.mark.parametrize("qh,kv,d,n,prefix", CASES)
def test_prefill_attention_edges(qh, kv, d, n, prefix):
    import torch
    g = torch.Generator(device="cuda").manual_seed(qh * 1000 + n)
    q = torch.randn(n, qh, d, generator=g, device="cuda")
    q[0] *= 30  # a row whose weights are nearly one position
    k, v = (torch.randn(prefix + n, kv, d, generator=g, device="cuda").half() for _ in range(2))
    k[prefix] *= 4  # the running maximum jumps there
    s = si_amd.make_shape(32, qh, kv, d)
    out, qs = empty((n, qh, d), torch.float32), empty((n, qh * d), torch.int8)
    sc, bs = empty((n, qh * d // 32), torch.int16), empty((n, qh * d // 32), torch.int16)
    need = si_amd.lib().si_attention_workspace(ctypes.byref(s), n, prefix + n)
    ws = empty((need,), torch.uint8)
    si_amd.call("si_attention", ctypes.byref(s), si_amd.ptr(q), n, si_amd.ptr(k), si_amd.ptr(v),
                0, None, prefix + 1, 1, prefix + n, si_amd.ptr(out), si_amd.ptr(qs),
                si_amd.ptr(sc), si_amd.ptr(bs), si_amd.ptr(ws), need, si_amd.stream_handle())
    hidden = torch.ones(n, prefix + n, dtype=torch.bool, device="cuda").triu_(prefix + 1)
    for h in range(qh):
        kg, vg = (t[:, h // (qh // kv)].double().contiguous() for t in (k, v))
        p = (q[:, h].double() @ kg.T.contiguous()) / d ** 0.5
        want = p.masked_fill_(hidden, -float("inf")).softmax(1) @ vg
        err = (out[:, h].double() - want).abs().amax(1) / want.abs().amax(1)
        assert err.max().item() < 1e-5, (h, int(err.argmax()), err.max().item())
    # the Q8_0 rows are those of the output itself
    o, w, dd = host(out).reshape(n, -1, 32), host(qs).reshape(n, -1, 32), host(sc)
    amax = np.abs(o).max(2)
    scale = amax / np.float32(127)
    assert np.array_equal(dd.view(np.float16), scale.astype(np.float16))
    with np.errstate(divide="ignore", invalid="ignore"):
        inv = np.where(scale > 0, np.float32(1) / scale, 0).astype(np.float32)
    assert np.array_equal(w, np.rint(o * inv[..., None]).clip(-127, 127).astype(np.int8))
    assert np.array_equal(host(bs), w.astype(np.int32).sum(2).astype(np.int16))


@pytest.mark.parametrize("offset", [0, 1, 4, 8])
@pytest.mark.parametrize("qh,kv,d,n,prefix", [(14, 2, 64, 5, 30), (12, 2, 128, 33, 7),
                                              (3, 1, 96, 43, 64), (5, 5, 32, 32, 32),
                                              (64, 32, 96, 300, 3), (32, 32, 128, 1300, 0)])
def test_prefill_attention_cache_address(qh, kv, d, n, prefix, offset):
    """A cache that starts off a 16-byte boundary, which the copies into LDS do not
    take: the same kernel with its tiles through registers, and the same values
    within the bound above of both."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(qh + n)
    q = torch.randn(n, qh, d, generator=g, device="cuda")
    rows = (prefix + n) * kv * d
    k, v = (torch.randn(rows, generator=g, device="cuda").half() for _ in range(2))
    # (no row past the last is weighed: what lies there would be seen)
    kb, vb = (torch.full((rows + 16,), float("nan"), dtype=torch.float16, device="cuda")
              for _ in range(2))
    kb[offset:offset + rows], vb[offset:offset + rows] = k, v
    s = si_amd.make_shape(32, qh, kv, d)
    need = si_amd.lib().si_attention_workspace(ctypes.byref(s), n, prefix + n)
    ws = empty((need,), torch.uint8)
    outs, names = [], []
    for kc, vc in ((k, v), (kb[offset:], v), (k, vb[offset:]), (kb[offset:], vb[offset:])):
        out = empty((n, qh, d), torch.float32)
        names.append(si_amd.kernel_times_ms("k_", lambda: si_amd.call(
            "si_attention", ctypes.byref(s), si_amd.ptr(q), n, si_amd.ptr(kc), si_amd.ptr(vc), 0,
            None, prefix + 1, 1, prefix + n, si_amd.ptr(out), None, None, None, si_amd.ptr(ws),
            need, si_amd.stream_handle()))[0][0])
        outs.append(out.double())
    by_registers = "k_attn_prefill<%d, 2, 2, false>" % d
    assert names[0].startswith("k_attn_prefill") and names[0] != by_registers
    for name, out in zip(names[1:], outs[1:]):
        assert name == (names[0] if offset % 8 == 0 else by_registers), names
        err = (outs[0] - out).abs().amax(2) / outs[0].abs().amax(2)
        assert err.max().item() < 2e-5
