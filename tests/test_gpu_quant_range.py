"""quantize_q8 and SwiGLU at the ends of their short forms' ranges: block maxima
around 2^-100 and 2^100 (where the kernels change formulation), zero, subnormal
and infinite maxima, NaN among the values, ties, against the oracle's bytes."""
import numpy as np
import pytest

import si_amd
from oracle.oracle_py import Oracle
from tests.gpu_helpers import dev, empty, host, planar_to_aos

pytestmark = pytest.mark.gpu
QK = 32

MAXIMA = [0.0, 1e-45, 1e-40, 3e-39, 4.3e-37, 1e-36, 1e-31, 2.0 ** -100, 2.0 ** -99.9, 1e-20, 1.0,
          127.0, 65504.0, 8.4e6, 2.0 ** 99.9, 2.0 ** 100, 1e31, 3.4e38, np.inf]


@pytest.mark.parametrize("neighbour", [-1, 0, 1])
def test_quantize_range_edges(neighbour):
    rng = np.random.default_rng(11 + neighbour)
    blocks = []
    for m in MAXIMA:
        m = np.float32(m)
        if neighbour and 0 < m < np.inf:
            m = np.nextafter(m, np.float32(np.inf if neighbour > 0 else 0), dtype=np.float32)
        with np.errstate(all="ignore"):
            x = (rng.uniform(-1, 1, (4, QK)) * m).astype(np.float32)
            x[1] = (np.arange(QK) - 15.5) * (m / np.float32(127))  # ties
            x[2, ::5] = np.nan
            x[3] = 0
        x[:, 7] = m
        x[0, 9] = -m
        blocks.append(x)
    x = np.concatenate(blocks).astype(np.float32)
    want = Oracle().quantize_q8(x.reshape(-1))
    n = x.size
    import torch
    tq, td, ts = (empty((k,), t) for k, t in ((n, torch.int8), (n // QK, torch.int16),
                                              (n // QK, torch.int16)))
    si_amd.call("si_quantize_q8_rows", si_amd.ptr(dev(x)), 1, n, si_amd.ptr(tq), si_amd.ptr(td),
                si_amd.ptr(ts), si_amd.stream_handle())
    qs, d, s = host(tq), host(td).view(np.uint16), host(ts)
    got = planar_to_aos(qs, d)
    bad = [i for i in range(len(want)) if got[i].tobytes() != want[i].tobytes()]
    assert not bad, [(i // 4, i % 4, got[i], want[i]) for i in bad[:3]]
    assert np.array_equal(s, qs.reshape(-1, QK).astype(np.int32).sum(1).astype(np.int16))


def test_swiglu_range_edges():
    """Against 64 bits, g from where e^-g vanishes to where it overflows; silu's float rounding
    steps (e^-g, 1 + e^-g, the quotient, the product) bound the error by 4 * 2^-24 relative."""
    import torch
    f = 4096
    g = np.concatenate([np.linspace(-88.7, 110, f - 8), [0.0, 1e-40, -1e-30, 88.8, 104, 1e30, -88,
                                                       -87.5]]).astype(np.float32)
    u = np.random.default_rng(3).normal(0, 1, f).astype(np.float32)
    act, qs, d = empty((f,), torch.float32), empty((f,), torch.int8), empty((f // QK,), torch.int16)
    si_amd.call("si_swiglu_q8", si_amd.ptr(dev(np.concatenate([g, u]))), 1, f, si_amd.ptr(act),
                si_amd.ptr(qs), si_amd.ptr(d), None, si_amd.stream_handle())
    got = host(act).astype(np.float64)
    g64 = g.astype(np.float64)
    with np.errstate(over="ignore"):
        want = g64 / (1 + np.exp(-g64)) * u
    assert (np.abs(got - want) <= 4 * 2.0 ** -24 * np.abs(want) + 1e-44).all()
    # e^-g overflows: the quotient is a zero, an infinite g keeps its value, NaN stays NaN
    edge = np.array([-89, -1000, -np.inf, np.inf, np.nan] + [0.0] * 27, np.float32)
    si_amd.call("si_swiglu_q8", si_amd.ptr(dev(np.concatenate([edge, np.ones(QK, np.float32)]))),
                1, QK, si_amd.ptr(act), si_amd.ptr(qs), si_amd.ptr(d), None,
                si_amd.stream_handle())
    got = host(act)[:5]
    assert got[0] == 0 and got[1] == 0 and np.isnan(got[2]) and got[3] == np.inf and \
        np.isnan(got[4])


def test_swiglu_small_gates():
    """silu(g) = g / 2 for |g| below 2^-60, rounded once: subnormal gates, those a
    quarter of which is subnormal, and zeros of either sign, bit for bit."""
    import torch
    bits = np.concatenate([np.arange(1, 64), 1 << np.arange(23), (1 << np.arange(23)) + 1,
                           [0x7fffff], np.arange(1, 66) * 0x800000, np.arange(1, 66) * 0x800000 + 1,
                           np.arange(1, 66) * 0x800000 + 0x7fffff]).astype(np.uint32)
    bits = np.concatenate([bits, bits | 0x80000000, [0, 0x80000000]]).astype(np.uint32)
    g = np.resize(bits, (len(bits) + QK - 1) // QK * QK).view(np.float32)
    for scale in (np.float32(1), np.float32(2.0 ** 100), np.float32(-1.5 * 2.0 ** 90)):
        u = np.full_like(g, scale)
        f = len(g)
        act, qs, d = (empty((k,), t) for k, t in ((f, torch.float32), (f, torch.int8),
                                                  (f // QK, torch.int16)))
        si_amd.call("si_swiglu_q8", si_amd.ptr(dev(np.concatenate([g, u]))), 1, f, si_amd.ptr(act),
                    si_amd.ptr(qs), si_amd.ptr(d), None, si_amd.stream_handle())
        want = (g.astype(np.float64) / 2).astype(np.float32) * u
        got = host(act)
        bad = got.view(np.uint32) != want.view(np.uint32)
        assert not bad.any(), [(float(x).hex(), y, z) for x, y, z in zip(g[bad][:4], got[bad], want[bad])]


def _significand_blocks(first, count):
    """Blocks whose maxima are 1.s for count significands s: their values lie where
    the product with 1 / d falls on a tie, or next to one, so the int8 values
    tell the right inverse from its neighbours.  Returns (values, 1 / d, d)."""
    amax = (np.uint32(0x3f800000) + np.arange(first, first + count, dtype=np.uint32)).view(np.float32)
    d = amax / np.float32(127)
    inv = np.float32(1) / d
    k = np.arange(QK) * 4 - 0.5 + np.arange(QK) % 2  # 0.5 past odd and even numbers
    k[:2] = 63.5, 98.5
    x = k.astype(np.float32) / inv[:, None]
    x[:, 31] = amax
    x[:, 30] = -amax
    return x, inv, d


def _values(x, inv):
    return np.rint(np.clip(x * inv[:, None], -127, 127)).astype(np.int8)


def test_quantize_every_significand():
    """The short forms of amax / 127 and 1 / d (a product with its remainder, the
    hardware's reciprocal with one Newton step) against the IEEE divisions for
    all 2^23 significands: a reciprocal one step off is wrong for 32 of them
    after that step, so this pins the chip's."""
    x, inv, _ = _significand_blocks(1234567, 1 << 16)
    want = _values(x, inv)
    for off in (np.inf, -np.inf):  # the values do tell (the mistake is made in the oracle)
        near = np.nextafter(inv, np.float32(off), dtype=np.float32)
        assert (want != _values(x, near)).any(1).mean() > 0.99
    import torch
    count = 1 << 20
    n = count * QK
    tq, td = empty((n,), torch.int8), empty((count,), torch.int16)
    for first in range(0, 1 << 23, count):
        x, inv, d = _significand_blocks(first, count)
        tx = torch.from_numpy(x).cuda()
        si_amd.call("si_quantize_q8_rows", si_amd.ptr(tx), 1, n, si_amd.ptr(tq), si_amd.ptr(td),
                    None, si_amd.stream_handle())
        assert np.array_equal(host(td).view(np.uint16), d.astype(np.float16).view(np.uint16))
        bad = (host(tq).reshape(count, QK) != _values(x, inv)).any(1)
        assert not bad.any(), (first + np.flatnonzero(bad)[:4], int(bad.sum()))
        print(f"significands {first:#x}..{first + count - 1:#x} the same", flush=True)
