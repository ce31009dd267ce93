"""The fp6 GEMM's block-major scales: rows padded to 8 on either side, K that
ends inside a stage, a K split; against the default tile kernel, which the
same call runs when the workspace has no room for them (the same sums in the
same order, so the outputs are equal bit for bit)."""
import numpy as np
import pytest

import si_amd
from tests.gpu_helpers import aos_to_planar, dev, empty, host, q4

pytestmark = pytest.mark.gpu


def _up(b):
    return (b + 255) // 256 * 256


@pytest.mark.parametrize("m,n,k", [(1, 8, 320), (65, 40, 96), (130, 200, 1056), (515, 136, 2080),
                                   (777, 1000, 896)])
def test_f6_scales(oracle, m, n, k):
    import torch
    L = si_amd.lib()
    rng = np.random.default_rng(m + n + k)
    w = q4(oracle, rng, n, k)
    qs, d, _ = aos_to_planar(oracle.quantize_q8(rng.standard_normal((m, k)).astype(np.float32)))
    tile = L.si_q4_tile(n, k)
    wqs = empty(n * k // 2, torch.uint8)
    wd = empty(L.si_q4_scale_count(n, k, tile), torch.int16)
    wd.zero_()
    si_amd.call("si_q4_repack", si_amd.ptr(dev(w)), n, k, tile, si_amd.ptr(wqs), si_amd.ptr(wd),
                None)
    xqs, xd = dev(qs), dev(d.view(np.int16))
    total = L.si_gemm_f6_workspace(m, n, k)
    nb = k // 32
    # the operands without the activations' scales
    least = total - _up(m * nb * 48 + (m + 7) // 8 * 8 * nb * 2) + _up(m * nb * 48)
    assert n % 8 == 0 and least < total

    def run(wsb):
        ws = empty(wsb, torch.uint8)
        ws.fill_(0x7c)  # padding rows: fp16 NaN scales, which reach no output
        out = empty(m * n, torch.float32)
        ran = [kn for kn, _ in si_amd.kernel_times_ms("k_gemm", lambda: si_amd.call(
            "si_gemm_q4q8", si_amd.ptr(wqs), si_amd.ptr(wd), tile, n, k, si_amd.ptr(xqs),
            si_amd.ptr(xd), m, None, None, si_amd.ptr(out), n, si_amd.SI_GEMM_F6, si_amd.ptr(ws),
            wsb, None))]
        return ran[0], host(out)

    kern, got = run(total)
    assert kern.startswith("k_gemm_f6"), kern
    kern, want = run(least)
    assert kern.startswith("k_gemm_fast"), kern
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    with pytest.raises(RuntimeError):
        run(least - 1)


@pytest.mark.parametrize("m,f,k,gu_given", [(7, 32, 96, False), (40, 64, 96, False),
                                            (64, 160, 128, True), (130, 96, 128, False),
                                            (777, 4864, 896, True)])
def test_f6_scales_gateup(oracle, m, f, k, gu_given):
    """The fused gate|up pass with and without room for the scales: the short
    workspace runs the tile kernel, also at the rows the streaming kernel would
    take and with no gate|up output, to the same bytes."""
    import torch
    L = si_amd.lib()
    rng = np.random.default_rng(m + f + k)
    w = np.concatenate([q4(oracle, rng, f, k), q4(oracle, rng, f, k)])
    qs, d, _ = aos_to_planar(oracle.quantize_q8(rng.standard_normal((m, k)).astype(np.float32)))
    wqs = empty(f * k, torch.uint8)
    wd = empty(L.si_q4_scale_count(2 * f, k, 32), torch.int16)
    wd.zero_()
    si_amd.call("si_q4_repack", si_amd.ptr(dev(w)), 2 * f, k, 32, si_amd.ptr(wqs), si_amd.ptr(wd),
                None)
    xqs, xd = dev(qs), dev(d.view(np.int16))
    total = L.si_gemm_f6_workspace(m, 2 * f, k)
    nb = k // 32
    least = total - _up(m * nb * 48 + (m + 7) // 8 * 8 * nb * 2) + _up(m * nb * 48)
    assert least < total

    def run(wsb):
        ws = empty(total, torch.uint8)
        ws.fill_(0x7c)
        gu = empty(m * 2 * f, torch.float32) if gu_given else None
        act = empty(m * f, torch.float32)
        aq, ad, asum = (empty(c, t) for c, t in ((m * f, torch.int8), (m * f // 32, torch.int16),
                                                 (m * f // 32, torch.int16)))
        ran = si_amd.kernel_times_ms("k_gemm", lambda: si_amd.call(
            "si_gemm_gateup_q8", si_amd.ptr(wqs), si_amd.ptr(wd), 32, f, k, si_amd.ptr(xqs),
            si_amd.ptr(xd), m, si_amd.ptr(gu), si_amd.ptr(act), si_amd.ptr(aq), si_amd.ptr(ad),
            si_amd.ptr(asum), si_amd.SI_GEMM_F6, si_amd.ptr(ws), wsb, None))
        return ran[0][0], [host(t) for t in (act, aq, ad, asum) + ((gu,) if gu_given else ())]

    kern, got = run(total)
    assert kern.startswith("k_gemm_f6"), kern
    kern, want = run(least)
    assert kern.startswith("k_gemm_fast"), kern
    for a, b in zip(got, want):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8))
    with pytest.raises(RuntimeError, match="from %d on" % least):
        run(least - 1)
