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
