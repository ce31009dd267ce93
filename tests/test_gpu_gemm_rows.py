"""The one-tile GEMM at row counts whose 32-row halves do not divide an XCD's CUs: every output
element is computed (each half, K range and column tile has one workgroup), to the bits of the
same rows in calls of 32, which place one half per workgroup."""
import numpy as np
import pytest

import si_amd
from tests.gpu_helpers import aos_to_planar, dev, empty, host, q4

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [65, 130, 161, 224, 257, 320, 333, 352, 384, 385, 448, 480])
@pytest.mark.parametrize("n,k", [(1152, 896), (40, 3584), (896, 4864)])
def test_gemm_rows_placement(oracle, m, n, k):
    import torch
    L = si_amd.lib()
    rng = np.random.default_rng(m + n + k)
    w = q4(oracle, rng, n, k)
    qs, d, _ = aos_to_planar(oracle.quantize_q8(rng.standard_normal((m, k)).astype(np.float32)))
    qs, d = qs.reshape(m, k), d.view(np.int16).reshape(m, k // 32)
    tile = L.si_q4_tile(n, k)
    wqs = empty(n * k // 2, torch.uint8)
    wd = empty(L.si_q4_scale_count(n, k, tile), torch.int16)
    wd.zero_()
    si_amd.call("si_q4_repack", si_amd.ptr(dev(w)), n, k, tile, si_amd.ptr(wqs), si_amd.ptr(wd),
                None)

    def run(r0, r1):
        rows = r1 - r0
        wsb = L.si_gemm_workspace(rows, n, k)
        ws = empty(max(wsb, 1), torch.uint8)
        out = empty(rows * n, torch.float32)
        out.fill_(float("nan"))
        xqs, xd = dev(np.ascontiguousarray(qs[r0:r1])), dev(np.ascontiguousarray(d[r0:r1]))
        ran = [kn for kn, _ in si_amd.kernel_times_ms("k_gemm", lambda: si_amd.call(
            "si_gemm_q4q8", si_amd.ptr(wqs), si_amd.ptr(wd), tile, n, k, si_amd.ptr(xqs),
            si_amd.ptr(xd), rows, None, None, si_amd.ptr(out), n, 0, si_amd.ptr(ws), wsb, None))]
        assert ran[0].startswith("k_gemm_bd"), ran
        return host(out).reshape(rows, n)

    got = run(0, m)
    want = np.concatenate([run(r, min(r + 32, m)) for r in range(0, m, 32)])
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
