"""The layout of the attention's partial states in a workspace: the outputs, which
the kernels store and read 16 bytes a lane, start 16-byte aligned for every
count of states (one query of 5 heads and 9 queries of 5 heads have odd ones),
and the parts fill the stated bytes without overlap."""
import os
import subprocess

import si_amd

CSRC = os.path.join(si_amd.PKG, "csrc")
PROGRAM = r"""
#include "si_kernels.hpp"
#include <cstdio>
int main() {
    alignas(256) static char ws[1];
    for (int hdim : {32, 64, 96, 128})
        for (size_t n = 1; n <= 97; ++n) {
            const si::AttnParts p(ws, n, hdim);
            const size_t o = (char *)p.o - ws, m = (char *)p.m - ws, l = (char *)p.l - ws;
            const size_t on = n * hdim * 4, mn = n * 4, total = n * (hdim + 2) * 4;
            const size_t a[3][2] = {{o, on}, {m, mn}, {l, mn}};
            for (int i = 0; i < 3; ++i) {
                if (a[i][0] + a[i][1] > total) return printf("past the end: n %zu\n", n), 1;
                for (int j = 0; j < i; ++j)
                    if (a[i][0] < a[j][0] + a[j][1] && a[j][0] < a[i][0] + a[i][1])
                        return printf("overlap: n %zu\n", n), 1;
            }
            if (o % 16) return printf("outputs at %zu: n %zu\n", o, n), 1;
        }
    return 0;
}
"""


def test_outputs_aligned(tmp_path):
    src, exe = tmp_path / "parts.hip", tmp_path / "parts"
    src.write_text(PROGRAM)
    subprocess.run(["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "-std=c++17", "-I", CSRC, "-I",
                    si_amd.INCLUDE_DIR, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
