"""Set-up that belongs to one GPU (a kernel's LDS limit) is done once on each, not
once in the process: on the first device, on the second after it, again after a
failure, and by no call after that, also with many threads."""
import os
import subprocess

import si_amd

PROGRAM = r"""
#include "si_kernels.hpp"
#include <cstdio>
#include <thread>
#include <vector>
int main() {
    static si::PerDevice p;
    int n = 0;
    auto set = [&] { ++n; return true; };
    p.once(0, set);
    p.once(0, set);
    if (n != 1) return printf("device 0: %d\n", n), 1;
    p.once(1, set);
    p.once(63, set);
    p.once(1, set);
    if (n != 3) return printf("devices 1 and 63: %d\n", n), 1;
    p.once(2, [&] { ++n; return false; });
    p.once(2, set);
    p.once(2, set);
    if (n != 5) return printf("after a failure: %d\n", n), 1;
    p.once(64, set);
    p.once(64, set);
    p.once(-1, set);
    if (n != 8) return printf("no bit of its own: %d\n", n), 1;
    std::atomic<int> m[32] = {};
    std::vector<std::thread> t;
    for (int i = 0; i < 8; ++i)
        t.emplace_back([&] {
            for (int k = 0; k < 1000; ++k)
                for (int d = 32; d < 63; ++d) p.once(d, [&] { ++m[d - 32]; return true; });
        });
    for (auto &x : t) x.join();
    for (int d = 32; d < 63; ++d)
        if (m[d - 32] < 1 || m[d - 32] > 8) return printf("device %d: %d\n", d, m[d - 32].load()), 1;
    return 0;
}
"""


def test_once_per_device(tmp_path):
    src, exe = tmp_path / "per_device.hip", tmp_path / "per_device"
    src.write_text(PROGRAM)
    subprocess.run(["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "-std=c++17", "-pthread", "-I",
                    os.path.join(si_amd.PKG, "csrc"), "-I", si_amd.INCLUDE_DIR, str(src), "-o",
                    str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


def test_every_lds_limit_is_per_device():
    """No kernel's limit is set but through it."""
    csrc = os.path.join(si_amd.PKG, "csrc")
    calls = [f for f in sorted(os.listdir(csrc))
             for line in open(os.path.join(csrc, f)) if "hipFuncSetAttribute(" in line]
    assert calls == ["si_kernels.hpp"]
