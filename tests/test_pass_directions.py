"""Passes that exist for some directions only refuse the others: asked dry (no
launch, no GPU) through the library's own launchers."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "shock-turbulence_amd")

SRC = r"""
#include "st_kernels.h"
#include <cstdio>
#include <cstring>
int main()
{
    using namespace st;
    DirTab t;
    std::memset(&t, 0, sizeof(t));
    t.n = 32;
    t.M = 4;
    t.P = 8;
    PassArgs a;
    std::memset(&a, 0, sizeof(a));
    a.dry = 1;
    a.ni = a.N = 32768;
    a.nslot = 1;
    RaggedSpec sp;
    std::memset(&sp, 0, sizeof(sp));                   // no member: no launch
    const int kinds[] = {K_GRAD, K_GRAD_CROSS, K_FQ_GRAD, K_GAUSS_ETA_LAST, K_HDIV, K_HDIV_RKF};
    for (int k : kinds)
        for (int d = 0; d < 3; d++) {
            sp.dir = d;
            printf("%d%d ", run_pass(k, t, 256, d, 32, 32, 32, a, nullptr) == hipSuccess,
                   run_pass_ragged(k, sp, nullptr) == hipSuccess);
        }
    return 0;
}
"""


def test_directions(tmp_path):
    src, exe = tmp_path / "d.cpp", tmp_path / "d"
    src.write_text(SRC)
    subprocess.run(["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-arch=gfx950", "-std=c++17", "-I",
                    os.path.join(PKG, "csrc"), str(src), "-x", "none", os.path.join(PKG, "libst.so"),
                    "-Wl,-rpath," + PKG, "-o", str(exe)], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    got = [r.stdout.split()[3 * k:3 * k + 3] for k in range(6)]
    yes, no = "11", "00"
    assert got == [[yes, no, yes],               # x and z gradients
                   [no, yes, no],                # y gradients
                   [yes, no, no],                # x filter with x gradients
                   [no, no, yes],                # z Gaussian with the fluxes and their z divergence
                   [yes, yes, no],               # x and y divergence of the stored fluxes
                   [yes, yes, no]], got
