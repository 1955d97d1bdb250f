"""The threads that share host copies (csrc/st_copiers.h, plain C++): every
byte at the sizes where the shares change, pieces that follow each other at
once and after pauses around the polling time, and no processor time taken
while a transfer waits for the device."""
import os
import subprocess

import pytest

HDR = os.path.join(os.path.dirname(__file__), "..", "shock-turbulence_amd", "csrc", "st_copiers.h")

SRC = r"""
#include "%s"
#include <cstdio>
#include <cstdlib>
#include <vector>
#include <sys/resource.h>

static double cpu()
{
    rusage r;
    getrusage(RUSAGE_SELF, &r);
    return r.ru_utime.tv_sec + r.ru_stime.tv_sec + 1e-6 * (r.ru_utime.tv_usec + r.ru_stime.tv_usec);
}

static void nap(int us) { std::this_thread::sleep_for(std::chrono::microseconds(us)); }

int main()
{
    const size_t most = (2 << 20) + 77;
    std::vector<unsigned char> a(most), b(most + 2);
    unsigned r = 1;
    for (auto &x : a) x = (unsigned char)((r = r * 1664525u + 1013904223u) >> 24);
    st::Copiers c;
    const size_t sizes[] = {0, 1, 63, 64, 65, 319, 320, 321, 4095, 65536, (1 << 20) + 1, 2 << 20, most};
    for (int pause : {0, 20, 90, 100, 110, 1000})
        for (int k = 0; k < 30; k++)
            for (size_t n : sizes) {
                std::memset(b.data(), 0, n + 2);
                if (pause && k %% 3 == 0) c.wake();
                if (pause && k < 5) nap(pause);
                c.copy(b.data() + 1, a.data(), n);
                if (std::memcmp(b.data() + 1, a.data(), n) || b[0] || b[n + 1]) return 2;
            }
    c.wake();                                   // a transfer that waits for the device
    const double t = cpu();
    nap(500000);
    const double used = cpu() - t;
    c.copy(b.data(), a.data(), most);
    printf("%%.4f\n", used);
    return std::memcmp(b.data(), a.data(), most) ? 3 : 0;
}
"""


def test_copies_and_idle_time(tmp_path):
    src, exe = tmp_path / "c.cpp", tmp_path / "c"
    src.write_text(SRC % os.path.abspath(HDR))
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-pthread", str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.returncode
    # up to four threads polling for half a second would take 2 s; 100 us each are allowed
    assert float(r.stdout) < 0.1, r.stdout
