"""The RK launch's default residency in waves (bg_internal.h): compiled and run
on the host.  The block size does not change how many waves a CU holds, except
that blocks of two waves go from three to four per SIMD."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <cstdio>
#include "bacon_amd/csrc/bg_internal.h"
int main() {
    for (uint32_t block : {64u, 128u, 192u, 256u})
        printf("%u %u %u\n", block, bg::blocks_of_waves(bg::kRkWavesFew, block),
               bg::blocks_of_waves(bg::kRkWavesMany, block));
    for (bool arrays : {false, true})
        for (unsigned long long n : {1ull, 131072ull, 131073ull, 262144ull, 262145ull}) {
            bool look = false;
            const uint32_t w = bg::rk_default_waves(arrays, n, 256, look);
            printf("%d %llu %u %d\n", (int)arrays, n, w, (int)look);
        }
}
"""


def test_default_residency(tmp_path):
    src, exe = tmp_path / "rule.cpp", tmp_path / "rule"
    src.write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-w",
                    f"-I{ROOT}", "-o", str(exe), str(src)], check=True, timeout=100)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=20).stdout.split("\n")
    rows = [tuple(int(x) for x in r.split()) for r in out if r]
    for block, few, many in rows[:4]:
        assert abs(few * block // 64 - 8) <= 1  # 192: nine waves
        assert many * block // 64 == (16 if block == 128 else 12)
    for arrays, n, waves, look in rows[4:]:
        assert look == (arrays and 131072 < n <= 262144)
        assert waves == (8 if arrays and not look else 12)
