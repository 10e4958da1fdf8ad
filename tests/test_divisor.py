"""The kernels' division by a fixed divisor (euc_amd/csrc/internal.hpp, Divisor)
against the processor's own, on the CPU: every small pair, the neighbourhoods of
powers of two and of multiples of the divisor, and random pairs up to 2^32 - 1."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <hip/hip_runtime.h>
#include <cstdio>
#include "internal.hpp"
static int check(uint32_t n, uint32_t d, const euchip::Divisor &v) {
    if (euchip::divide(n, v) == n / d) return 0;
    printf("%u / %u: %u\n", n, d, euchip::divide(n, v));
    return 1;
}
int main() {
    int bad = 0;
    uint64_t s = 12345;
    auto rnd = [&] { s = s * 6364136223846793005ull + 1442695040888963407ull; return (uint32_t)(s >> 32); };
    auto some = [&](uint32_t d) {
        const euchip::Divisor v = euchip::make_divisor(d);
        for (uint32_t n = 0; n < 600; n++) bad += check(n, d, v) + check(~n, d, v);
        for (int b = 0; b < 32; b++)
            for (int e = -2; e <= 2; e++) bad += check((1u << b) + e, d, v);
        for (int i = 0; i < 200; i++) {
            const uint32_t n = rnd() >> (rnd() & 31u), m = (uint32_t)(n / d * (uint64_t)d);
            bad += check(n, d, v) + check(m, d, v) + check(m - 1u, d, v) + check(m + d, d, v);
        }
    };
    for (uint32_t d = 1; d < 2000; d++) some(d), some(0u - d);
    for (int b = 0; b < 32; b++)
        for (int e = -2; e <= 2; e++)
            if ((uint32_t)((1u << b) + e)) some((1u << b) + e);
    for (int i = 0; i < 3000; i++) some((rnd() >> (rnd() & 31u)) | 1u);
    return bad != 0;
}
"""


def test_divisor(tmp_path):
    src, exe = tmp_path / "divisor.cpp", tmp_path / "divisor"
    src.write_text(SOURCE)
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-I",
                           os.path.join(ROOT, "euc_amd", "csrc"), str(src), "-o", str(exe)])
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[:500]
