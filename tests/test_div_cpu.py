"""Quotients by a multiplication (QW_DIV_MUL of kernels/qw_kargs.h, qw_div of the kernels): exact wherever x * d < 2^32."""
import os
import subprocess

from qwental_amd import build

SOURCE = r"""
#include "qw_kargs.h"
#include <stdio.h>
int main(void) {
    for (uint64_t d = 2; d < 65536; d = d < 5000 ? d + 1 : d + 61) {
        const uint32_t mul = QW_DIV_MUL((uint32_t)d), top = (uint32_t)(((1ull << 32) - 1) / d);
        for (uint32_t q = 0; q * d < top; q = q < 64 ? q + 1 : q + 1 + q / 3) // both sides of multiples of d
            for (int e = -1; e < 2; e++) {
                const uint64_t x = q * d + (uint64_t)e;
                if (x < top && (uint32_t)((x * mul) >> 32) != x / d) return printf("%llu / %llu\n", (unsigned long long)x, (unsigned long long)d), 1;
            }
        if ((uint32_t)(((uint64_t)(top - 1) * mul) >> 32) != (top - 1) / d) return printf("%u / %llu\n", top - 1, (unsigned long long)d), 1;
    }
    return 0;
}
"""


def test_quotients(tmp_path):
    src = tmp_path / "div.c"
    src.write_text(SOURCE)
    exe = str(tmp_path / "div")
    subprocess.run(["gcc", "-O2", "-include", "stdint.h", "-I", os.path.join(build.CSRC, "kernels"), str(src), "-o", exe], check=True)
    r = subprocess.run([exe], stdout=subprocess.PIPE, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
