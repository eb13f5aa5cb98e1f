"""How the launchers keep within what one launch takes (crumpet_common.h),
compiled for the host with g++."""

from __future__ import annotations

import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]

PROGRAM = r"""
#include <cstdio>
#include <cstdint>
#include "crumpet_common.h"
int main() {
    using namespace crumpet;
    // 256 threads: 2^24 - 1 workgroups fit 32 bits of threads, 2^24 do not
    if (!launch_takes((1u << 24) - 1, 256) || launch_takes(1u << 24, 256) || !launch_takes(0, 256)) return 1;
    if (launch_takes(uint64_t(1) << 40, 256)) return 2;
    const uint64_t sizes[] = {1, 2, 4095, (1u << 20) - 1, 1u << 20, (1u << 20) + 1, (1u << 24) - 1, 1u << 24,
                              123456789, (1u << 29) - 1, 1u << 29};
    for (uint64_t n : sizes) {
        const GridXY g = grid_xy(n);
        const uint64_t all = uint64_t(g.x) * g.y;
        if (!launch_takes(g.x, 256) || g.y > 65535 || all < n || all - n >= g.x) return 3;
        if (n <= (1u << 20) && (g.x != n || g.y != 1)) return 4;  // as one row: no idle workgroups
        // row numbers stay within 32 bits: 4 rows a workgroup at 2^29 of them
        if (all * 4 >= (uint64_t(1) << 32)) return 5;
    }
    printf("OK\n");
    return 0;
}
"""


def test_launches_stay_within_32_bits_of_threads(tmp_path):
    src = tmp_path / "limits.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "limits"
    subprocess.check_call(["g++", "-O2", "-std=c++17", f"-I{ROOT / 'crumpet_amd' / 'csrc'}", str(src), "-o", str(exe)])
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.startswith("OK"), out.returncode
