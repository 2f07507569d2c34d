"""The edge-line queue's entries (csrc/line_entry.h) hold any point of a cloud:
what a point and a side are packed to gives both back, beyond 2^30 points too."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "openholo_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include "line_entry.h"
int main()
{
    const int64_t points[] = {0, 1, 63, (1ll << 30) - 1, 1ll << 30, (1ll << 31) - 1, 1ll << 31, (1ll << 32) + 5,
                              (1ll << 40) + 7};
    int bad = 0;
    for (int64_t p : points)
        for (int side = 0; side < 2; ++side) {
            const auto e = ohx::line_entry(p, side);
            if (ohx::line_point(e) != p || ohx::line_side(e) != side) {
                std::printf("point %lld side %d: %lld %d\n", (long long)p, side, (long long)ohx::line_point(e),
                            ohx::line_side(e));
                ++bad;
            }
        }
    return bad != 0;
}
"""


def test_entries_hold_any_point(tmp_path):
    src, exe = tmp_path / "entries.cpp", tmp_path / "entries"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
