"""Which groups run on tiles of one geometry group (host only): those that fill at least half of the
lanes of their tiles.  A group of 27 sites (FCC 18^3, SC 6^3) leaves 37 lanes of 64 idle and reads the
tables."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "espins_amd", "csrc")
PROGRAM = """
#include "esp_geo.h"
#include <cstdio>
int main() {
  for (int mt = 1; mt <= 4096; ++mt) std::printf("%d %d\\n", espg::tile_count(mt), (int)espg::tiles_serve(mt));
}
"""


def test_tiles_are_at_least_half_full(tmp_path):
    src, exe = tmp_path / "tiles.cpp", tmp_path / "tiles"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split()
    for mt, (n, serve) in enumerate(zip(map(int, out[::2]), map(int, out[1::2])), 1):
        assert n == -(-mt // 64)
        assert serve == (mt / (64 * n) >= 0.5)
    assert not int(out[2 * 26 + 1]) and int(out[2 * 31 + 1])
