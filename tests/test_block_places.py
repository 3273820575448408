"""Blocks of a colour phase (host only): place_block deals every (replica, block) exactly once, and
all blocks of a replica to one XCD (block index mod 8), but for the last R mod 8 replicas -- for
every replica count, not only multiples of 8."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "espins_amd", "csrc")
PROGRAM = """
#include "esp_geo.h"
#include <cstdio>
#include <vector>
int main() {
  for (int R : {1, 2, 7, 8, 9, 15, 16, 20, 41, 100, 125, 244, 257, 1000})
    for (int nblk : {1, 2, 3, 8, 17, 64, 1025}) {
      const uint32_t full = espg::xcd_full(R, nblk);
      const espg::FastDiv d = espg::make_fastdiv((uint32_t)nblk);
      std::vector<int> seen((size_t)R * nblk, 0), xcd(R, -1);
      for (uint32_t L = 0; L < (uint32_t)(R * nblk); ++L) {
        int r = -1, b = -1;
        espg::place_block(L, full, d, r, b);
        if (r < 0 || r >= R || b < 0 || b >= nblk || seen[(size_t)r * nblk + b]++) return std::printf("R %d nblk %d L %u\\n", R, nblk, L), 1;
        if (r < R / 8 * 8 && xcd[r] >= 0 && xcd[r] != (int)(L % 8)) return std::printf("R %d nblk %d replica %d\\n", R, nblk, r), 1;
        xcd[r] = (int)(L % 8);
      }
    }
  return 0;
}
"""


def test_blocks_of_a_replica_share_an_xcd(tmp_path):
    src, exe = tmp_path / "places.cpp", tmp_path / "places"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
