"""Plane masks and z strip entries of the CD 3D row march over whole ranges of
grids, halos and chunks (csrc/swx_planes.hpp compiled for the host): every
plane that the march loads for a chunk has a bit of its own in the 64-bit
masks, and the strip entry of every plane whose bit is set is one that exists.
A shift counts modulo 64, as the hardware does it."""
import os
import shutil
import subprocess

import pytest

from conftest import PKG_ROOT

PROGRAM = r"""
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include "swx_planes.hpp"
using namespace swx;
int bad = 0;
void load(uint64_t zown, int k, int K0, int K1, int nz, int h) {
  const int m = k - K0;
  const bool ahead = k < K1 + RM_AHEAD, bit = zown >> (m & 63) & 1;
  const int z = bit ? z_entry(k, nz, h) : 0;
  if (ahead && (!bit || (k < K1 && z >= 0 && z < 2 * h))) return;
  if (!bad++) std::printf("plane %d of chunk %d..%d: nz %d halo %d entry %d\n", k, K0, K1, nz, h, z);
}
int main() {
  for (int set : {1, 2, 3, 6, 12, 61, 62, 63, 64, 100})
    for (int h = 0; h <= 40; h++)
      for (int nz = 2 * h + 3; nz <= 2 * h + 200; nz++) {
        const int kch = std::min(set, RM_PLANES);
        for (int K0 = 0; K0 < nz; K0 += kch) {
          const int K1 = std::min(K0 + kch, nz);
          uint64_t zown = 0;
          for (int l = 0; l < 64; l++)
            if (K0 + l < K1 && psi_owner(K0 + l, nz, h) >= 0) zown |= uint64_t(1) << l;
          // the loads of the march, in its order
          load(zown, K0, K0, K1, nz, h);
          load(zown, K0 + 1, K0, K1, nz, h);
          for (int k = K0; k < K1; k += 3) {
            load(zown, k + 2, K0, K1, nz, h);
            if (k + 1 >= K1) break;
            load(zown, k + 3, K0, K1, nz, h);
            if (k + 2 >= K1) break;
            load(zown, k + 4, K0, K1, nz, h);
          }
        }
      }
  if (bad) std::printf("%d loads out of range\n", bad);
  return bad != 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_row_march_loads_only_strip_entries_that_exist(tmp_path):
    src, exe = tmp_path / "planes.cpp", tmp_path / "planes"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", f"-I{os.path.join(PKG_ROOT, 'csrc')}", str(src), "-o", str(exe)],
                   check=True, timeout=120)
    r = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
