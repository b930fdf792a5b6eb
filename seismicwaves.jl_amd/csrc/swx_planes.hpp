// Planes of a CD 3D row-march chunk and their z C-PML entries: plain integer
// arithmetic, so that a host program can run it over whole ranges of grids.
#pragma once

namespace swx {

// strip index of the cell owning psi along an axis of size n (or -1)
constexpr int psi_owner(int i, int n, int h) {
  if (i < h) return i;
  if (i >= n - h - 1 && i <= n - 2) return i + 1 - n + 2 * h;
  return -1;
}

// z strip entry of a plane that owns a psi_z
constexpr int z_entry(int k, int nz, int h) { return k < h ? k : k + 1 - nz + 2 * h; }

// Most planes per chunk of the row march.  Its plane masks have 64 bits, and a
// plane's fields are loaded up to RM_AHEAD planes after the chunk's last one:
// with more planes their bits would be those of the chunk's first planes (a
// shift counts modulo 64), whose strip entries do not exist there.
constexpr int RM_AHEAD = 2;
constexpr int RM_PLANES = 64 - RM_AHEAD;

}  // namespace swx
