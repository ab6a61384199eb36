/*
 * bdem_grid.hpp - which grids list a contact the same number of times from
 * both bodies (internal; plain C++).
 */
#pragma once

namespace bdem {

/* The cell hash x + z nz + y nx nz (Collision_Detection_BroadPhase.cuh:42-50)
 * is one number for two cells where nx and nz differ or are small, so a
 * stencil row may hold the particles of a cell that is not in it: a partner
 * is then listed twice, or by one body of a pair only.  True when no two
 * cells that are near enough to matter share a hash: the cells of two bodies
 * in contact are at most `reach` apart in each direction, a stencil row at
 * most one, so offsets up to reach + 1 are tried.  Then a particle's rows are
 * disjoint and hold a contact partner's cell if and only if it is one of the
 * 27; what remains one-sided are rows cut off at the end of the cell table,
 * which concern keys in its last two cells and beyond only. */
inline bool hash_is_local(int nx, int ny, int nz, int reach) {
  if (reach < 1 || reach > 8) return false;
  const int k = reach + 1;
  const int kx = k < nx - 1 ? k : nx - 1, ky = k < ny - 1 ? k : ny - 1, kz = k < nz - 1 ? k : nz - 1;
  for (int y = 0; y <= ky; ++y)   /* offsets come in pairs of opposite sign */
    for (int z = -kz; z <= kz; ++z) {
      const long long h = (long long)z * nz + (long long)y * nx * nz;
      if ((y != 0 || z != 0) && h >= -kx && h <= kx) return false;
    }
  return true;
}

/* Cells between two bodies in contact, at most: for spheres (or bounding
 * spheres) of radius up to rmax, with a hundredth of a cell for rounding.  0
 * when that is no small number. */
inline int contact_reach(float rmax, float cell_x, float cell_y, float cell_z) {
  const float c = cell_x < cell_y ? (cell_x < cell_z ? cell_x : cell_z) : (cell_y < cell_z ? cell_y : cell_z);
  const float q = 2.0f * rmax / c;
  return q >= 0.0f && q < 7.0f ? (int)(q + 0.01f) + 1 : 0;
}

}  // namespace bdem
