// launch_rules.hpp -- sizes of launches and workspaces as plain functions of their arguments.
#pragma once

#include <cstddef>

namespace micm_hip
{
  // Cells per workgroup of the tiled LU / substitution kernels: the largest power of
  // two up to 16 whose tile of `doubles_per_cell` leaves room for two workgroups per CU
  // (two independent workgroups hide each other's level latency: 210/560 LU 1.4x,
  // 60/200 2.1x against one workgroup of twice the cells), else one cell if it fits;
  // 0 when one cell does not fit.
  constexpr int tile_cells(std::size_t doubles_per_cell, std::size_t lds_limit)
  {
    for (int tc = 16; tc >= 1; tc /= 2)
      if (2 * doubles_per_cell * tc * sizeof(double) <= lds_limit)
        return tc;
    return doubles_per_cell * sizeof(double) <= lds_limit ? 1 : 0;
  }

  // The same for the LU kernel, which is built for tiles of 16 cells, 8 and 1 (kLuTiles): with
  // 160 KB of LDS, factors whose tiles would have 4 or 2 cells (1,281 entries and more) take the
  // kernel with the dense block, and those that cannot run one cell at a time.
  constexpr int kLuTiles[] = { 16, 8, 1 };
  constexpr int lu_tile_cells(std::size_t doubles_per_cell, std::size_t lds_limit)
  {
    const int most = tile_cells(doubles_per_cell, lds_limit);
    for (int tc : kLuTiles)
      if (tc <= most)
        return tc;
    return 0;
  }
}  // namespace micm_hip
