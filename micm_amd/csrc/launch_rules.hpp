// launch_rules.hpp -- sizes of launches and workspaces as plain functions of their arguments.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

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

  // A launch takes fewer than 2^32 threads; of more, HIP runs the number modulo 2^32 and reports
  // nothing.  Cells are therefore launched in slices of at most kMostThreads threads, whole
  // groups of 64 cells for each of the eight XCDs.
  constexpr int64_t kMostThreads = int64_t(1) << 31;
  constexpr int64_t kSliceCells = 512;
  constexpr int64_t slice_cells(int64_t threads_per_cell)
  {
    return std::max(kMostThreads / std::max<int64_t>(threads_per_cell, 1) / kSliceCells, int64_t(1)) * kSliceCells;
  }

  // launch(first cell, cells) over n_cells cells in slices, until one returns other than 0.
  template<class Launch>
  int for_slices(int64_t n_cells, int64_t threads_per_cell, const Launch& launch)
  {
    const int64_t most = slice_cells(threads_per_cell);
    for (int64_t first = 0; first < n_cells; first += most)
      if (const int rc = launch(first, std::min(most, n_cells - first)))
        return rc;
    return 0;
  }

  // Results of one cell on the host: seven counters, the final time and the status.
  constexpr std::size_t kResultBytes = 7 * sizeof(int64_t) + sizeof(double) + sizeof(int32_t);
  constexpr std::size_t kStagingMost = 256 * 1024;

  // Grouped arrays go through pinned memory below this size only: a copy to pageable memory takes
  // 21 us up to 16 KiB and 11 from there on, and the host reads the pinned buffer more slowly
  // (pageable / pinned, us: 10 KiB 21 / 13, 17 KiB 11.2 / 12.5, 80 KiB 15 / 22, 240 KiB 26 / 46).
  constexpr std::size_t kStagingGrouped = 16 * 1024;

  // Pinned memory of a State for its copies to the host: the largest of the results (three copies
  // in one wait) up to kStagingMost and of the variables and the rate constants (in whole groups
  // of 64 cells) below kStagingGrouped; 0 where none is, so that a State of many cells has none.
  constexpr std::size_t staging_bytes(int64_t n_cells, int64_t n_species, int64_t n_reactions)
  {
    const std::size_t cells = static_cast<std::size_t>(n_cells), padded = (cells + 63) / 64 * 64;
    const std::size_t results = cells * kResultBytes;
    const std::size_t variables = padded * sizeof(double) * static_cast<std::size_t>(n_species);
    const std::size_t rates = padded * sizeof(double) * static_cast<std::size_t>(n_reactions);
    std::size_t bytes = results <= kStagingMost ? results : 0;
    for (std::size_t copy : { variables, rates })
      if (copy < kStagingGrouped)
        bytes = std::max(bytes, copy);
    return bytes;
  }
}  // namespace micm_hip
