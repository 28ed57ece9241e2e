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

  // Whether the single-phase LU (substitution) takes the kernel with the factor's dense block, one
  // cell per workgroup, rather than the tiled one.  Up to kTailCells cells, the workgroups that
  // three to a CU hold at once, the block does: a tile of many cells leaves most CUs idle.  With
  // more cells it does for factors of at least kTailFactor entries and kTailProducts products,
  // whose work the block's rows hold; sparser ones gain by it only where a CU holds few of their
  // tiles: the LU from 1,650 entries (tiles of four, two to a CU) and 2,048 cells on, the
  // substitution from 1,280 entries and 3,600 products on.  LU / substitution, us, block against
  // tiled:
  //   16 species (131 entries), 768 cells 12.5 : 14.5 / 8.1 : 15.8, 1,500 cells 17.4 : 14.5 / 11.0 : 15.7;
  //   20 (165), 768 cells 16.5 : 16.6 / 11.7 : 16.9; 50 (919), 1,500 41 : 51 / 34 : 52, 20,000 318 : 312 / 315 : 282
  //   160 (1,252, 1,882 products), 1,500 48 : 47 / 42 : 37, 4,096 99 : 64 / 95 : 84
  //   120 (1,417, 4,291), 1,500 54 : 47 / 41 : 49, 8,000 192 : 158 / 167 : 174
  //   200 (1,697, 3,653), 1,500 56 : 46 / 48 : 60, 2,500 77 : 97 / 71 : 120
  //   60/200 (1,304, 7,668), 1,500 45 : 54 / 36 : 69, 20,000 382 : 439 / 347 : 456
  //   TS1 (2,381, 6,986), 4,096 122 : 163 / 105 : 222; 210/560 (8,548, 121,036), 4,096 525 : 1,654 / 344 : 1,307
  constexpr int64_t kTailCells = 768, kTailFactor = 1200, kTailProducts = 6000;

  constexpr bool lu_with_block(int64_t factor, int64_t products, int64_t n_cells)
  {
    return n_cells <= kTailCells || (factor >= kTailFactor && products >= kTailProducts) ||
           (factor >= 1650 && n_cells > 2048);
  }

  constexpr bool substitution_with_block(int64_t factor, int64_t products, int64_t n_cells)
  {
    return n_cells <= kTailCells || (factor >= kTailFactor && products >= kTailProducts) ||
           (factor >= 1280 && products >= 3600);
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
