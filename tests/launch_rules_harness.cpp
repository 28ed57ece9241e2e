// launch_rules_harness.cpp -- micm_amd/csrc/launch_rules.hpp for tests/test_launch_rules.py.
#include "../micm_amd/csrc/launch_rules.hpp"

#include <cstdint>

using namespace micm_hip;

extern "C" int tile_cells_host(int64_t doubles_per_cell, int64_t lds_limit)
{
  return tile_cells(static_cast<std::size_t>(doubles_per_cell), static_cast<std::size_t>(lds_limit));
}

extern "C" int with_block_host(int64_t factor, int64_t products, int64_t n_cells, int substitution)
{
  return substitution ? substitution_with_block(factor, products, n_cells) : lu_with_block(factor, products, n_cells);
}

// The slices of n_cells cells as (first, cells) pairs; their number, or -1 past `most` of them.
extern "C" int64_t slices_host(int64_t n_cells, int64_t threads_per_cell, int64_t* out, int64_t most)
{
  int64_t n = 0;
  const int rc = for_slices(n_cells, threads_per_cell, [&](int64_t first, int64_t cells) {
    if (n == most)
      return 1;
    out[2 * n] = first;
    out[2 * n + 1] = cells;
    ++n;
    return 0;
  });
  return rc ? -1 : n;
}

extern "C" int64_t staging_bytes_host(int64_t n_cells, int64_t n_species, int64_t n_reactions)
{
  return static_cast<int64_t>(staging_bytes(n_cells, n_species, n_reactions));
}
