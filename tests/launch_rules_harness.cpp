// launch_rules_harness.cpp -- micm_amd/csrc/launch_rules.hpp for tests/test_launch_rules.py.
#include "../micm_amd/csrc/launch_rules.hpp"

#include <cstdint>

using namespace micm_hip;

extern "C" int tile_cells_host(int64_t doubles_per_cell, int64_t lds_limit)
{
  return tile_cells(static_cast<std::size_t>(doubles_per_cell), static_cast<std::size_t>(lds_limit));
}

extern "C" int lu_tile_cells_host(int64_t doubles_per_cell, int64_t lds_limit)
{
  return lu_tile_cells(static_cast<std::size_t>(doubles_per_cell), static_cast<std::size_t>(lds_limit));
}
