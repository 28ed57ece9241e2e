// tiny.hpp -- Solves of the smallest mechanisms, one cell per lane (tiny.hip): those whose columns
// of 64 cells fit kTinyLds.  With four stages that is 4 species and 54 columns for the rate
// constants and for the rates or Jacobian terms (less the lists), 5 species and 39, 6 and 22; none
// of 7 species with more than a reaction or two, none of 8.
#pragma once

#include "device.hpp"
#include "mechanism.hpp"

namespace micm_hip
{
  // TinyTables on the device.
  struct DevTiny
  {
    const TinyEntry* forcing;
    const TinyEntry* jacobian;
    int32_t n_forcing, n_jacobian;  // n_forcing < 0: the mechanism has no such tables
    uint64_t pattern;
  };

  struct TinyArgs
  {
    DevMech m;
    DevCoop c;
    DevTiny t;
    DevParams p;
    int64_t n_cells;  // cells, or the most that `list` holds
    const int32_t* list;
    const int* list_count;
    const CellControl* resume;
    double* y;
    const double* k;
    const double* atol;
    int32_t* status;
    int64_t* stats;
    double* final_time;
  };

  // Dynamic LDS of one wavefront of 64 cells; 0 where the mechanism has no tables (more than
  // kTinySpecies species) or needs more than kTinyLds.
  constexpr size_t kTinyLds = 48 * 1024;
  size_t tiny_lds(const DevMech& m, const DevCoop& c, const DevTiny& t, int stages);

  // Per-cell steps, whatever the number of cells.
  hipError_t tiny_solve(const TinyArgs& a, size_t lds, hipStream_t stream);
  // One step size for all cells, at most 64 (kWave) of them.
  hipError_t tiny_lockstep(const TinyArgs& a, size_t lds, hipStream_t stream);
}  // namespace micm_hip
