// coop_tail.hpp -- the cooperative Solve of mechanisms of 16 to 256 species with the factor's
// last rows as a dense block (coop_tail.hip), as the launch code sees it.
#pragma once

#include "device.hpp"

namespace micm_hip
{
  constexpr int kTailThreads = 256;
  // Doubles of LDS that the block's factorisation uses besides the factor: two buffers of a
  // pivot row and a pivot column.
  constexpr int kTailBuffer = 4 * 64;

  __host__ __device__ inline size_t tail_scratch_doubles(int n, int n_reactions, int n_terms)
  {
    int scratch = kTailBuffer;
    if (n_reactions > scratch)
      scratch = n_reactions;
    if (n_terms > scratch)
      scratch = n_terms;
    const int padded = (n + 16 - 1) / 16 * 16;
    return static_cast<size_t>(scratch > padded ? scratch : padded);
  }
  // y starts at an even position, so that the scratch area (16-byte accesses) does too
  __host__ __device__ inline size_t tail_lds_doubles(int nnz, int n, int n_reactions, int n_terms)
  {
    return ((static_cast<size_t>(nnz) + 1 + 2 * static_cast<size_t>(n) + 1 + 1) & ~size_t(1)) +
           tail_scratch_doubles(n, n_reactions, n_terms);
  }

  struct CoopTailArgs
  {
    DevMech m;
    DevCoop c;
    DevTail t;
    DevParams p;
    int64_t n_fixed;  // cells, without a list
    const int32_t* list;
    const int* list_count;
    int* next;  // queue counter, zeroed before the launch
    const CellControl* resume;
    double* y;
    const double* k;
    const double* atol;
    int32_t* status;
    int64_t* stats;
    double* final_time;
    double* k_rows;  // gridDim.x rows of n_reactions
    Tape tape;       // records null: not recorded
  };

  // Workgroups per CU of the build for min_waves waves per SIMD (3 or 2), 0 where it does not fit.
  int coop_tail_occupancy(int min_waves, size_t lds);
  hipError_t coop_tail_launch(int min_waves, unsigned blocks, size_t lds, hipStream_t stream, const CoopTailArgs& a);

  // The single phases with the block, one cell per workgroup (`blocks`: whole groups of cells
  // for every XCD), and their LDS.
  size_t tail_factor_lds(const DevTail& t);
  size_t tail_solve_lds(const DevMech& m, const DevTail& t);
  hipError_t lu_decompose_tail(const DevMech& m, const DevTail& t, int64_t n_cells, unsigned blocks, const double* jac,
                               double* lower, double* upper, hipStream_t stream);
  hipError_t lu_solve_tail(const DevMech& m, const DevTail& t, int64_t n_cells, unsigned blocks, const double* lower,
                           const double* upper, double* x, hipStream_t stream);
}  // namespace micm_hip
