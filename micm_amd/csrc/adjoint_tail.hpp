// adjoint_tail.hpp -- the reverse sweep of the discrete adjoint (adjoint.hpp) for mechanisms
// whose factor has a dense block (tail.hpp).
#pragma once

#include "coop_tail.hpp"

namespace micm_hip
{
  // Tables of PackedAdjoint and the lists they are ordered by.
  struct DevAdjointLists
  {
    const int32_t *weight_offsets, *weight_species;
    const double* weight_coef;
    const int32_t *rxn_offsets, *rxn_terms, *rxn_indep;
    const int32_t *indep_offsets, *indep_terms;
    const int32_t* second_offsets;
    const uint64_t* second;
    int32_t n_second;  // < 0: the mechanism has no such tables
  };

  size_t adjoint_tail_lds(const DevMech& m, const DevCoop& c, const DevTail& t, const DevAdjointLists& a, int stages);

  int adjoint_tail_occupancy(size_t lds);

  // Grouped arrays; one workgroup per cell, `blocks` of them.
  hipError_t adjoint_tail(const DevMech& m, const DevCoop& c, const DevTail& t, const DevAdjointLists& a,
                          const DevParams& p, int64_t n_cells, unsigned blocks, size_t lds, const double* k,
                          const Tape& tape, const double* seed, double* grad_y, double* grad_logk, hipStream_t stream);
}  // namespace micm_hip
