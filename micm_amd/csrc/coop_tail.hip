// coop_tail.hip -- the cooperative Solve of mechanisms of 16 to 256 species: one workgroup of
// 256 threads per cell, the factor's last rows as a dense block (tail.hpp).
#include "coop_tail.hpp"

#include "path.hpp"
#include "tail.hpp"

namespace micm_hip
{
namespace
{
  // a value that all lanes hold, as one in scalar registers
  __device__ __forceinline__ double uniform(double v)
  {
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                            __builtin_amdgcn_readfirstlane(__double2loint(v)));
  }

  // LDS holds what other threads read: the factor (head, block, zero), y, one vector x (stage
  // inputs, right-hand sides and solutions, x[n] = 0) and a scratch area shared in time by
  // the reaction rates, the Jacobian's partial products, the block's pivots and the error
  // terms.  Thread i keeps species i's stage vectors, f(y) and accumulated Jacobian diagonal
  // in registers; rate constants are read from a per-workgroup copy in global memory.
  //
  // Bound by the dependency chain of one attempt.  An attempt of the slowest cell, two waves
  // per SIMD, against the level-scheduled compact layout it replaced: 210/560 366 -> 128 us,
  // 60/200 110 -> 45 us, TS1 190 -> 69 us.
  template<int MINW, bool RECORD>
  __global__ void __launch_bounds__(kTailThreads, MINW)
      k_coop_tail(DevMech m, DevCoop c, DevTail t, DevParams p, int64_t n_fixed, const int32_t* __restrict__ list,
                  const int* list_count, int* next, const CellControl* resume, double* __restrict__ y_state,
                  const double* __restrict__ k_state, const double* __restrict__ atol, int32_t* status_out,
                  int64_t* stats_out, double* final_time_out, double* __restrict__ k_wg, Tape tape)
  {
    constexpr int NT = kTailThreads;
    extern __shared__ double lds[];
    __shared__ int s_idx;
    __shared__ int s_flags[NT / kWave];
    const int tid = threadIdx.x;
    const int n = m.n_species;
    const bool mine = tid < n;  // this thread has a species
    CoopLds L{};
    L.alu = lds;
    L.y = lds + t.nnz + 1;
    double* const x = L.y + n;
    L.scratch = lds + ((static_cast<size_t>(t.nnz) + 1 + 2 * static_cast<size_t>(n) + 1 + 1) & ~size_t(1));
    L.jterm = L.scratch;
    L.k = k_wg + static_cast<size_t>(blockIdx.x) * m.n_reactions;
    c.jac_to_alu = t.jac_pos;
    const int64_t count = list ? static_cast<int64_t>(*list_count) : n_fixed;
    const int diag = mine ? t.diag_pos[tid] : 0;
    const double atol_r = mine ? atol[tid] : 1.0;
    const int sum_groups = (n + kTailBlock - 1) / kTailBlock;
    RowsAhead ahead = rows_ahead(t.rows);
    double one = 1.0;
    asm("" : "+v"(one));
    while (true)
    {
      if (tid == 0)
        s_idx = atomicAdd(next, 1);
      coop_sync<NT>();
      const int64_t idx = __builtin_amdgcn_readfirstlane(s_idx);
      coop_sync<NT>();
      if (idx >= count)
        return;
      const int64_t cell = list ? list[idx] : idx;
      const size_t g = cell / kGroup;
      const int cl = cell % kGroup;
      {
        Lane ys = lane_view(y_state, g, n, cl);
        Lane ks = lane_view(const_cast<double*>(k_state), g, m.n_reactions, cl);
        if (mine)
          L.y[tid] = ys[tid];
        if (tid == 0)
          x[n] = 0.0;
        for (int r = tid; r < m.n_reactions; r += NT)
          L.k[r] = ks[r];
      }
      CellControl cc;
      if (resume)
        cc = resume[cell];
      else
        control_init(p, cc);
      // recorded Solve: the cell's checkpoints are appended to its tape
      int64_t n_rec = RECORD ? tape.counts[cell] : 0;
      double* const rec_base =
          RECORD ? tape.records + static_cast<size_t>(cell) * tape.max_records * (static_cast<size_t>(n) + 1) : nullptr;
      auto record = [&](double tag) {
        if (n_rec < tape.max_records)
        {
          double* rec = rec_base + static_cast<size_t>(n_rec) * (static_cast<size_t>(n) + 1);
          if (tid == 0)
            rec[0] = tag;
          if (mine)
            rec[1 + tid] = L.y[tid];
        }
        ++n_rec;
      };
      coop_sync<NT>();
      double f0 = 0.0, jdiag = 0.0;
      while (true)
      {
        bool fresh = false;
        if (cc.flags & kNewStep)
        {
          if (!begin_step(p, cc))
            break;
          f0 = coop_forcing_own<NT>(m, c, L, L.y);
          coop_sync<NT>();
          cc.stats[MICM_HIP_STAT_FUNCTION_CALLS] += 1;
          cc.stats[MICM_HIP_STAT_JACOBIAN_UPDATES] += 1;
          cc.last_alpha = 0.0;
          cc.flags &= ~kNewStep;
          fresh = true;
        }
        const double alpha = next_alpha(p, cc);
        // -J(y) again (y and k are those of the step), its diagonal replaced by the
        // accumulated one: the same values as keeping -J and adding alpha in place
        for (int q = tid; q <= t.nnz; q += NT)
          L.alu[q] = 0.0;
        coop_jacobian<NT, true>(m, c, L);
        if (mine)
        {
          if (fresh)
            jdiag = L.alu[diag];
          jdiag += alpha * 1.0;
          L.alu[diag] = jdiag;
        }
        coop_sync<NT>();
        coop_levels_piped<NT, true>(t.lu, t.lu.terms, L.alu, L.alu, L.alu);
        const bool masked = __builtin_amdgcn_readfirstlane(!tail_factor<false>(t, L.alu, L.scratch, s_flags));
        if (masked)
          tail_factor_masked(t, L.alu);
        cc.stats[MICM_HIP_STAT_DECOMPOSITIONS] += 1;
        // stage vectors of this thread's species (indexed by unrolled loops only)
        double K[6] = { 0.0, 0.0, 0.0, 0.0, 0.0, 0.0 };
        double f = f0;
        const double y_r = mine ? L.y[tid] : 0.0;
        for (int s = 0; s < p.stages; ++s)
        {
          const int sc = s * (s - 1) / 2;
          if (s > 0 && p.new_f[s])
          {
            double v = y_r;
#pragma unroll
            for (int j = 0; j < 5; ++j)
              if (j < s)
                v += p.a[sc + j] * K[j];
            if (mine)
              x[tid] = v;
            coop_sync<NT>();
            f = coop_forcing_own<NT>(m, c, L, x);
            cc.stats[MICM_HIP_STAT_FUNCTION_CALLS] += 1;
          }
          double v = f;
#pragma unroll
          for (int j = 0; j < 5; ++j)
            if (j < s)
              v += (p.c[sc + j] / cc.H) * K[j];
          if (mine)
            x[tid] = v;
          coop_sync<NT>();
          tail_solve(t, L.alu, x, masked, ahead);
          const double Ks = mine ? x[tid] : 0.0;
#pragma unroll
          for (int j = 0; j < 6; ++j)
            K[j] = j == s ? Ks : K[j];
          cc.stats[MICM_HIP_STAT_SOLVES] += 1;
        }
        double ynew = y_r, e = 0.0;
#pragma unroll
        for (int s = 0; s < 6; ++s)
          if (s < p.stages)
            ynew += p.m[s] * K[s];
#pragma unroll
        for (int s = 0; s < 6; ++s)
          if (s < p.stages)
            e += p.e[s] * K[s];
        if (tid < sum_groups * kTailBlock)
        {
          const double a = fabs(y_r), b = fabs(ynew);
          const double q = e / (atol_r + p.rtol * (a > b ? a : b));
          L.scratch[tid] = mine ? q * q : 0.0;
        }
        coop_sync<NT>();
        // every wavefront adds the terms in species order
        double acc = 0.0;
        {
          const double* terms = L.scratch + (tid & (kTailBlock - 1));
          double q = terms[0];
          for (int h = 0; h < sum_groups; ++h)
          {
            const double qn = terms[kTailBlock * (h + 1 < sum_groups ? h + 1 : h)];
            acc = ordered_sub16<0>(acc, q, one);
            q = qn;
          }
        }
        acc = uniform(acc);
        const double error = smax(sqrt(acc / static_cast<double>(n > 0 ? n : 1)), 1.0e-10);
        const double h_used = cc.H;
        if (control_update(p, cc, error))
        {
          if constexpr (RECORD)
            record(h_used);
          if (mine)
            L.y[tid] = ynew;
        }
        coop_sync<NT>();
        if (cc.status != MICM_HIP_STATE_RUNNING)
          break;
      }
      if constexpr (RECORD)
      {
        record(kClampTag);
        if (tid == 0)
          tape.counts[cell] = n_rec;
      }
      if (mine)
      {
        Lane ys = lane_view(y_state, g, n, cl);
        ys[tid] = smax(L.y[tid], 0.0);
      }
      if (tid == 0)
      {
        status_out[cell] = cc.status;
        for (int i = 0; i < 7; ++i)
          stats_out[cell * 7 + i] = cc.stats[i];
        final_time_out[cell] = cc.t;
      }
      coop_sync<NT>();
    }
  }

  // ---- single phases with the dense block, one cell per workgroup.  The cells of one group
  // go to one XCD one after another and share the group's 128-byte lines in its L2 (workgroup b
  // runs on XCD b % 8).
  __device__ __forceinline__ bool cell_of_block(int64_t n_cells, size_t& g, int& cl)
  {
    constexpr unsigned kXcds = 8;
    const unsigned x = blockIdx.x % kXcds, j = blockIdx.x / kXcds;
    const int64_t grp = static_cast<int64_t>(j / kGroup) * kXcds + x;
    g = static_cast<size_t>(grp);
    cl = static_cast<int>(j % kGroup);
    return grp * kGroup + cl < n_cells;
  }

  // A[map[p]] = src[p] of the cell for map[p] >= 0, eight loads in flight per thread; true on
  // the threads that saw a -0.
  __device__ __forceinline__ bool load_cell(double* A, const int32_t* map, const double* __restrict__ src, size_t g, int cl,
                                            int n)
  {
    constexpr int NT = kTailThreads;
    const double* base = src + g * static_cast<size_t>(n) * kGroup + cl;
    bool negative_zero = false;
    for (int p0 = threadIdx.x; p0 < n; p0 += 8 * NT)
    {
      double v[8];
      int to[8];
#pragma unroll
      for (int j = 0; j < 8; ++j)
      {
        const int p = p0 + j * NT < n ? p0 + j * NT : p0;
        v[j] = base[static_cast<size_t>(p) * kGroup];
        to[j] = map ? map[p] : p;
      }
#pragma unroll
      for (int j = 0; j < 8; ++j)
      {
        negative_zero = negative_zero || (v[j] == 0.0 && __builtin_signbit(v[j]));
        if (p0 + j * NT < n && to[j] >= 0)
          A[to[j]] = v[j];
      }
    }
    return negative_zero;
  }

  // Whether any thread of the workgroup says so; ends with a barrier.
  __device__ __forceinline__ bool any_thread(bool v, int* flags)
  {
    const uint64_t who = __ballot(v);
    if ((threadIdx.x & (kWave - 1)) == 0)
      flags[threadIdx.x / kWave] = who != 0;
    __syncthreads();
    const bool any = (flags[0] | flags[1] | flags[2] | flags[3]) != 0;
    __syncthreads();
    return any;
  }

  // LuDecompositionDoolittle::Decompose for one cell (lu_decomposition_doolittle.inl:325-403).
  // Bound as the Solve's factorisation is by its chain, not by the 87 KB a 210/560 cell reads
  // and writes: 4,096 cells in 525 us, 1,654 with the level schedule alone.
  __global__ void __launch_bounds__(kTailThreads, 2)
      k_lu_decompose_tail(DevMech m, DevTail t, int64_t n_cells, const double* __restrict__ jac,
                          double* __restrict__ lower, double* __restrict__ upper)
  {
    constexpr int NT = kTailThreads;
    extern __shared__ double lds[];
    __shared__ int s_flags[NT / kWave];
    size_t g;
    int cl;
    if (!cell_of_block(n_cells, g, cl))
      return;
    const int tid = threadIdx.x;
    double* A = lds;
    double* buf = lds + ((static_cast<size_t>(t.nnz) + 2) & ~size_t(1));
    for (int q = tid; q <= t.nnz; q += NT)
      A[q] = 0.0;
    __syncthreads();
    const bool exact = any_thread(load_cell(A, t.jac_pos, jac, g, cl, m.nnz_jac), s_flags);
    coop_levels_piped<NT, true>(t.lu, t.lu.terms, A, A, A);
    if (exact || !tail_factor<true>(t, A, buf, s_flags))
      tail_factor_masked(t, A);
    double* lo = lower + g * static_cast<size_t>(m.nnz_lower) * kGroup + cl;
    for (int p = tid; p < m.nnz_lower; p += NT)
    {
      const int a = t.lower_pos[p];
      lo[static_cast<size_t>(p) * kGroup] = a >= 0 ? A[a] : 1.0;
    }
    double* up = upper + g * static_cast<size_t>(m.nnz_upper) * kGroup + cl;
    for (int p = tid; p < m.nnz_upper; p += NT)
      up[static_cast<size_t>(p) * kGroup] = A[t.upper_pos[p]];
  }

  // LinearSolver::Solve for one cell (linear_solver.inl:235-294), dividing by L[i][i] as the
  // reference does where it is not 1.  210/560, 4,096 cells: 344 us, 1,307 with the level
  // schedules alone.
  __global__ void __launch_bounds__(kTailThreads, 2)
      k_lu_solve_tail(DevMech m, DevTail t, int64_t n_cells, const double* __restrict__ lower,
                      const double* __restrict__ upper, double* __restrict__ xs)
  {
    constexpr int NT = kTailThreads;
    extern __shared__ double lds[];
    __shared__ int s_flags[NT / kWave];
    size_t g;
    int cl;
    if (!cell_of_block(n_cells, g, cl))
      return;
    const int tid = threadIdx.x;
    const int n = m.n_species;
    double* A = lds;
    double* x = A + t.nnz + 1;
    double* ld = x + n + 1;
    RowsAhead ahead = rows_ahead(t.rows);
    // the block's structural zeros and the zero behind it
    for (int q = t.head + tid; q <= t.nnz; q += NT)
      A[q] = 0.0;
    if (tid == 0)
      x[n] = 0.0;
    __syncthreads();
    (void)load_cell(A, t.lower_pos, lower, g, cl, m.nnz_lower);
    (void)load_cell(A, t.upper_pos, upper, g, cl, m.nnz_upper);
    const bool exact = load_cell(x, nullptr, xs, g, cl, n);
    bool diagonal = false;
    for (int i = tid; i < n; i += NT)
    {
      ld[i] = lower[(g * m.nnz_lower + m.lower_diag[i]) * kGroup + cl];
      diagonal = diagonal || ld[i] != 1.0;
    }
    const bool masked = any_thread(exact, s_flags);
    if (any_thread(diagonal, s_flags))
    {
      // rows without off-diagonal L entries only divide; they are inputs of every level
      for (int i = tid; i < t.first; i += NT)
        if (m.fwd_offsets[i] == m.fwd_offsets[i + 1])
          x[i] = x[i] / ld[i];
      __syncthreads();
      tail_solve_lower_diagonal(t, A, x, ld, ahead);
    }
    else
    {
      tail_solve(t, A, x, masked, ahead);
    }
    __syncthreads();
    for (int i = tid; i < n; i += NT)
      xs[(g * n + i) * kGroup + cl] = x[i];
  }

  template<int MINW, bool RECORD>
  hipError_t launch(unsigned blocks, size_t lds, hipStream_t stream, const CoopTailArgs& a)
  {
    const void* fn = reinterpret_cast<const void*>(k_coop_tail<MINW, RECORD>);
    if (const hipError_t e =
            hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
        e != hipSuccess)
      return e;
    hipLaunchKernelGGL((k_coop_tail<MINW, RECORD>), dim3(blocks), dim3(kTailThreads), lds, stream, a.m, a.c, a.t, a.p,
                       a.n_fixed, a.list, a.list_count, a.next, a.resume, a.y, a.k, a.atol, a.status, a.stats,
                       a.final_time, a.k_rows, a.tape);
    return hipGetLastError();
  }
}  // namespace

  int coop_tail_occupancy(int min_waves, size_t lds)
  {
    int per_cu = 0;
    const hipError_t e =
        min_waves == 3 ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_coop_tail<3, false>, kTailThreads, lds)
                       : hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_coop_tail<2, false>, kTailThreads, lds);
    return e == hipSuccess ? per_cu : 0;
  }

  hipError_t coop_tail_launch(int min_waves, unsigned blocks, size_t lds, hipStream_t stream, const CoopTailArgs& a)
  {
    if (a.tape.records)
      return min_waves == 3 ? launch<3, true>(blocks, lds, stream, a) : launch<2, true>(blocks, lds, stream, a);
    return min_waves == 3 ? launch<3, false>(blocks, lds, stream, a) : launch<2, false>(blocks, lds, stream, a);
  }

  size_t tail_factor_lds(const DevTail& t)
  {
    return sizeof(double) * (((static_cast<size_t>(t.nnz) + 2) & ~size_t(1)) + kTailBuffer);
  }

  size_t tail_solve_lds(const DevMech& m, const DevTail& t)
  {
    return sizeof(double) * (static_cast<size_t>(t.nnz) + 1 + 2 * static_cast<size_t>(m.n_species) + 1);
  }

  hipError_t lu_decompose_tail(const DevMech& m, const DevTail& t, int64_t n_cells, unsigned blocks, const double* jac,
                               double* lower, double* upper, hipStream_t stream)
  {
    const size_t lds = tail_factor_lds(t);
    if (const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k_lu_decompose_tail),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
        e != hipSuccess)
      return e;
    hipLaunchKernelGGL(k_lu_decompose_tail, dim3(blocks), dim3(kTailThreads), lds, stream, m, t, n_cells, jac, lower, upper);
    return hipGetLastError();
  }

  hipError_t lu_solve_tail(const DevMech& m, const DevTail& t, int64_t n_cells, unsigned blocks, const double* lower,
                           const double* upper, double* x, hipStream_t stream)
  {
    const size_t lds = tail_solve_lds(m, t);
    if (const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k_lu_solve_tail),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
        e != hipSuccess)
      return e;
    hipLaunchKernelGGL(k_lu_solve_tail, dim3(blocks), dim3(kTailThreads), lds, stream, m, t, n_cells, lower, upper, x);
    return hipGetLastError();
  }
}  // namespace micm_hip
