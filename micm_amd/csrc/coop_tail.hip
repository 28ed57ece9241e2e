// coop_tail.hip -- the cooperative Solve of mechanisms of 16 to 256 species: one workgroup of
// 256 threads per cell, the factor's last rows as a dense block (tail.hpp).
#include "coop_tail.hpp"

#include "path.hpp"
#include "tail.hpp"

namespace micm_hip
{
namespace
{
  // LDS holds what other threads read: the factor (head, block, zero), y, one vector x (stage
  // inputs, right-hand sides and solutions, x[n] = 0) and a scratch area shared in time by
  // the reaction rates, the Jacobian's partial products, the block's pivots and the error
  // terms.  Thread i keeps species i's stage vectors, f(y) and accumulated Jacobian diagonal
  // in registers; rate constants are read from a per-workgroup copy in global memory.
  //
  // Bound by the dependency chain of one attempt.  An attempt of the slowest cell, two waves
  // per SIMD, against the level-scheduled compact layout it replaced: 210/560 366 -> 131 us,
  // 60/200 110 -> 46 us, TS1 190 -> 71 us.
  template<int MINW, bool RECORD>
  __global__ void __launch_bounds__(kTailThreads, MINW)
      k_coop_tail(DevMech m, DevCoop c, DevTail t, DevParams p, int64_t n_fixed, const int32_t* __restrict__ list,
                  const int* list_count, int* next, const CellControl* resume, double* __restrict__ y_state,
                  double* __restrict__ k_state, const double* __restrict__ atol, int32_t* status_out,
                  int64_t* stats_out, double* final_time_out, const double* __restrict__ cond_state,
                  const double* __restrict__ custom_state, double* __restrict__ k_wg, Tape tape)
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
      const int64_t idx = s_idx;
      coop_sync<NT>();
      if (idx >= count)
        return;
      const int64_t cell = list ? list[idx] : idx;
      const size_t g = cell / kGroup;
      const int cl = cell % kGroup;
      {
        Lane ys = lane_view(y_state, g, n, cl);
        Lane ks = lane_view(k_state, g, m.n_reactions, cl);
        if (mine)
          L.y[tid] = ys[tid];
        if (tid == 0)
          x[n] = 0.0;
        if (cond_state)
        {
          // UpdateStateParameters fused into the launch
          Lane cd = lane_view(const_cast<double*>(cond_state), g, 3, cl);
          Lane cu = lane_view(const_cast<double*>(custom_state), g, m.n_custom, cl);
          const double T = cd[0], P = cd[1], rho = cd[2];
          for (int r = tid; r < m.n_reactions; r += NT)
          {
            const double kr = rate_constant(m, r, T, P, rho, cu);
            L.k[r] = kr;
            ks[r] = kr;
          }
        }
        else
        {
          for (int r = tid; r < m.n_reactions; r += NT)
            L.k[r] = ks[r];
        }
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
        // accumulated one: the same values as keeping -J and adding alpha in place.  A
        // factor with values that are not finite is formed again with the block's products
        // tested one by one.
        bool masked = false;
        while (true)
        {
          for (int q = tid; q <= t.nnz; q += NT)
            L.alu[q] = 0.0;
          coop_jacobian<NT, true>(m, c, L);
          if (mine)
          {
            if (fresh && !masked)
              jdiag = L.alu[diag];
            if (!masked)
              jdiag += alpha * 1.0;
            L.alu[diag] = jdiag;
          }
          coop_sync<NT>();
          coop_levels_piped<NT, true>(t.lu, t.lu.terms, L.alu, L.alu, L.alu);
          if (masked)
          {
            tail_factor_masked(t, L.alu);
            break;
          }
          if (tail_factor(t, L.alu, L.scratch, s_flags))
            break;
          masked = true;
        }
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
                       a.final_time, a.cond, a.custom, a.k_rows, a.tape);
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
}  // namespace micm_hip
