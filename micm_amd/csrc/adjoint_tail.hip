// adjoint_tail.hip -- the reverse sweep of the discrete adjoint, one workgroup of 256 threads
// per cell, the factor's last rows as a dense block.
#include "adjoint_tail.hpp"

#include "tail.hpp"

#include <algorithm>

namespace micm_hip
{
namespace
{
  // sum_q src[idx[q]] over [b, e), added in order
  __device__ __forceinline__ double list_sum(const int32_t* idx, int b, int e, const double* src)
  {
    double v = 0.0;
    for (int q = b; q < e; q += 8)
    {
      double s[8];
      int ix[8];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        ix[j] = idx[q + j];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        s[j] = src[ix[j]];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (q + j < e)
          v += s[j];
    }
    return v;
  }

  // The equations of adjoint.hpp, every sum in the order of k_adjoint.  Thread i holds lam_i
  // and gbar_i; LDS holds the factor (block layout), y, one vector x (stage inputs, right-hand
  // sides, rbar), the stage vectors K and Kbar, per reaction k, w and thb, the Jacobian terms
  // d_t(y), and a scratch area for rates, pivots and the terms of the gathers.
  //
  // Bound by the chain of one record, as the Solve's attempt is (replaying it is an attempt), up to
  // a few cells per CU, and then by the lanes' issue.  Against k_adjoint: the block in both
  // directions, a second derivative per thread from one packed word instead of a species'
  // list of four dependent reads each, lists read eight entries at a time.  Four waves per
  // SIMD: they spill 55 registers and lose nothing by it (64 cells of 60/200: 84.7 ms, with
  // two waves and no spills 85.6; 1,024 cells 111 against 156).
  // All records of 1,024 cells of 60/200 373 -> 111 ms (20/50 116 -> 61), of 256 of TS1
  // 418 -> 139, of 210/560 1,477 -> 298.
  __global__ void __launch_bounds__(kTailThreads, 4)
      k_adjoint_tail(DevMech m, DevCoop c, DevTail t, DevAdjointLists a, DevParams p, int64_t n_cells,
                     const double* __restrict__ k_state, Tape tape, const double* __restrict__ seed,
                     double* __restrict__ grad_y, double* __restrict__ grad_logk)
  {
    constexpr int NT = kTailThreads;
    extern __shared__ double lds[];
    __shared__ int s_flags[NT / kWave];
    int tid = threadIdx.x;
    const int n = m.n_species, R = m.n_reactions, S = p.stages;
    const bool mine = static_cast<int>(threadIdx.x) < n;
    const int own = mine ? threadIdx.x : 0;
    double* const alu = lds;
    double* const y = alu + t.nnz + 1;
    double* const x = y + n;
    double* const gb = x + n + 1;
    double* const K = gb + n;
    double* const Kb = K + static_cast<size_t>(S) * n;
    double* const kk = Kb + static_cast<size_t>(S) * n;
    double* const w = kk + R;
    double* const th = w + R;
    double* const jterm = th + R;
    double* const tmp = lds + ((static_cast<size_t>(jterm - lds) + c.n_terms + 1) & ~size_t(1));
    CoopLds L{};
    L.alu = alu;
    L.y = y;
    L.k = kk;
    L.scratch = tmp;
    L.jterm = jterm;
    c.jac_to_alu = t.jac_pos;
    const size_t rec_len = static_cast<size_t>(n) + 1;
    const int diag = t.diag_pos[own];
    // w_r(u) of every reaction
    auto weights = [&](const double* u) {
      for (int r = tid; r < R; r += NT)
        w[r] = gather_sum(0.0, a.weight_species, a.weight_coef, a.weight_offsets[r], a.weight_offsets[r + 1], u);
    };
    for (int64_t cell = blockIdx.x; cell < n_cells; cell += gridDim.x)
    {
      const size_t g = cell / kGroup;
      const int cl = cell % kGroup;
      const Lane gy = lane_view(grad_y, g, n, cl), gk = lane_view(grad_logk, g, R, cl);
      const int64_t count = tape.counts[cell];
      if (count > tape.max_records)
      {
        // an overflowed tape lacks the cell's first records: no gradient
        if (mine)
          gy[tid] = __builtin_nan("");
        for (int r = tid; r < R; r += NT)
          gk[r] = __builtin_nan("");
        continue;
      }
      const Lane ks = lane_view(const_cast<double*>(k_state), g, R, cl);
      for (int r = tid; r < R; r += NT)
      {
        kk[r] = ks[r];
        th[r] = 0.0;
      }
      double lam = mine ? lane_view(const_cast<double*>(seed), g, n, cl)[tid] : 0.0;
      if (tid == 0)
        x[n] = 0.0;
      const double* const records = tape.records + static_cast<size_t>(cell) * tape.max_records * rec_len;
      double y_next = 0.0, H_next = 0.0;
      if (count > 0)
      {
        H_next = records[(count - 1) * rec_len];
        y_next = records[(count - 1) * rec_len + 1 + own];
      }
      for (int64_t rix = count - 1; rix >= 0; --rix)
      {
        const double H = H_next, y_r = y_next;
        if (rix > 0)
        {
          H_next = records[(rix - 1) * rec_len];
          y_next = records[(rix - 1) * rec_len + 1 + own];
        }
        if (H == kClampTag)
        {
          // y = max(y, 0): no derivative where the value was clamped
          if (y_r < 0.0)
            lam = 0.0;
          continue;
        }
        here(tid);
        // ---- the recorded step again: -J(y) into the factor, alpha, LU, stages
        coop_sync<NT>();
        if (mine)
          y[tid] = y_r;
        for (int q = tid; q <= t.nnz; q += NT)
          alu[q] = 0.0;
        coop_sync<NT>();
        coop_jacobian<NT, true>(m, c, L);  // jterm = d_t(y)
        const double alpha = 1.0 / (H * p.gamma0);
        if (mine)
          alu[diag] += alpha * 1.0;
        coop_sync<NT>();
        coop_levels_piped<NT, true>(t.lu, t.lu.terms, alu, alu, alu);
        const bool masked = __builtin_amdgcn_readfirstlane(!tail_factor<false>(t, alu, tmp, s_flags));
        if (masked)
          tail_factor_masked(t, alu);
        RowsAhead ahead = rows_ahead(t.rows);
        double f = 0.0;
        for (int s = 0; s < S; ++s)
        {
          const int sc = s * (s - 1) / 2;
          if (s == 0 || p.new_f[s])
          {
            double v = y_r;
            if (s > 0)
            {
              for (int j = 0; j < s; ++j)
                v += p.a[sc + j] * K[static_cast<size_t>(j) * n + own];
              if (mine)
                x[tid] = v;
              coop_sync<NT>();
            }
            f = coop_forcing_own<NT>(m, c, L, s == 0 ? y : x);
          }
          double v = f;
          for (int j = 0; j < s; ++j)
            v += (p.c[sc + j] / H) * K[static_cast<size_t>(j) * n + own];
          if (mine)
            x[tid] = v;
          coop_sync<NT>();
          tail_solve(t, alu, x, masked, ahead);
          if (mine)
            K[static_cast<size_t>(s) * n + tid] = x[tid];
        }
        // ---- reverse over the stages
        if (mine)
          for (int s = 0; s < S; ++s)
            Kb[static_cast<size_t>(s) * n + tid] = p.m[s] * lam;
        RowsAhead ahead_t = rows_ahead(t.t_rows);
        double gbar = 0.0;
        for (int s = S - 1; s >= 0; --s)
        {
          const int sc = s * (s - 1) / 2;
          const double* Ks = K + static_cast<size_t>(s) * n;
          if (mine)
            x[tid] = Kb[static_cast<size_t>(s) * n + tid];
          coop_sync<NT>();
          tail_solve_transposed(t, alu, x, masked, ahead_t);
          here(tid);
          weights(x);
          coop_sync<NT>();
          // Jbar = rbar K_s^T through k and y
          for (int r = tid; r < R; r += NT)
          {
            const int b = a.rxn_offsets[r], e = a.rxn_offsets[r + 1];
            double acc = 0.0;
            for (int q = b; q < e; q += 4)
            {
              int it[4], is[4];
#pragma unroll
              for (int j = 0; j < 4; ++j)
              {
                it[j] = a.rxn_terms[q + j];
                is[j] = a.rxn_indep[q + j];
              }
#pragma unroll
              for (int j = 0; j < 4; ++j)
                if (q + j < e)
                  acc += jterm[it[j]] * Ks[is[j]];
            }
            th[r] += w[r] * acc;
          }
          for (int e0 = tid; e0 < a.n_second; e0 += 2 * NT)
          {
            uint64_t pk[2];
#pragma unroll
            for (int j = 0; j < 2; ++j)
              pk[j] = a.second[e0 + j * NT < a.n_second ? e0 + j * NT : e0];
#pragma unroll
            for (int j = 0; j < 2; ++j)
            {
              const uint32_t r = pk[j] & 0xffffu, i = (pk[j] >> 16) & 0xffffu;
              const uint32_t d0 = (pk[j] >> 32) & 0xffffu, d1 = static_cast<uint32_t>(pk[j] >> 48);
              double d = kk[r];
              const double y0 = y[d0 != 0xffffu ? d0 : 0], y1 = y[d1 != 0xffffu ? d1 : 0];
              d = d0 != 0xffffu ? d * y0 : d;
              d = d1 != 0xffffu ? d * y1 : d;
              if (e0 + j * NT < a.n_second)
                tmp[e0 + j * NT] = w[r] * Ks[i] * d;
            }
          }
          coop_sync<NT>();
          const bool evaluates = s == 0 || p.new_f[s];
          if (mine)
          {
            double acc = 0.0;
            const int b = a.second_offsets[tid], e = a.second_offsets[tid + 1];
#pragma unroll 4
            for (int q = b; q < e; ++q)
              acc += tmp[q];
            lam += acc;
            const double rb = x[tid];
            gbar += rb;
            for (int j = 0; j < s; ++j)
              Kb[static_cast<size_t>(j) * n + tid] += (p.c[sc + j] / H) * rb;
            if (evaluates)
            {
              gb[tid] = gbar;
              double v = y_r;
              for (int j = 0; j < s; ++j)
                v += p.a[sc + j] * K[static_cast<size_t>(j) * n + tid];
              x[tid] = v;  // Y_s
            }
          }
          if (!evaluates)
            continue;
          coop_sync<NT>();
          here(tid);
          // w(gbar) and the rates at Y_s, both by the reaction's thread
          weights(gb);
          coop_rates<NT>(m, c, L, x);
          coop_sync<NT>();
          for (int r = tid; r < R; r += NT)
            th[r] += w[r] * tmp[r];
          coop_sync<NT>();
          coop_term_products<NT>(m, c, L, x, [&](int q, double d, uint64_t pk) { tmp[q] = w[pk & 0xffffu] * d; });
          coop_sync<NT>();
          if (mine)
          {
            const double yb = list_sum(a.indep_terms, a.indep_offsets[tid], a.indep_offsets[tid + 1], tmp);
            lam += yb;
            for (int j = 0; j < s; ++j)
              Kb[static_cast<size_t>(j) * n + tid] += p.a[sc + j] * yb;
            gbar = 0.0;
          }
        }
      }
      if (mine)
        gy[tid] = lam;
      // (each reaction's sum is read by the thread that formed it)
      for (int r = tid; r < R; r += NT)
        gk[r] = th[r];
      coop_sync<NT>();
    }
  }
}  // namespace

  size_t adjoint_tail_lds(const DevMech& m, const DevCoop& c, const DevTail& t, const DevAdjointLists& a, int stages)
  {
    const int tmp = std::max(std::max(m.n_reactions, c.n_terms), std::max(a.n_second, kTailBuffer));
    return sizeof(double) * (static_cast<size_t>(t.nnz) + 1 + static_cast<size_t>(3 + 2 * stages) * m.n_species + 1 +
                             3 * static_cast<size_t>(m.n_reactions) + c.n_terms + 1 + static_cast<size_t>(tmp));
  }

  int adjoint_tail_occupancy(size_t lds)
  {
    int per_cu = 0;
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_adjoint_tail, kTailThreads, lds) == hipSuccess ? per_cu
                                                                                                               : 0;
  }

  hipError_t adjoint_tail(const DevMech& m, const DevCoop& c, const DevTail& t, const DevAdjointLists& a,
                          const DevParams& p, int64_t n_cells, unsigned blocks, size_t lds, const double* k,
                          const Tape& tape, const double* seed, double* grad_y, double* grad_logk, hipStream_t stream)
  {
    if (const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k_adjoint_tail),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
        e != hipSuccess)
      return e;
    hipLaunchKernelGGL(k_adjoint_tail, dim3(blocks), dim3(kTailThreads), lds, stream, m, c, t, a, p, n_cells, k, tape,
                       seed, grad_y, grad_logk);
    return hipGetLastError();
  }
}  // namespace micm_hip
