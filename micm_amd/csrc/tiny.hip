// tiny.hip -- Solves of the smallest mechanisms (tiny.hpp), one cell per lane.
#include "tiny.hpp"

#include "path.hpp"

namespace micm_hip
{
namespace
{
  constexpr int kWave = 64;

  __host__ __device__ constexpr int padded(int n)
  {
    return (n + kTinyBatch - 1) / kTinyBatch * kTinyBatch;
  }

  // LDS: the lists, packed operands, and per lane (stride kWave) y, k, the rates or Jacobian
  // terms, f, -J and the stage vectors.
  struct TinyLds
  {
    TinyEntry *forcing, *jacobian;
    uint64_t *reactions, *terms;
    double *y, *k, *source, *f, *jac, *stages;
  };

  __host__ __device__ inline size_t tiny_layout(const DevMech& m, const DevCoop& c, const DevTiny& t, size_t stages, char* base,
                                                  TinyLds* out)
  {
    const int n = m.n_species, R = m.n_reactions, T = c.n_terms;
    size_t at = 0;
    auto take = [&](size_t bytes) {
      const size_t here = at;
      at += (bytes + 15) & ~size_t(15);
      return base + here;
    };
    TinyLds l;
    l.forcing = reinterpret_cast<TinyEntry*>(take(sizeof(TinyEntry) * t.n_forcing));
    l.jacobian = reinterpret_cast<TinyEntry*>(take(sizeof(TinyEntry) * t.n_jacobian));
    l.reactions = reinterpret_cast<uint64_t*>(take(sizeof(uint64_t) * padded(R)));
    l.terms = reinterpret_cast<uint64_t*>(take(sizeof(uint64_t) * padded(T)));
    constexpr size_t column = sizeof(double) * kWave;
    l.y = reinterpret_cast<double*>(take(column * n));
    l.k = reinterpret_cast<double*>(take(column * padded(R)));
    l.source = reinterpret_cast<double*>(take(column * padded(R > T ? R : T)));
    l.f = reinterpret_cast<double*>(take(column * (n + 1)));
    l.jac = reinterpret_cast<double*>(take(column * (n * n + 1)));
    l.stages = reinterpret_cast<double*>(take(column * n * stages));
    if (out)
      *out = l;
    return at;
  }

  template<class V>
  __device__ __forceinline__ void copy_in(V* to, const V* from, int n)
  {
    const uint32_t* src = reinterpret_cast<const uint32_t*>(from);
    uint32_t* dst = reinterpret_cast<uint32_t*>(to);
    for (int q = threadIdx.x; q < n * static_cast<int>(sizeof(V) / sizeof(uint32_t)); q += kWave)
      dst[q] = src[q];
  }

  // The lists' sums into a lane's columns, without a branch in a batch of entries.
  __device__ __forceinline__ void tiny_gather(const TinyEntry* list, int n_entries, uint32_t spare, const double* source,
                                              double* dst)
  {
    double acc = 0.0;
#pragma unroll 1
    for (int q = 0; q < n_entries; q += kTinyBatch)
    {
      TinyEntry e[kTinyBatch];
      double v[kTinyBatch];
#pragma unroll
      for (int j = 0; j < kTinyBatch; ++j)
        e[j] = list[q + j];
#pragma unroll
      for (int j = 0; j < kTinyBatch; ++j)
        v[j] = source[e[j].from * kWave];
#pragma unroll
      for (int j = 0; j < kTinyBatch; ++j)
      {
        acc += e[j].coef * v[j];
        dst[e[j].to * kWave] = acc;
        acc = e[j].to != spare ? 0.0 : acc;
      }
    }
  }

  // One cell per lane, the linear algebra of its n <= N species in registers: the factor as N x N
  // with each product guarded by the fill pattern (uniform branches), so that every sum has
  // the reference's products in its order.  The sparse gathers walk lists in LDS that all
  // lanes share, the operands in columns of their own.
  //
  // Bound by the chain of one lane's attempt, 7 us of three species and two reactions (two
  // forcings 1.9 us, three substitutions 1.8, the Jacobian 1.1, error and control 1.1, LU 0.75),
  // whatever the number of cells up to a wavefront per SIMD.  A workgroup per cell spends 13 us on
  // the same attempt, on barriers and table reads, and a CU holds few of them: 1,000 cells 173
  // -> 88 us, 100,000 cells 9.9 -> 0.6 ms.
  //
  // LOCKSTEP: the cells of one wavefront share the step control; their error terms are added
  // in the order of the State's dense matrix.
  template<int N, bool LOCKSTEP>
  __global__ void __launch_bounds__(kWave) k_tiny(TinyArgs a)
  {
    extern __shared__ char lds_tiny[];
    __shared__ double s_terms[LOCKSTEP ? kWave * N : 1];
    const DevMech& m = a.m;
    const DevParams& p = a.p;
    const int n = m.n_species, R = m.n_reactions, T = a.c.n_terms;
    const int lane = threadIdx.x;
    TinyLds L;
    tiny_layout(m, a.c, a.t, p.stages, lds_tiny, &L);
    copy_in(L.forcing, a.t.forcing, a.t.n_forcing);
    copy_in(L.jacobian, a.t.jacobian, a.t.n_jacobian);
    copy_in(L.reactions, a.c.rxn_pack, R);
    copy_in(L.terms, a.c.term_pack, T);
    const int64_t count = a.list ? static_cast<int64_t>(*a.list_count) : a.n_cells;
    const int64_t idx = static_cast<int64_t>(blockIdx.x) * kWave + lane;
    const bool active = idx < count;
    if (!LOCKSTEP && static_cast<int64_t>(blockIdx.x) * kWave >= count)
      return;
    // (a lane without a cell repeats the first one's)
    const int64_t at = active ? idx : static_cast<int64_t>(blockIdx.x) * kWave;
    const int64_t cell = a.list ? a.list[at] : at;
    const size_t g = cell / kGroup;
    const int cl = cell % kGroup;
    const Lane ys = lane_view(a.y, g, n, cl);
    const Lane ks = lane_view(const_cast<double*>(a.k), g, R, cl);
    if (lane < kTinyBatch)
    {
      // the padding's operands: any that there are
      if (R + lane < padded(R))
        L.reactions[R + lane] = 0;
      if (T + lane < padded(T))
        L.terms[T + lane] = 0;
    }
    for (int r = 0; r < padded(R); ++r)
      L.k[r * kWave + lane] = r < R ? ks[r] : 0.0;
    for (int q = 0; q < n * n; ++q)
      L.jac[q * kWave + lane] = 0.0;
    for (int i = 0; i < n; ++i)
      L.f[i * kWave + lane] = 0.0;
    double y[N], atol[N];
#pragma unroll
    for (int i = 0; i < N; ++i)
    {
      y[i] = i < n ? ys[i] : 0.0;
      atol[i] = i < n ? a.atol[i] : 1.0;
    }
    __syncthreads();
    const uint64_t pattern = a.t.pattern;
    auto in = [&](int i, int j) { return ((pattern >> (kTinySpecies * i + j)) & 1u) != 0; };
    auto forcing = [&](const double (&v)[N], double (&f)[N]) {
#pragma unroll
      for (int i = 0; i < N; ++i)
        if (i < n)
          L.y[i * kWave + lane] = v[i];
#pragma unroll 1
      for (int r0 = 0; r0 < R; r0 += kTinyBatch)
      {
        uint64_t pk[kTinyBatch];
        double rate[kTinyBatch], o0[kTinyBatch], o1[kTinyBatch], o2[kTinyBatch];
#pragma unroll
        for (int j = 0; j < kTinyBatch; ++j)
          pk[j] = L.reactions[r0 + j];
#pragma unroll
        for (int j = 0; j < kTinyBatch; ++j)
        {
          rate[j] = L.k[(r0 + j) * kWave + lane];
          o0[j] = L.y[(pk[j] & 0xffffu) * kWave + lane];
          o1[j] = L.y[((pk[j] >> 16) & 0xffffu) * kWave + lane];
          o2[j] = L.y[((pk[j] >> 32) & 0xffffu) * kWave + lane];
        }
#pragma unroll
        for (int j = 0; j < kTinyBatch; ++j)
        {
          const uint32_t operands = static_cast<uint32_t>(pk[j] >> 48);
          double v = rate[j];
          v = operands > 0 ? v * o0[j] : v;
          v = operands > 1 ? v * o1[j] : v;
          v = operands > 2 ? v * o2[j] : v;
          L.source[(r0 + j) * kWave + lane] = v;
        }
      }
      tiny_gather(L.forcing, a.t.n_forcing, n, L.source + lane, L.f + lane);
#pragma unroll
      for (int i = 0; i < N; ++i)
        f[i] = i < n ? L.f[i * kWave + lane] : 0.0;
    };
    // -J at the y that forcing was last called with
    auto jacobian = [&]() {
#pragma unroll 1
      for (int q = 0; q < T; q += kTinyBatch)
      {
        uint64_t pk[kTinyBatch];
        double d[kTinyBatch], o0[kTinyBatch], o1[kTinyBatch];
#pragma unroll
        for (int j = 0; j < kTinyBatch; ++j)
          pk[j] = L.terms[q + j];
#pragma unroll
        for (int j = 0; j < kTinyBatch; ++j)
        {
          d[j] = L.k[(pk[j] & 0xffffu) * kWave + lane];
          o0[j] = L.y[((pk[j] >> 16) & 0xffffu) * kWave + lane];
          o1[j] = L.y[((pk[j] >> 32) & 0xffffu) * kWave + lane];
        }
#pragma unroll
        for (int j = 0; j < kTinyBatch; ++j)
        {
          const uint32_t operands = static_cast<uint32_t>(pk[j] >> 48);
          double v = d[j];
          v = operands > 0 ? v * o0[j] : v;
          v = operands > 1 ? v * o1[j] : v;
          L.source[(q + j) * kWave + lane] = v;
        }
      }
      tiny_gather(L.jacobian, a.t.n_jacobian, n * n, L.source + lane, L.jac + lane);
    };
    CellControl cc;
    if (a.resume)
      cc = a.resume[cell];
    else
      control_init(p, cc);
    double f0[N], jdiag[N], A[N][N];
#pragma unroll
    for (int i = 0; i < N; ++i)
      f0[i] = jdiag[i] = 0.0;
    while (cc.status == MICM_HIP_STATE_RUNNING)
    {
      bool fresh = false;
      if (cc.flags & kNewStep)
      {
        if (!begin_step(p, cc))
          break;
        cc.stats[MICM_HIP_STAT_FUNCTION_CALLS] += 1;
        cc.stats[MICM_HIP_STAT_JACOBIAN_UPDATES] += 1;
        cc.last_alpha = 0.0;
        cc.flags &= ~kNewStep;
        fresh = true;
      }
      const double alpha = next_alpha(p, cc);
      cc.stats[MICM_HIP_STAT_DECOMPOSITIONS] += 1;
      double f[N], ynew[N], yerr[N];
#pragma unroll
      for (int i = 0; i < N; ++i)
      {
        f[i] = f0[i];
        ynew[i] = y[i];
        yerr[i] = 0.0;
      }
      // one copy of the code for all stages: a launch starts with a cold instruction cache
#pragma unroll 1
      for (int s = 0; s < p.stages; ++s)
      {
        const int sc = s * (s - 1) / 2;
        if (s == 0 ? fresh : p.new_f[s] != 0)
        {
          double v[N];
#pragma unroll
          for (int i = 0; i < N; ++i)
            v[i] = y[i];
#pragma unroll 1
          for (int j = 0; j < s; ++j)
          {
            const double aj = p.a[sc + j];
#pragma unroll
            for (int i = 0; i < N; ++i)
              if (i < n)
                v[i] += aj * L.stages[(j * n + i) * kWave + lane];
          }
          forcing(v, f);
        }
        if (s == 0)
        {
          if (fresh)
          {
#pragma unroll
            for (int i = 0; i < N; ++i)
              f0[i] = f[i];
            jacobian();
          }
#pragma unroll
          for (int i = 0; i < N; ++i)
#pragma unroll
            for (int j = 0; j < N; ++j)
              A[i][j] = i < n && j < n ? L.jac[(i * n + j) * kWave + lane] : 0.0;
#pragma unroll
          for (int i = 0; i < N; ++i)
          {
            if (fresh)
              jdiag[i] = A[i][i];
            jdiag[i] += alpha * 1.0;
            A[i][i] = jdiag[i];
          }
          // Doolittle, pivot by pivot
#pragma unroll
          for (int q = 0; q < N; ++q)
#pragma unroll
            for (int i = q + 1; i < N; ++i)
              if (in(i, q))
              {
                A[i][q] = A[i][q] / A[q][q];
#pragma unroll
                for (int j = q + 1; j < N; ++j)
                  if (in(q, j))
                    A[i][j] -= A[i][q] * A[q][j];
              }
        }
        else if (p.new_f[s])
        {
          cc.stats[MICM_HIP_STAT_FUNCTION_CALLS] += 1;
        }
        double x[N];
#pragma unroll
        for (int i = 0; i < N; ++i)
          x[i] = f[i];
#pragma unroll 1
        for (int j = 0; j < s; ++j)
        {
          const double cj = p.c[sc + j] / cc.H;
#pragma unroll
          for (int i = 0; i < N; ++i)
            if (i < n)
              x[i] += cj * L.stages[(j * n + i) * kWave + lane];
        }
#pragma unroll
        for (int i = 1; i < N; ++i)
#pragma unroll
          for (int j = 0; j < i; ++j)
            if (in(i, j))
              x[i] -= A[i][j] * x[j];
#pragma unroll
        for (int i = N - 1; i >= 0; --i)
          if (i < n)
          {
#pragma unroll
            for (int j = i + 1; j < N; ++j)
              if (in(i, j))
                x[i] -= A[i][j] * x[j];
            x[i] = x[i] / A[i][i];
          }
        // y + sum m_s K_s and sum e_s K_s, stage by stage
        const double ms = p.m[s], es = p.e[s];
#pragma unroll
        for (int i = 0; i < N; ++i)
          if (i < n)
          {
            L.stages[(s * n + i) * kWave + lane] = x[i];
            ynew[i] += ms * x[i];
            yerr[i] += es * x[i];
          }
        cc.stats[MICM_HIP_STAT_SOLVES] += 1;
      }
      double terms[N];
#pragma unroll
      for (int i = 0; i < N; ++i)
      {
        const double b = fabs(y[i]), d = fabs(ynew[i]);
        const double q = yerr[i] / (atol[i] + p.rtol * (b > d ? b : d));
        terms[i] = q * q;
      }
      double acc = 0.0, n_terms = static_cast<double>(n);
      if constexpr (LOCKSTEP)
      {
        // term (cell, species) at its place in the State's order (groups of error_group cells,
        // species by species)
        const int64_t gi = idx / p.error_group, first = gi * p.error_group;
        const int64_t rows = a.n_cells - first < p.error_group ? a.n_cells - first : p.error_group;
#pragma unroll
        for (int i = 0; i < N; ++i)
          if (active && i < n)
            s_terms[first * n + i * rows + (idx - first)] = terms[i];
        __syncthreads();
        const int total = static_cast<int>(a.n_cells) * n;
        for (int q = 0; q < total; q += 8)
        {
          double v[8];
#pragma unroll
          for (int j = 0; j < 8; ++j)
            v[j] = s_terms[q + j < total ? q + j : q];
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if (q + j < total)
              acc += v[j];
        }
        __syncthreads();
        n_terms = static_cast<double>(total);
      }
      else
      {
#pragma unroll
        for (int i = 0; i < N; ++i)
          if (i < n)
            acc += terms[i];
      }
      const double error = smax(sqrt(acc / n_terms), 1.0e-10);
      if (control_update(p, cc, error))
      {
#pragma unroll
        for (int i = 0; i < N; ++i)
          y[i] = ynew[i];
      }
    }
    if (!active)
      return;
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (i < n)
        ys[i] = smax(y[i], 0.0);
    a.status[cell] = cc.status;
    for (int i = 0; i < 7; ++i)
      a.stats[cell * 7 + i] = cc.stats[i];
    a.final_time[cell] = cc.t;
  }

  template<bool LOCKSTEP>
  hipError_t launch(const TinyArgs& a, unsigned blocks, size_t lds, hipStream_t stream)
  {
    if (a.m.n_species <= 4)
      hipLaunchKernelGGL((k_tiny<4, LOCKSTEP>), dim3(blocks), dim3(kWave), lds, stream, a);
    else
      hipLaunchKernelGGL((k_tiny<kTinySpecies, LOCKSTEP>), dim3(blocks), dim3(kWave), lds, stream, a);
    return hipGetLastError();
  }
}  // namespace

  size_t tiny_lds(const DevMech& m, const DevCoop& c, const DevTiny& t, int stages)
  {
    if (t.n_forcing < 0)
      return 0;
    const size_t bytes = tiny_layout(m, c, t, stages, nullptr, nullptr);
    return bytes <= kTinyLds ? bytes : 0;
  }

  hipError_t tiny_solve(const TinyArgs& a, size_t lds, hipStream_t stream)
  {
    return launch<false>(a, static_cast<unsigned>((a.n_cells + kWave - 1) / kWave), lds, stream);
  }

  hipError_t tiny_lockstep(const TinyArgs& a, size_t lds, hipStream_t stream)
  {
    return launch<true>(a, 1, lds, stream);
  }
}  // namespace micm_hip
