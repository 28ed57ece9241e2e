// tail.hpp -- the factorisation and both substitutions of one cell with the factor's last
// rows and columns as a dense block (TailTables): the Markowitz order leaves the rows that
// fill in to the end, so a block of 16 to 64 rows holds most of a factorisation's products
// (210 species: 74,000 of 121,000 in 64 rows) and nearly all of its dependency chain (110
// of 125 levels).  Every sum keeps the reference's order:
//
//   factor    element (i, j) of the block subtracts L[i][k] U[k][j] for k ascending, as in
//             lu_decomposition_doolittle.inl:347-398: the pivots before the block as a
//             level schedule, the block's own one pivot at a time with all its elements in
//             registers
//   forward   x_i -= L_ij x_j, j ascending (linear_solver.inl:250-265): the columns before
//             the block as levels, then one column of the block after another, lane = row
//   backward  x_i -= U_ij x_j, j ascending, then / U_ii (linear_solver.inl:270-287): the
//             block's rows one after another, then the rows before it as levels
//
// The block is run without its structural zeros' tests: a zero's product 0 * u subtracted
// from a partial sum leaves it as it is, since no partial sum is ever -0 (the Jacobian, the
// right-hand sides and every difference of unlike values round to +0) -- unless u is
// infinite or NaN.  Every result of the block is therefore checked to be finite, and a cell
// with one that is not is done again with each product tested against the fill pattern
// (MASKED), which is exact for every operand.
#pragma once

#include "coop.hpp"

#include <type_traits>

namespace micm_hip
{
  constexpr int kTailThreads = 256;

  // v - p[K0] - ... - p[15], subtracted in that order, p[k] being lane k's p of the reader's
  // DPP row of sixteen lanes.  One instruction a product: the multiply by m1 = -1 is exact,
  // so the fused form rounds once, as the subtraction does.  5.4 clocks a product on
  // MI355X against 12 through LDS (the products' writes, reads and subtractions).  The two
  // wait states cover a p written by the instruction before.
  template<int K0>
  __device__ __forceinline__ double ordered_sub16(double v, double p, double m1)
  {
#define MICM_SUB(k) "v_fmac_f64_dpp %0, %1, %2 row_newbcast:" #k " row_mask:0xf bank_mask:0xf\n\t"
#define MICM_SUB4(a, b, c, d) MICM_SUB(a) MICM_SUB(b) MICM_SUB(c) MICM_SUB(d)
    static_assert(K0 == 0 || K0 == 4 || K0 == 8 || K0 == 12, "sums start at a multiple of four");
    if constexpr (K0 == 0)
      asm("s_nop 1\n\t" MICM_SUB4(0, 1, 2, 3) MICM_SUB4(4, 5, 6, 7) MICM_SUB4(8, 9, 10, 11) MICM_SUB4(12, 13, 14, 15)
          : "+v"(v)
          : "v"(p), "v"(m1));
    else if constexpr (K0 == 4)
      asm("s_nop 1\n\t" MICM_SUB4(4, 5, 6, 7) MICM_SUB4(8, 9, 10, 11) MICM_SUB4(12, 13, 14, 15)
          : "+v"(v)
          : "v"(p), "v"(m1));
    else if constexpr (K0 == 8)
      asm("s_nop 1\n\t" MICM_SUB4(8, 9, 10, 11) MICM_SUB4(12, 13, 14, 15) : "+v"(v) : "v"(p), "v"(m1));
    else
      asm("s_nop 1\n\t" MICM_SUB4(12, 13, 14, 15) : "+v"(v) : "v"(p), "v"(m1));
#undef MICM_SUB4
#undef MICM_SUB
    return v;
  }

  // The value of lane 4 (l / 4) + A in every lane l.
  template<int A>
  __device__ __forceinline__ double quad_lane(double v)
  {
    constexpr int ctrl = A * 0x55;  // quad_perm [A, A, A, A]
    const uint64_t b = static_cast<uint64_t>(__double_as_longlong(v));
    const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(b), ctrl, 0xf, 0xf, true));
    const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(b >> 32), ctrl, 0xf, 0xf, true));
    return __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(hi) << 32) | lo));
  }

  // Doubles of LDS that tail_factor uses besides the factor: two buffers of a pivot row and
  // a pivot column.
  constexpr int kTailBuffer = 4 * kTailMax;

  // Pivots 16 (PA - p0) ... + 15 of a block of 4 - p0 sixteens: thread (ti, tj) holds the
  // elements (ti + 16 (a - p0), tj + 16 (b - p0)) as e[a][b].  At a pivot its row and column
  // go through LDS (two buffers, so one barrier a pivot); every four lanes divide one
  // column value each and pass the quotients on by DPP, and each thread updates its
  // elements below and right of the pivot.  Elements that are final already see a zero
  // factor.
  template<int PA, bool MASKED>
  __device__ __forceinline__ void tail_pivots(double (&e)[4][4], const DevTail& t, int p0, int ti, int tj, double* buf,
                                              const uint64_t (&rm)[4])
  {
    for (int kk = 0; kk < kTailBlock; ++kk)
    {
      double* row = buf + (kk & 1) * (2 * kTailMax);
      double* col = row + kTailMax;
      if (ti == kk)
      {
#pragma unroll
        for (int b = PA; b < 4; ++b)
          row[tj * 4 + b] = e[PA][b];
      }
      if (tj == kk)
      {
#pragma unroll
        for (int a = PA; a < 4; ++a)
          col[ti * 4 + a] = e[a][PA];
      }
      lds_barrier<kTailThreads>();
      const double piv = row[kk * 4 + PA];
      const double c = col[ti * 4 + (PA == 3 ? 3 : (tj & 3))];
      double u[4];
#pragma unroll
      for (int b = PA; b < 4; ++b)
        u[b] = row[tj * 4 + b];
      const double q = c / piv;
      double l[4];
      if constexpr (PA == 3)
      {
        l[3] = q;
      }
      else
      {
        if constexpr (PA <= 0)
          l[0] = quad_lane<0>(q);
        if constexpr (PA <= 1)
          l[1] = quad_lane<1>(q);
        l[2] = quad_lane<2>(q);
        l[3] = quad_lane<3>(q);
      }
      if constexpr (!MASKED)
      {
        const double u_pa = tj > kk ? u[PA] : 0.0, l_pa = ti > kk ? l[PA] : 0.0;
#pragma unroll
        for (int a = PA; a < 4; ++a)
        {
          const double la = a == PA ? l_pa : l[a];
#pragma unroll
          for (int b = PA; b < 4; ++b)
            e[a][b] -= la * (b == PA ? u_pa : u[b]);
          if (tj == kk && (a > PA || ti > kk))
            e[a][PA] = l[a];
        }
      }
      else
      {
        const int k = kTailBlock * (PA - p0) + kk;
        const uint64_t rk = const_load(t.row_mask, k);
#pragma unroll
        for (int a = PA; a < 4; ++a)
          if ((a > PA || ti > kk) && ((rm[a] >> k) & 1u))
          {
#pragma unroll
            for (int b = PA; b < 4; ++b)
              if ((b > PA || tj > kk) && ((rk >> (tj + kTailBlock * (b - p0))) & 1u))
                e[a][b] -= l[a] * u[b];
            if (tj == kk)
              e[a][PA] = l[a];
          }
      }
    }
  }

  // The block's own factorisation in place (A: the factor, its head and the block's sums
  // over the head's pivots final), 256 threads.  False (on every thread) when an element is
  // not finite; the block is then left as it is, if not MASKED.  buf: kTailBuffer doubles;
  // flags: one int per wave.  Ends with a barrier.
  //
  // One pivot costs an LDS round trip with a barrier (140 clocks), a division (53) and ten
  // clocks for each of a thread's elements, whatever the fill; the level schedule of the
  // same rows takes two levels a pivot at 1,400 each.
  template<bool MASKED>
  __device__ inline bool tail_factor(const DevTail& t, double* A, double* buf, int* flags)
  {
    const int tid = threadIdx.x;
    const int ti = tid >> 4, tj = tid & 15;
    const int p0 = 4 - t.size / kTailBlock;
    const int stride = t.size + 1;
    double* base = A + t.head + ti * stride + tj;
    double e[4][4];
    uint64_t rm[4] = { 0, 0, 0, 0 };
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b)
      {
        e[a][b] = 0.0;
        if (a >= p0 && b >= p0)
          e[a][b] = base[kTailBlock * (stride * (a - p0) + (b - p0))];
      }
    if constexpr (MASKED)
    {
#pragma unroll
      for (int a = 0; a < 4; ++a)
        if (a >= p0)
          rm[a] = t.row_mask[ti + kTailBlock * (a - p0)];
    }
    if (p0 <= 0)
      tail_pivots<0, MASKED>(e, t, p0, ti, tj, buf, rm);
    if (p0 <= 1)
      tail_pivots<1, MASKED>(e, t, p0, ti, tj, buf, rm);
    if (p0 <= 2)
      tail_pivots<2, MASKED>(e, t, p0, ti, tj, buf, rm);
    tail_pivots<3, MASKED>(e, t, p0, ti, tj, buf, rm);
    bool finite = true;
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b)
        finite = finite && __builtin_isfinite(e[a][b]);
    const uint64_t bad = __ballot(!finite);
    if ((tid & (kWave - 1)) == 0)
      flags[tid / kWave] = bad != 0;
    lds_barrier<kTailThreads>();
    const bool ok = (flags[0] | flags[1] | flags[2] | flags[3]) == 0;
    if (MASKED || ok)
    {
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b)
          if (a >= p0 && b >= p0)
            base[kTailBlock * (stride * (a - p0) + (b - p0))] = e[a][b];
    }
    lds_barrier<kTailThreads>();
    return ok;
  }

  // Rows of a substitution in levels of sixteen (DevRows), one task to a DPP row: lane k
  // forms the products 16 g + k, the row subtracts them in order.  Records are read two
  // levels ahead, as in coop_levels_piped; x[n] is a zero for the empty slots' lanes.
  __device__ inline void tail_rows(const DevRows& r, const double* A, double* x, double m1)
  {
    const int tid = threadIdx.x;
    const int nl = r.n_levels;
    struct Rec
    {
      uint32_t h;
      uint4 t;
    };
    auto load = [&](int l) {
      const int at = l < nl ? l : 0;
      Rec c;
      c.h = r.heads[at * kRowSlots + (tid >> 4)];
      c.t = r.terms[at * kTailThreads + tid];
      return c;
    };
    if (nl == 0)
      return;
    auto step = [&](int l, const Rec& cur, Rec& ahead) {
      if (l >= nl)
        return;
      const int groups = const_load(r.groups, l);
      ahead = load(l + 2);
      settle(cur.t);
      settle(uint4{ cur.h, 0u, 0u, 0u });
      const uint32_t o = cur.h & 0xffffu, d = cur.h >> 16;
      double v = x[o];
      const double dv = d < kUnitDivisor ? A[d] : 1.0;
      const double p0 = A[cur.t.x & 0xffffu] * x[cur.t.x >> 16];
      if (groups <= 1)
      {
        v = ordered_sub16<0>(v, p0, m1);
      }
      else
      {
        const double p1 = A[cur.t.y & 0xffffu] * x[cur.t.y >> 16];
        if (groups == 2)
        {
          v = ordered_sub16<0>(v, p0, m1);
          v = ordered_sub16<0>(v, p1, m1);
        }
        else
        {
          const double p2 = A[cur.t.z & 0xffffu] * x[cur.t.z >> 16];
          const double p3 = A[cur.t.w & 0xffffu] * x[cur.t.w >> 16];
          v = ordered_sub16<0>(v, p0, m1);
          v = ordered_sub16<0>(v, p1, m1);
          v = ordered_sub16<0>(v, p2, m1);
          v = ordered_sub16<0>(v, p3, m1);
        }
      }
      if (d < kUnitDivisor)
        v = v / dv;
      if ((tid & 15) == 0)
        x[o] = v;
      lds_barrier<kTailThreads>();
    };
    Rec r0 = load(0), r1 = load(1), r2;
    for (int l = 0; l < nl; l += 3)
    {
      step(l, r0, r2);
      step(l + 1, r1, r0);
      step(l + 2, r2, r1);
    }
  }

  // Rows 16 (G - p0) + 15 down to 16 (G - p0) of the block's back substitution.  xg[g]: lane
  // l holds x of column 16 (g - p0) + l % 16, zero until it is known, so the products of the
  // columns up to the row's own are zeros; z: lane i holds the forward result of row i.
  template<int G, bool MASKED>
  __device__ __forceinline__ void tail_back(double (&xg)[4], const DevTail& t, int p0, const double* block, double z,
                                            double m1)
  {
    const int l16 = threadIdx.x & 15;
    const int stride = t.size + 1;
    const int first = kTailBlock * (G - p0);
    const double* row = block + (first + kTailBlock - 1) * stride;  // the current row
    double u[4], diag;
#pragma unroll
    for (int g = G; g < 4; ++g)
      u[g] = row[kTailBlock * (g - p0) + l16];
    diag = row[first + kTailBlock - 1];
    auto rows = [&](auto quad) {
      constexpr int K0 = decltype(quad)::value;
      for (int rr = K0 + 3; rr >= K0; --rr)
      {
        const int i = first + rr;
        // the next row's operands (the last row reads row 0 of the block again, unused)
        const double* next = i > 0 ? row - stride : block;
        double un[4];
#pragma unroll
        for (int g = G; g < 4; ++g)
          un[g] = next[kTailBlock * (g - p0) + l16];
        const double dn = next[i > 0 ? i - 1 : 0];
        double v = readlane_f64(z, static_cast<uint32_t>(i));
        double p[4];
        const uint64_t rm = MASKED ? const_load(t.row_mask, i) : 0;
#pragma unroll
        for (int g = G; g < 4; ++g)
        {
          p[g] = u[g] * xg[g];
          if constexpr (MASKED)
          {
            const int j = kTailBlock * (g - p0) + l16;
            p[g] = j > i && ((rm >> j) & 1u) ? p[g] : 0.0;
          }
        }
        v = ordered_sub16<K0>(v, p[G], m1);
#pragma unroll
        for (int g = G + 1; g < 4; ++g)
          v = ordered_sub16<0>(v, p[g], m1);
        v = v / diag;
        xg[G] = l16 == rr ? v : xg[G];
#pragma unroll
        for (int g = G; g < 4; ++g)
          u[g] = un[g];
        diag = dn;
        row = next;
      }
    };
    rows(std::integral_constant<int, 12>{});
    rows(std::integral_constant<int, 8>{});
    rows(std::integral_constant<int, 4>{});
    rows(std::integral_constant<int, 0>{});
  }

  // The block's forward columns and back rows by one wavefront; xt: x of the block's first
  // row, replaced by the solution.  False (x unchanged) when a result is not finite, if not
  // MASKED.
  template<bool MASKED>
  __device__ inline bool tail_substitute(const DevTail& t, const double* block, double* xt, double m1)
  {
    const int lane = threadIdx.x & (kWave - 1), l16 = lane & 15;
    const int d = t.size, stride = d + 1;
    const int p0 = 4 - d / kTailBlock;
    const bool has = lane < d;
    const int r = has ? lane : 0;  // lanes past the block hold row 0, which no column changes
    double v = xt[r];
    const double* row = block + r * stride;
    const uint64_t rm = MASKED ? t.row_mask[r] : 0;
    double a[8];
#pragma unroll
    for (int q = 0; q < 8; ++q)
      a[q] = row[q];
    for (int c0 = 0; c0 < d; c0 += 8)
    {
      double an[8];
      const int n0 = c0 + 8 < d ? c0 + 8 : 0;
#pragma unroll
      for (int q = 0; q < 8; ++q)
        an[q] = row[n0 + q];
#pragma unroll
      for (int q = 0; q < 8; ++q)
      {
        const int c = c0 + q;
        const double xc = readlane_f64(v, static_cast<uint32_t>(c));
        if constexpr (MASKED)
        {
          const double nv = v - a[q] * xc;
          v = r > c && ((rm >> c) & 1u) ? nv : v;
        }
        else
        {
          v -= (r > c ? a[q] : 0.0) * xc;
        }
      }
#pragma unroll
      for (int q = 0; q < 8; ++q)
        a[q] = an[q];
    }
    double xg[4] = { 0.0, 0.0, 0.0, 0.0 };
    bool finite = !has || __builtin_isfinite(v);
    tail_back<3, MASKED>(xg, t, p0, block, v, m1);
    if (p0 <= 2)
      tail_back<2, MASKED>(xg, t, p0, block, v, m1);
    if (p0 <= 1)
      tail_back<1, MASKED>(xg, t, p0, block, v, m1);
    if (p0 <= 0)
      tail_back<0, MASKED>(xg, t, p0, block, v, m1);
#pragma unroll
    for (int g = 0; g < 4; ++g)
      finite = finite && __builtin_isfinite(xg[g]);
    const bool ok = __ballot(!finite) == 0;
    if (MASKED || ok)
    {
#pragma unroll
      for (int g = 0; g < 4; ++g)
        if (g >= p0 && lane < kTailBlock)
          xt[kTailBlock * (g - p0) + l16] = xg[g];
    }
    return ok;
  }

  // x <- U^-1 L^-1 x (x[n] = 0 behind it); masked: the factor holds values that are not
  // finite.  Ends with a barrier.
  __device__ inline void tail_solve(const DevTail& t, const double* A, double* x, bool masked)
  {
    double m1 = -1.0;
    asm("" : "+v"(m1));
    tail_rows(t.fwd, A, x, m1);
    if (threadIdx.x < kWave)
    {
      const double* block = A + t.head;
      double* xt = x + t.first;
      bool done = false;
      if (!masked)
        done = tail_substitute<false>(t, block, xt, m1);
      if (!done)
        tail_substitute<true>(t, block, xt, m1);
    }
    lds_barrier<kTailThreads>();
    tail_rows(t.bwd, A, x, m1);
  }
}  // namespace micm_hip
