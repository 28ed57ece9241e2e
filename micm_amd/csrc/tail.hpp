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
// (the masked forms), which is exact for every operand.
#pragma once

#include "coop.hpp"
#include "coop_tail.hpp"

#include <type_traits>

namespace micm_hip
{
  static_assert(kTailBuffer == 4 * kTailMax && kTailBlock == 16, "as coop_tail.hpp has them");

  // What depends on v is formed here, each time: kept across a Solve's loops, the straight-line
  // code's lane comparisons and addresses spill 46 vector and 350 scalar registers of the
  // three-wave build (an attempt: 60/200 46.5 -> 44.5 us, 20/50 27.5 -> 25.3, 210/560 130 -> 127.6).
  __device__ __forceinline__ void here(int& v)
  {
    asm volatile("" : "+v"(v));
  }

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

  // Pivots 16 (PA - p0) ... + 15 of a block of 4 - p0 sixteens: thread (ti, tj) holds the
  // elements (ti + 16 (a - p0), tj + 16 (b - p0)) as e[a][b].  At a pivot its row and column
  // go through LDS (two buffers, so one barrier a pivot); every four lanes divide one
  // column value each and pass the quotients on by DPP, and each thread updates its
  // elements below and right of the pivot.  Elements that are final already see a zero
  // factor, which leaves them as they are but for the sign of a zero in L; that matters to no
  // product, and with ZEROS (L is a result) they are kept by a select instead.
  template<int PA, bool ZEROS>
  __device__ __forceinline__ void tail_pivots(double (&e)[4][4], int ti, int tj, double* buf)
  {
#pragma unroll 1
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
      const double u_pa = tj > kk ? u[PA] : 0.0, l_pa = ti > kk ? l[PA] : 0.0;
#pragma unroll
      for (int a = PA; a < 4; ++a)
      {
        const double la = a == PA ? l_pa : l[a];
#pragma unroll
        for (int b = PA; b < 4; ++b)
        {
          if (ZEROS && b == PA)
          {
            const double v = e[a][b] - la * u[b];
            e[a][b] = tj > kk ? v : e[a][b];
          }
          else
          {
            e[a][b] -= la * (b == PA ? u_pa : u[b]);
          }
        }
        if (tj == kk && (a > PA || ti > kk))
          e[a][PA] = l[a];
      }
    }
  }

  // The block's own factorisation in place (A: the factor, its head and the block's sums
  // over the head's pivots final), 256 threads.  False (on every thread), the block left as
  // it is, when an element is not finite.  buf: kTailBuffer doubles; flags: one int per
  // wave.  ZEROS: tail_pivots.  Ends with a barrier.
  //
  // One pivot costs an LDS round trip with a barrier (140 clocks), a division (53) and ten
  // clocks for each of a thread's elements, whatever the fill; the level schedule of the
  // same rows takes two levels a pivot at 1,400 each.
  template<bool ZEROS>
  __device__ inline bool tail_factor(const DevTail& t, double* A, double* buf, int* flags)
  {
    int tid = threadIdx.x;
    here(tid);
    const int ti = tid >> 4, tj = tid & 15;
    const int p0 = 4 - t.size / kTailBlock;
    const int stride = t.size + 1;
    double* base = A + t.head + ti * stride + tj;
    double e[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b)
      {
        e[a][b] = 0.0;
        if (a >= p0 && b >= p0)
          e[a][b] = base[kTailBlock * (stride * (a - p0) + (b - p0))];
      }
    if (p0 <= 0)
      tail_pivots<0, ZEROS>(e, ti, tj, buf);
    if (p0 <= 1)
      tail_pivots<1, ZEROS>(e, ti, tj, buf);
    if (p0 <= 2)
      tail_pivots<2, ZEROS>(e, ti, tj, buf);
    tail_pivots<3, ZEROS>(e, ti, tj, buf);
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
    if (ok)
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

  // The block's factorisation in LDS with every product tested against the fill pattern
  // (for values that are not finite; small code, not speed).  Ends with a barrier.
  __device__ inline void tail_factor_masked(const DevTail& t, double* A)
  {
    const int tid = threadIdx.x;
    const int d = t.size, stride = d + 1;
    double* B = A + t.head;
#pragma unroll 1
    for (int k = 0; k < d; ++k)
    {
      const uint64_t rk = const_load(t.row_mask, k);
      if (tid > k && tid < d && ((t.row_mask[tid] >> k) & 1u))
        B[tid * stride + k] = B[tid * stride + k] / B[k * stride + k];
      __syncthreads();
#pragma unroll 1
      for (int q = tid; q < d * kTailMax; q += kTailThreads)
      {
        const int i = q / kTailMax, j = q % kTailMax;
        if (i > k && j > k && j < d && ((t.row_mask[i] >> k) & 1u) && ((rk >> j) & 1u))
          B[i * stride + j] -= B[i * stride + k] * B[k * stride + j];
      }
      __syncthreads();
    }
  }

  // Record of one thread in a level of DevRows: its DPP row's task and the lane's four terms.
  struct RowRecord
  {
    uint32_t head;
    uint4 terms;
  };

  __device__ __forceinline__ RowRecord row_record(const DevRows& r, int l)
  {
    // a uniform base and an unsigned lane offset: scalar address arithmetic
    const uint32_t* heads = r.heads + l * kRowSlots;
    const uint4* terms = r.terms + l * kTailThreads;
    return RowRecord{ heads[threadIdx.x >> 4], terms[threadIdx.x] };
  }

  // The records of a substitution's first two levels, read before it starts.
  struct RowsAhead
  {
    RowRecord r0, r1;
  };

  __device__ __forceinline__ RowsAhead rows_ahead(const DevRows& r)
  {
    return RowsAhead{ row_record(r, 0), row_record(r, 1) };
  }

  // What a level's tasks divide by: nothing, U[i][i], or L[i][i] (a lower factor whose diagonal
  // is not 1, as the single-phase substitution takes it).
  enum class Divide
  {
    kNone,
    kUpper,
    kLower
  };

  // One level of sixteen tasks, one to a DPP row: lane k forms the products 16 g + k, the
  // row subtracts them in order and divides (by one where a task has no divisor).  A
  // wavefront skips the groups that none of its tasks has (its lanes' words are all `pad`).
  // Every lane of a row writes the row's result: an exec mask around the write costs 70 of a
  // level's 570 clocks.
  template<Divide DIV>
  __device__ __forceinline__ void tail_level(const RowRecord& rec, uint32_t pad, const double* A, double* x, double m1,
                                             const double* ld)
  {
    const uint32_t o = rec.head & 0xffffu, d = rec.head >> 16;
    const uint32_t w[4] = { rec.terms.x, rec.terms.y, rec.terms.z, rec.terms.w };
    double v = x[o], dv = 1.0;
    if constexpr (DIV == Divide::kUpper)
      dv = A[d < kUnitDivisor ? d : 0];
    if constexpr (DIV == Divide::kLower)
      dv = ld[d == kUnitDivisor ? o : 0];
    auto product = [&](int g) { return A[w[g] & 0xffffu] * x[w[g] >> 16]; };
    const double p0 = product(0);
    if (!__any(w[1] != pad))
    {
      v = ordered_sub16<0>(v, p0, m1);
    }
    else if (!__any(w[2] != pad))
    {
      const double p1 = product(1);
      v = ordered_sub16<0>(v, p0, m1);
      v = ordered_sub16<0>(v, p1, m1);
    }
    else
    {
      const double p1 = product(1), p2 = product(2), p3 = product(3);
      v = ordered_sub16<0>(v, p0, m1);
      v = ordered_sub16<0>(v, p1, m1);
      v = ordered_sub16<0>(v, p2, m1);
      v = ordered_sub16<0>(v, p3, m1);
    }
    if constexpr (DIV != Divide::kNone)
    {
      v = v / ((DIV == Divide::kUpper ? d < kUnitDivisor : d == kUnitDivisor) ? dv : 1.0);
      asm("" : "+v"(v));
    }
    x[o] = v;
    lds_barrier<kTailThreads>();
  }

  // Rows 16 G + 15 down to 16 G of the back substitution of a block of D rows.  xg[g]: lane l
  // holds x of column 16 g + l % 16, zero until it is known, so the products of the columns
  // up to the row's own are zeros; zs: the forward result in LDS.  A row's operands are read
  // while the row before it is summed.  Every address is a lane's base and a constant: the
  // one wavefront issues an instruction every five clocks, so a row costs its products (5.4
  // clocks each) and its instructions: 9.6 us for both triangles of 64 rows, 3.6 us of 32
  // (13.6 and 5.7 us with the rows in a loop and their addresses formed in it).
  //
  // TRANSPOSED: the rows of L^T, the block's columns below its diagonal, without divisions.
  template<int D, int G, bool TRANSPOSED>
  __device__ __forceinline__ void tail_back(double (&xg)[D / kTailBlock], const double* block, const double* zs,
                                            double m1)
  {
    constexpr int Q = D / kTailBlock, S = D + 1;
    int l16 = threadIdx.x & 15;
    here(l16);
    constexpr int row = TRANSPOSED ? 1 : S, column = TRANSPOSED ? S : 1;
    const double* lane = block + l16 * column;
    double u[Q], diag = 1.0, z;
    constexpr int last = kTailBlock * G + kTailBlock - 1;
#pragma unroll
    for (int g = G; g < Q; ++g)
      u[g] = lane[last * row + kTailBlock * g * column];
    if constexpr (!TRANSPOSED)
      diag = block[last * S + last];
    z = zs[last];
#pragma unroll
    for (int rr = kTailBlock - 1; rr >= 0; --rr)
    {
      const int i = kTailBlock * G + rr;
      double v = z, p[Q];
#pragma unroll
      for (int g = G; g < Q; ++g)
        p[g] = u[g] * xg[g];
      const double d = diag;
      if (rr > 0)
      {
#pragma unroll
        for (int g = G; g < Q; ++g)
          u[g] = lane[(i - 1) * row + kTailBlock * g * column];
        if constexpr (!TRANSPOSED)
          diag = block[(i - 1) * S + i - 1];
        z = zs[i - 1];
      }
      __builtin_amdgcn_sched_barrier(0);
      if (rr >= 12)
        v = ordered_sub16<12>(v, p[G], m1);
      else if (rr >= 8)
        v = ordered_sub16<8>(v, p[G], m1);
      else if (rr >= 4)
        v = ordered_sub16<4>(v, p[G], m1);
      else
        v = ordered_sub16<0>(v, p[G], m1);
#pragma unroll
      for (int g = G + 1; g < Q; ++g)
        v = ordered_sub16<0>(v, p[g], m1);
      if constexpr (!TRANSPOSED)
      {
        v = v / d;
        asm("" : "+v"(v));  // on every lane: no branch around the division
      }
      xg[G] = l16 == rr ? v : xg[G];
    }
  }

  // The block's forward columns by one wavefront, lane = row; xt: x of the block's first row,
  // replaced by the result.  False (xt unchanged) when a result is not finite.
  template<int D>
  __device__ __forceinline__ bool tail_forward(const double* block, double* xt)
  {
    constexpr int S = D + 1;
    const int lane = threadIdx.x & (kWave - 1);
    int r = lane < D ? lane : 0;  // lanes past the block hold row 0, which no column changes
    here(r);
    double v = xt[r];
    const double* row = block + r * S;
    double a[8];
#pragma unroll
    for (int q = 0; q < 8; ++q)
      a[q] = row[q];
#pragma unroll
    for (int c0 = 0; c0 < D; c0 += 8)
    {
      double an[8];
      if (c0 + 8 < D)
      {
#pragma unroll
        for (int q = 0; q < 8; ++q)
          an[q] = row[c0 + 8 + q];
      }
#pragma unroll
      for (int q = 0; q < 8; ++q)
        if (c0 + q < D - 1)
          v -= (r > c0 + q ? a[q] : 0.0) * readlane_f64(v, static_cast<uint32_t>(c0 + q));
#pragma unroll
      for (int q = 0; q < 8; ++q)
        a[q] = an[q];
    }
    const bool ok = __ballot(!__builtin_isfinite(v)) == 0;
    if (ok && lane < D)
      xt[lane] = v;
    return ok;
  }

  // tail_forward with the block's U^T, lane = column: a column's result is divided by its
  // U[c][c] before the later ones subtract its products.  Every lane divides, so a column
  // costs a division and a broadcast (about 100 clocks) and a row of the block one
  // conflict-free read.
  template<int D>
  __device__ __forceinline__ bool tail_forward_transposed(const double* block, double* xt)
  {
    constexpr int S = D + 1;
    const int lane = threadIdx.x & (kWave - 1);
    int r = lane < D ? lane : 0;
    here(r);
    double v = xt[r];
    double u[4], d[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
    {
      u[q] = block[q * S + r];
      d[q] = block[q * S + q];
    }
#pragma unroll
    for (int c0 = 0; c0 < D; c0 += 4)
    {
      double un[4], dn[4];
      if (c0 + 4 < D)
      {
#pragma unroll
        for (int q = 0; q < 4; ++q)
        {
          un[q] = block[(c0 + 4 + q) * S + r];
          dn[q] = block[(c0 + 4 + q) * (S + 1)];
        }
      }
#pragma unroll
      for (int q = 0; q < 4; ++q)
      {
        double z = readlane_f64(v, static_cast<uint32_t>(c0 + q)) / d[q];
        asm("" : "+v"(z));
        const double nv = v - u[q] * z;
        v = r > c0 + q ? nv : (r == c0 + q ? z : v);
      }
#pragma unroll
      for (int q = 0; q < 4; ++q)
      {
        u[q] = un[q];
        d[q] = dn[q];
      }
    }
    const bool ok = __ballot(!__builtin_isfinite(v)) == 0;
    if (ok && lane < D)
      xt[lane] = v;
    return ok;
  }

  // The block's back rows by one wavefront, as tail_forward.
  template<int D, bool TRANSPOSED = false>
  __device__ __forceinline__ bool tail_backward(const double* block, double* xt, double m1)
  {
    constexpr int Q = D / kTailBlock;
    double xg[Q];
#pragma unroll
    for (int g = 0; g < Q; ++g)
      xg[g] = 0.0;
    if constexpr (Q > 3)
      tail_back<D, 3, TRANSPOSED>(xg, block, xt, m1);
    if constexpr (Q > 2)
      tail_back<D, 2, TRANSPOSED>(xg, block, xt, m1);
    if constexpr (Q > 1)
      tail_back<D, 1, TRANSPOSED>(xg, block, xt, m1);
    tail_back<D, 0, TRANSPOSED>(xg, block, xt, m1);
    bool finite = true;
#pragma unroll
    for (int g = 0; g < Q; ++g)
      finite = finite && __builtin_isfinite(xg[g]);
    const bool ok = __ballot(!finite) == 0;
    if (ok && (threadIdx.x & (kWave - 1)) < kTailBlock)
    {
#pragma unroll
      for (int g = 0; g < Q; ++g)
        xt[kTailBlock * g + (threadIdx.x & 15)] = xg[g];
    }
    return ok;
  }

  // tail_forward with every product tested against the fill pattern (for values that are not
  // finite, or a right-hand side with -0; loops, about a third of the speed).  ld: divide by
  // the rows' L[i][i] (null: they are 1).
  __device__ inline void tail_forward_masked(const DevTail& t, const double* block, double* xt, const double* ld)
  {
    const int lane = threadIdx.x & (kWave - 1);
    const int d = t.size, r = lane < d ? lane : 0;
    const double* row = block + r * (d + 1);
    const uint64_t rm = t.row_mask[r];
    double v = xt[r];
#pragma unroll 1
    for (int c = 0; c < d; ++c)
    {
      double xc = readlane_f64(v, static_cast<uint32_t>(c));
      if (ld)
      {
        xc = xc / ld[c];
        v = r == c ? xc : v;
      }
      const double nv = v - row[c] * xc;
      v = r > c && ((rm >> c) & 1u) ? nv : v;
    }
    if (lane < d)
      xt[lane] = v;
  }

  // tail_backward with every product tested against the fill pattern.
  __device__ inline void tail_backward_masked(const DevTail& t, const double* block, double* xt, double m1)
  {
    const int l16 = threadIdx.x & 15;
    const int d = t.size;
#pragma unroll 1
    for (int i = d - 1; i >= 0; --i)
    {
      const double* row = block + i * (d + 1);
      const uint64_t rm = const_load(t.row_mask, i);
      double v = xt[i];
#pragma unroll 1
      for (int j = l16; j < d; j += kTailBlock)
      {
        const double p = row[j] * xt[j];
        v = ordered_sub16<0>(v, j > i && ((rm >> j) & 1u) ? p : 0.0, m1);
      }
      xt[i] = v / row[i];
      coop_sync<kWave>();
    }
  }

  // Both transposed triangles of the block with every product tested against the fill pattern.
  __device__ inline void tail_transposed_masked(const DevTail& t, const double* block, double* xt, bool forward,
                                                double m1)
  {
    const int lane = threadIdx.x & (kWave - 1), l16 = threadIdx.x & 15;
    const int d = t.size, r = lane < d ? lane : 0;
    if (forward)
    {
      double v = xt[r];
#pragma unroll 1
      for (int c = 0; c < d; ++c)
      {
        double z = readlane_f64(v, static_cast<uint32_t>(c)) / block[c * (d + 1) + c];
        asm("" : "+v"(z));
        const double nv = v - block[c * (d + 1) + r] * z;
        v = r == c ? z : r > c && ((const_load(t.row_mask, c) >> r) & 1u) ? nv : v;
      }
      if (lane < d)
        xt[lane] = v;
      return;
    }
#pragma unroll 1
    for (int i = d - 1; i >= 0; --i)
    {
      double v = xt[i];
#pragma unroll 1
      for (int j = l16; j < d; j += kTailBlock)
      {
        const double p = block[j * (d + 1) + i] * xt[j];
        v = ordered_sub16<0>(v, j > i && ((t.row_mask[j] >> i) & 1u) ? p : 0.0, m1);
      }
      xt[i] = v;
      coop_sync<kWave>();
    }
  }

  // Both triangles of the block by one wavefront.
  template<int D>
  __device__ __forceinline__ void tail_substitute(const DevTail& t, const double* block, double* xt, bool masked,
                                                  double m1)
  {
    if (masked || !tail_forward<D>(block, xt))
      tail_forward_masked(t, block, xt, nullptr);
    coop_sync<kWave>();
    if (masked || !tail_backward<D>(block, xt, m1))
      tail_backward_masked(t, block, xt, m1);
  }

  // Both transposed triangles, U^T and then L^T.
  template<int D>
  __device__ __forceinline__ void tail_substitute_transposed(const DevTail& t, const double* block, double* xt,
                                                             bool masked, double m1)
  {
    if (masked || !tail_forward_transposed<D>(block, xt))
      tail_transposed_masked(t, block, xt, true, m1);
    coop_sync<kWave>();
    if (masked || !tail_backward<D, true>(block, xt, m1))
      tail_transposed_masked(t, block, xt, false, m1);
  }

  // Levels [begin, end) of the rows' list, the record of level l + 2 read while level l runs.
  // Three records rotate, unrolled by three so that none moves; level counts are padded to
  // multiples of three, so that the next levels start with the same record.
  template<Divide DIV>
  __device__ __forceinline__ void tail_levels(const DevTail& t, const DevRows& r, int begin, int end, const double* A, double* x,
                                              double m1, const double* ld, RowsAhead& ahead)
  {
    const uint32_t pad = static_cast<uint32_t>(t.nnz) | (static_cast<uint32_t>(t.first + t.size) << 16);
    RowRecord spare;
    auto step = [&](int l, const RowRecord& cur, RowRecord& next) {
      next = row_record(r, l + 2);
      if (l < end)
      {
        settle(cur.terms);
        settle(uint4{ cur.head, 0u, 0u, 0u });
        tail_level<DIV>(cur, pad, A, x, m1, ld);
      }
    };
#pragma unroll 1
    for (int l = begin; l < end; l += kRowPadding)
    {
      step(l, ahead.r0, spare);
      step(l + 1, ahead.r1, ahead.r0);
      step(l + 2, spare, ahead.r1);
    }
  }

  // x <- U^-1 L^-1 x (x[n] = 0 behind it); masked: the factor holds values that are not
  // finite, or x holds a -0.  The levels before and after the block are one list that ends in
  // its first two levels again, whose records the next solve starts with (`ahead`).  Ends with
  // a barrier.
  __device__ inline void tail_solve(const DevTail& t, const double* A, double* x, bool masked, RowsAhead& ahead)
  {
    double m1 = -1.0;
    asm("" : "+v"(m1));
    tail_levels<Divide::kNone>(t, t.rows, 0, t.fwd_levels, A, x, m1, nullptr, ahead);
    if (threadIdx.x < kWave)
    {
      const double* b = A + t.head;
      double* xt = x + t.first;
      switch (t.size)
      {
        case 16: tail_substitute<16>(t, b, xt, masked, m1); break;
        case 32: tail_substitute<32>(t, b, xt, masked, m1); break;
        case 48: tail_substitute<48>(t, b, xt, masked, m1); break;
        default: tail_substitute<64>(t, b, xt, masked, m1); break;
      }
    }
    lds_barrier<kTailThreads>();
    tail_levels<Divide::kUpper>(t, t.rows, t.fwd_padded, t.bwd_end, A, x, m1, nullptr, ahead);
  }

  // The same with the transposed factors: U^T, then L^T; x[n] = 0, `ahead` of t.t_rows.
  __device__ inline void tail_solve_transposed(const DevTail& t, const double* A, double* x, bool masked, RowsAhead& ahead)
  {
    double m1 = -1.0;
    asm("" : "+v"(m1));
    tail_levels<Divide::kUpper>(t, t.t_rows, 0, t.t_fwd_levels, A, x, m1, nullptr, ahead);
    if (threadIdx.x < kWave)
    {
      const double* b = A + t.head;
      double* xt = x + t.first;
      switch (t.size)
      {
        case 16: tail_substitute_transposed<16>(t, b, xt, masked, m1); break;
        case 32: tail_substitute_transposed<32>(t, b, xt, masked, m1); break;
        case 48: tail_substitute_transposed<48>(t, b, xt, masked, m1); break;
        default: tail_substitute_transposed<64>(t, b, xt, masked, m1); break;
      }
    }
    lds_barrier<kTailThreads>();
    tail_levels<Divide::kNone>(t, t.t_rows, t.t_fwd_padded, t.t_bwd_end, A, x, m1, nullptr, ahead);
  }

  // The same for a lower factor with the diagonal ld (rows without terms already divided).
  __device__ inline void tail_solve_lower_diagonal(const DevTail& t, const double* A, double* x, const double* ld,
                                                   RowsAhead& ahead)
  {
    double m1 = -1.0;
    asm("" : "+v"(m1));
    tail_levels<Divide::kLower>(t, t.rows, 0, t.fwd_levels, A, x, m1, ld, ahead);
    if (threadIdx.x < kWave)
    {
      tail_forward_masked(t, A + t.head, x + t.first, ld + t.first);
      coop_sync<kWave>();
      tail_backward_masked(t, A + t.head, x + t.first, m1);
    }
    lds_barrier<kTailThreads>();
    tail_levels<Divide::kUpper>(t, t.rows, t.fwd_padded, t.bwd_end, A, x, m1, nullptr, ahead);
  }
}  // namespace micm_hip
