// ordered_sum.hpp -- a running sum of non-negative doubles, every addition rounded as if they
// were added one after another, by one workgroup in parallel.
//
// While a running sum stays within one binade it is a multiple m of u = 2^(e - 52), and adding
// t rounds t / u to a whole number, ties to the even sum: the new m depends on t and on the
// parity of m alone.  So a run of terms is a function of the parity it starts with (the
// increment of m for an even and for an odd start), such functions compose associatively, and
// a workgroup combines them with a scan; only the term that takes the sum into the next binade
// (one that is not finite among them) is added on its own, with the terms of its thread after
// it.  Sums outside [2^-900, 2^900) are added one by one.
#pragma once

#include <cstdint>
#include <cstring>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>

#include "tail.hpp"
#define MICM_HOST_DEVICE __host__ __device__
#else
// the arithmetic alone, for the host; with MICM_WORKGROUP_ON_HOST the workgroup's sum too, over
// the includer's own wavefront and barrier operations
#define MICM_HOST_DEVICE
#endif

namespace micm_hip
{
  // The increments, in units of the sum's last place, that a run of terms adds to an even and
  // to an odd sum (whole numbers); at most kRunLimit, which takes any sum out of its binade.
  struct RoundedRun
  {
    double inc[2];
  };
  constexpr double kRunLimit = 9007199254740992.0;  // 2^53

  MICM_HOST_DEVICE inline double run_limited(double v)
  {
    return v < kRunLimit ? v : kRunLimit;
  }

  // Whether a whole number is odd.
  MICM_HOST_DEVICE inline bool is_odd(double m)
  {
    const double h = m * 0.5;
    return __builtin_floor(h) != h;
  }

  MICM_HOST_DEVICE inline RoundedRun run_then(const RoundedRun& a, const RoundedRun& b)
  {
    return RoundedRun{ { run_limited(a.inc[0] + (is_odd(a.inc[0]) ? b.inc[1] : b.inc[0])),
                         run_limited(a.inc[1] + (is_odd(a.inc[1]) ? b.inc[0] : b.inc[1])) } };
  }

  // terms t[0 .. K), `scale` = 1 / u
  template<int K>
  MICM_HOST_DEVICE inline RoundedRun run_of(const double (&t)[K], double scale)
  {
    double even = 0.0, odd = 0.0;
    for (int q = 0; q < K; ++q)
    {
      const double x = run_limited(t[q] * scale);
      const double whole = __builtin_floor(x), part = x - whole;
      const double e = run_limited(even + whole), o = run_limited(odd + whole);
      even = part > 0.5 || (part == 0.5 && is_odd(e)) ? e + 1.0 : e;
      odd = part > 0.5 || (part == 0.5 && !is_odd(o)) ? o + 1.0 : o;
    }
    return RoundedRun{ { run_limited(even), run_limited(odd) } };
  }

  // The same where no term ties (`ties` false): one increment for both parities.
  template<int K>
  MICM_HOST_DEVICE inline double run_without_ties(const double (&t)[K], double scale, bool& ties)
  {
    double inc = 0.0;
    ties = false;
#pragma unroll
    for (int q = 0; q < K; ++q)
    {
      const double x = run_limited(t[q] * scale);
      const double near = __builtin_rint(x);
      ties = ties || __builtin_fabs(x - near) == 0.5;
      inc += near;
    }
    return run_limited(inc);
  }

  // The sum as a whole number of units, one unit, and one unit's inverse.
  struct SumUnits
  {
    double m, scale, unit;
  };

  MICM_HOST_DEVICE inline double double_from_bits(uint64_t b)
  {
    double d;
    memcpy(&d, &b, sizeof d);
    return d;
  }
  MICM_HOST_DEVICE inline uint64_t bits_of_double(double d)
  {
    uint64_t b;
    memcpy(&b, &d, sizeof b);
    return b;
  }

  MICM_HOST_DEVICE inline bool sum_in_range(double acc)
  {
    const int e = static_cast<int>(bits_of_double(acc) >> 52);  // acc >= 0
    return e >= 1023 - 900 && e < 1023 + 900;
  }

  MICM_HOST_DEVICE inline SumUnits sum_units(double acc)
  {
    const uint64_t b = bits_of_double(acc), e = b >> 52;
    return SumUnits{ static_cast<double>((b & 0xfffffffffffffull) | (uint64_t(1) << 52)),
                     double_from_bits((2 * 1023 + 52 - e) << 52), double_from_bits((e - 52) << 52) };
  }

#if defined(__HIPCC__) || defined(MICM_WORKGROUP_ON_HOST)
  constexpr int kSumChain = 2048;  // leading terms added as one chain

  template<int NT>
  struct SumScratch
  {
    double terms[kSumChain];
    double even[2][NT / 64], odd[2][NT / 64];
    int first[NT / 64];
    double acc;
    int next;
  };

  // term(f) for f = 0 .. n - 1 in order, by NT threads with K terms each a tile; the result on
  // every thread.  The first kSumChain terms, where the sum changes its binade often, are
  // added by one wavefront with one instruction each (ordered_sub16), 5.4 clocks a term: the
  // whole sum of a small State.  A tile costs about a microsecond, and one more for each
  // binade that the sum enters.
  template<int NT, int K, class Term>
  __device__ inline double ordered_sum(int64_t n, const Term& term, SumScratch<NT>& s)
  {
    constexpr int W = NT / 64;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t chain = n < kSumChain ? n : kSumChain;
    const int groups = static_cast<int>((chain + 15) / 16);
    // a wavefront has 64 K consecutive terms of a tile, 64 of them in each of its K registers
    // (coalesced); where their order matters they are read again, K consecutive ones a lane
    double t[K];
    auto load = [&](int64_t base, double (&v)[K]) {
#pragma unroll
      for (int q = 0; q < K; ++q)
      {
        const int64_t f = base + wave * (64 * K) + q * 64 + lane;
        v[q] = f < n ? term(f) : 0.0;
      }
    };
    auto load_ordered = [&](int64_t base, double (&v)[K]) {
#pragma unroll
      for (int q = 0; q < K; ++q)
      {
        const int64_t f = base + static_cast<int64_t>(tid) * K + q;
        v[q] = f < n ? term(f) : 0.0;
      }
    };
    for (int f = tid; f < 16 * groups; f += NT)
      s.terms[f] = f < chain ? term(f) : 0.0;
    if (kSumChain < n)
      load(kSumChain, t);
    __syncthreads();
    if (wave == 0)
    {
      double one = 1.0;
      asm("" : "+v"(one));
      double acc = 0.0;
      const double* p = s.terms + (lane & 15);
      double q[4];
#pragma unroll
      for (int k = 0; k < 4; ++k)
        q[k] = p[16 * (k < groups ? k : 0)];
      for (int g = 0; g < groups; g += 4)
      {
        double qn[4];
#pragma unroll
        for (int k = 0; k < 4; ++k)
          qn[k] = p[16 * (g + 4 + k < groups ? g + 4 + k : 0)];
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (g + k < groups)
            acc = ordered_sub16<0>(acc, q[k], one);
#pragma unroll
        for (int k = 0; k < 4; ++k)
          q[k] = qn[k];
      }
      if (lane == 0)
        s.acc = acc;
    }
    __syncthreads();
    double acc = s.acc;
    int pass = 0;  // the two buffers of the wavefronts' runs
    for (int64_t base = kSumChain; base < n; base += NT * K)
    {
      if (acc != acc)
        break;  // NaN stays
      // the next tile is read across this one's barriers, which wait for LDS only
      double ahead[K];
      if (base + NT * K < n)
        load(base + NT * K, ahead);
      int begin = 0;  // threads before it are done with this tile
      while (begin < NT)
      {
        double v[K];  // the lane's terms where the order matters
        if (acc == 0.0)
        {
          // the first lane with a term that is not zero adds its own
          load_ordered(base, v);
          bool any = false;
#pragma unroll
          for (int q = 0; q < K; ++q)
            any = any || v[q] != 0.0;
          const uint64_t who = __ballot(any && tid >= begin);
          if (lane == 0)
            s.first[wave] = who ? wave * 64 + __ffsll(static_cast<unsigned long long>(who)) - 1 : NT;
          lds_barrier<NT>();
          int first = NT;
          for (int w = 0; w < W; ++w)
            first = s.first[w] < first ? s.first[w] : first;
          if (first == NT)
          {
            lds_barrier<NT>();  // s.first is read before the next tile writes it
            break;
          }
          if (tid == first)
          {
#pragma unroll
            for (int q = 0; q < K; ++q)
              acc += v[q];
            s.acc = acc;
          }
          lds_barrier<NT>();
          acc = s.acc;
          begin = first + 1;
          lds_barrier<NT>();
          continue;
        }
        if (!sum_in_range(acc))
        {
          // wavefront after wavefront, lane after lane
          load_ordered(base, v);
          lds_barrier<NT>();  // the chain's s.acc is read before the first wavefront writes it
          for (int w = 0; w < W; ++w)
          {
            if (wave == w)
            {
#pragma unroll 1
              for (int l = 0; l < 64; ++l)
                if (w * 64 + l >= begin)
                {
#pragma unroll
                  for (int q = 0; q < K; ++q)
                    acc += readlane_f64(v[q], static_cast<uint32_t>(l));
                }
              if (lane == 0)
                s.acc = acc;
            }
            lds_barrier<NT>();
            acc = s.acc;
            lds_barrier<NT>();
          }
          break;
        }
        const SumUnits u = sum_units(acc);
        // the wavefront's run: one sum in any order where none of its terms ties, else
        // composed in order; terms of the tile before begin * K are done
        double x[K];
#pragma unroll
        for (int q = 0; q < K; ++q)
          x[q] = wave * (64 * K) + q * 64 + lane >= begin * K ? t[q] : 0.0;
        bool ties;
        double inc = run_without_ties<K>(x, u.scale, ties);
        const bool tied = __any(ties);
        RoundedRun run{ { 0.0, 0.0 } };
        auto scan = [&]() {
          // inclusive scan of the lanes' runs in order
          load_ordered(base, v);
          if (tid >= begin)
            run = run_of<K>(v, u.scale);
#pragma unroll 1
          for (int d = 1; d < 64; d *= 2)
          {
            RoundedRun before;
            before.inc[0] = __shfl_up(run.inc[0], d);
            before.inc[1] = __shfl_up(run.inc[1], d);
            if (lane >= d)
              run = run_then(before, run);
          }
        };
        if (!tied)
        {
#pragma unroll
          for (int d = 1; d < 64; d *= 2)
            inc = run_limited(inc + __shfl_xor(inc, d));
          if (lane == 0)
            s.even[pass][wave] = s.odd[pass][wave] = inc;
        }
        else
        {
          scan();
          if (lane == 63)
          {
            s.even[pass][wave] = run.inc[0];
            s.odd[pass][wave] = run.inc[1];
          }
        }
        lds_barrier<NT>();
        double m = u.m, m_wave = u.m;
#pragma unroll
        for (int w = 0; w < W; ++w)
        {
          m_wave = w == wave ? m : m_wave;
          m = run_limited(m + (is_odd(m) ? s.odd[pass][w] : s.even[pass][w]));
        }
        const int buffer = pass;
        pass ^= 1;
        if (m < kRunLimit)
        {
          acc = m * u.unit;
          break;
        }
        // the wavefront whose terms take the sum out of the binade finds the thread, which
        // adds its terms one by one
        if (m_wave < kRunLimit && m_wave + (is_odd(m_wave) ? s.odd[buffer][wave] : s.even[buffer][wave]) >= kRunLimit)
        {
          if (!tied)
            scan();
          RoundedRun before;
          before.inc[0] = __shfl_up(run.inc[0], 1);
          before.inc[1] = __shfl_up(run.inc[1], 1);
          const bool odd = is_odd(m_wave);
          const double m_before = lane == 0 ? m_wave : m_wave + (odd ? before.inc[1] : before.inc[0]);
          const double m_after = m_wave + (odd ? run.inc[1] : run.inc[0]);
          if (m_before < kRunLimit && m_after >= kRunLimit)
          {
            double a = m_before * u.unit;
#pragma unroll
            for (int q = 0; q < K; ++q)
              a += v[q];
            s.acc = a;
            s.next = tid + 1;
          }
        }
        lds_barrier<NT>();
        acc = s.acc;
        begin = s.next;
        lds_barrier<NT>();
      }
#pragma unroll
      for (int q = 0; q < K; ++q)
        t[q] = ahead[q];
    }
    return acc;
  }
#endif
}  // namespace micm_hip
