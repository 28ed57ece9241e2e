// ordered_sum_harness.cpp -- the arithmetic of micm_amd/csrc/ordered_sum.hpp on the host, for
// tests/test_ordered_sum.py: runs of eight terms composed in a balanced tree over the terms of
// one binade of the sum, the run that leaves the binade added term by term.
#include "../micm_amd/csrc/ordered_sum.hpp"

#include <vector>

using namespace micm_hip;

namespace
{
  RoundedRun tree(const std::vector<RoundedRun>& r, size_t b, size_t e)
  {
    if (e - b == 1)
      return r[b];
    const size_t h = (b + e) / 2;
    return run_then(tree(r, b, h), tree(r, h, e));
  }
}  // namespace

extern "C" double ordered_sum_host(const double* terms, int64_t n)
{
  constexpr int K = 8;
  double acc = 0.0;
  int64_t f = 0;
  auto add = [&](int64_t until) {
    for (; f < until && f < n; ++f)
      acc += terms[f];
  };
  while (f < n)
  {
    if (!sum_in_range(acc))
    {
      add(f + 1);
      continue;
    }
    const SumUnits u = sum_units(acc);
    std::vector<RoundedRun> runs;
    for (int64_t b = f; b < n; b += K)
    {
      double t[K];
      for (int q = 0; q < K; ++q)
        t[q] = b + q < n ? terms[b + q] : 0.0;
      bool ties;
      const double inc = run_without_ties<K>(t, u.scale, ties);
      runs.push_back(ties ? run_of<K>(t, u.scale) : RoundedRun{ { inc, inc } });
    }
    // the longest prefix that stays in the binade (by bisection over trees)
    size_t lo = 0, hi = runs.size();
    auto after = [&](size_t k) { return k ? u.m + tree(runs, 0, k).inc[is_odd(u.m) ? 1 : 0] : u.m; };
    if (after(hi) < kRunLimit)
    {
      acc = after(hi) * u.unit;
      break;
    }
    while (hi - lo > 1)
    {
      const size_t mid = (lo + hi) / 2;
      (after(mid) < kRunLimit ? lo : hi) = mid;
    }
    acc = after(lo) * u.unit;
    f += static_cast<int64_t>(lo) * K;
    add(f + K);
  }
  return acc;
}
