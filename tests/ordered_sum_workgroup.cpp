// ordered_sum_workgroup.cpp -- ordered_sum (micm_amd/csrc/ordered_sum.hpp) on the host, every
// thread of its workgroup a context of its own, for tests/test_ordered_sum_workgroup.py.  A
// wavefront runs until all its lanes stand at a barrier, then the next wavefront does, in
// ascending or descending order: of any two wavefronts either one is a whole stretch between
// barriers ahead, so a value that one still has to read when another may write it again is seen
// changed.  Lanes of one wavefront meet at its exchange operations.
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <stdexcept>
#include <vector>

#include <ucontext.h>

#define __device__
#define __forceinline__ inline
#define __host__
#define MICM_WORKGROUP_ON_HOST

namespace emulation
{
  constexpr int kLanes = 64;

  struct Thread
  {
    ucontext_t context;
    std::vector<char> stack;
    int at = 0;  // 0: runs, 1: at an exchange, 2: at a barrier, 3: done
    int site = 0;
    double value = 0.0;
  };

  struct Group
  {
    std::vector<Thread> threads;
    ucontext_t scheduler;
    int current = 0;
  };
  inline Group* group = nullptr;

  inline void stop(int at, int site)
  {
    Thread& t = group->threads[group->current];
    t.at = at;
    t.site = site;
    swapcontext(&t.context, &group->scheduler);
  }

  // the values that the wavefront's lanes brought
  inline double* exchange(double v, double* all)
  {
    const int first = group->current / kLanes * kLanes;
    group->threads[group->current].value = v;
    stop(1, 0);
    for (int l = 0; l < kLanes; ++l)
      all[l] = group->threads[first + l].value;
    stop(1, 1);  // every lane has them
    return all;
  }

  struct ThreadIndex
  {
    struct X
    {
      operator int() const { return group->current; }
    } x;
  };
}  // namespace emulation

static const emulation::ThreadIndex threadIdx;

inline int lane_of_thread() { return emulation::group->current % emulation::kLanes; }

inline uint64_t __ballot(bool v)
{
  double all[64];
  emulation::exchange(v ? 1.0 : 0.0, all);
  uint64_t m = 0;
  for (int l = 0; l < 64; ++l)
    m |= uint64_t(all[l] != 0.0) << l;
  return m;
}
inline bool __any(bool v) { return __ballot(v) != 0; }
inline int __ffsll(unsigned long long v) { return v ? __builtin_ctzll(v) + 1 : 0; }
inline double __shfl_up(double v, int d)
{
  double all[64];
  emulation::exchange(v, all);
  const int l = lane_of_thread();
  return l >= d ? all[l - d] : v;
}
inline double __shfl_xor(double v, int d)
{
  double all[64];
  emulation::exchange(v, all);
  return all[lane_of_thread() ^ d];
}
inline void __syncthreads(int site = __builtin_LINE()) { emulation::stop(2, site); }

namespace micm_hip
{
  template<int NT>
  inline void lds_barrier(int site = __builtin_LINE())
  {
    emulation::stop(2, site);
  }
  inline double readlane_f64(double v, uint32_t l)
  {
    double all[64];
    return emulation::exchange(v, all)[l];
  }
  // v + p[0] + ... + p[15], p[k] being lane k's of the sixteen lanes (m1 = 1)
  template<int K0>
  inline double ordered_sub16(double v, double p, double)
  {
    double all[64];
    emulation::exchange(p, all);
    const int first = lane_of_thread() / 16 * 16;
    for (int k = K0; k < 16; ++k)
      v += all[first + k];
    return v;
  }
}  // namespace micm_hip

#include "../micm_amd/csrc/ordered_sum.hpp"

namespace
{
  using namespace emulation;

  // everything that a run needs, for the contexts' entry
  struct Run
  {
    const double* terms;
    int64_t n;
    void* scratch;
    std::vector<double> result;
  };
  Run* run_now = nullptr;

  template<int NT, int K>
  void thread_main()
  {
    const double* t = run_now->terms;
    const int64_t n = run_now->n;
    const double v = micm_hip::ordered_sum<NT, K>(
        n, [=](int64_t f) { return t[f]; }, *static_cast<micm_hip::SumScratch<NT>*>(run_now->scratch));
    run_now->result[group->current] = v;
    stop(3, 0);
  }

  // 0: every thread has the same sum (in *sum); 1: wavefronts at different barriers; 2: threads
  // with different sums
  template<int NT, int K>
  int sum(const double* terms, int64_t n, int descending, double* out)
  {
    Group g;
    micm_hip::SumScratch<NT> scratch;
    std::memset(static_cast<void*>(&scratch), 0xff, sizeof scratch);  // NaN where nothing was written
    Run run{ terms, n, &scratch, std::vector<double>(NT) };
    g.threads.resize(NT);
    group = &g;
    run_now = &run;
    for (Thread& t : g.threads)
    {
      t.stack.resize(32 * 1024);
      getcontext(&t.context);
      t.context.uc_stack.ss_sp = t.stack.data();
      t.context.uc_stack.ss_size = t.stack.size();
      t.context.uc_link = nullptr;
      makecontext(&t.context, thread_main<NT, K>, 0);
    }
    constexpr int W = NT / kLanes;
    while (true)
    {
      for (int o = 0; o < W; ++o)
      {
        const int first = (descending ? W - 1 - o : o) * kLanes;
        if (g.threads[first].at == 3)
          continue;
        // from one exchange to the next until the wavefront's lanes stand at a barrier
        do
        {
          for (int l = 0; l < kLanes; ++l)
          {
            g.current = first + l;
            g.threads[first + l].at = 0;
            swapcontext(&g.scheduler, &g.threads[first + l].context);
          }
          for (int l = 1; l < kLanes; ++l)
            if (g.threads[first + l].at != g.threads[first].at || g.threads[first + l].site != g.threads[first].site)
              return 1;
        } while (g.threads[first].at == 1);
      }
      for (int w = 1; w < W; ++w)
        if (g.threads[w * kLanes].at != g.threads[0].at || g.threads[w * kLanes].site != g.threads[0].site)
          return 1;
      if (g.threads[0].at == 3)
        break;
    }
    for (int t = 1; t < NT; ++t)
      if (std::memcmp(&run.result[t], &run.result[0], sizeof(double)) != 0 &&
          (run.result[t] == run.result[t] || run.result[0] == run.result[0]))
        return 2;
    *out = run.result[0];
    return 0;
  }
}  // namespace

extern "C" int ordered_sum_workgroup(const double* terms, int64_t n, int threads, int descending, double* out)
{
  return threads == 1024 ? sum<1024, 8>(terms, n, descending, out) : sum<512, 16>(terms, n, descending, out);
}
