// tail_harness.cpp -- CPU execution of the tables of the factor's dense block
// (MechanismTables::tail, micm_amd/csrc/tail.hpp), for tests/test_tail.py.  Every level
// reads the values as they stood when it began, and every position is checked against the
// arrays' sizes.
#include "../micm_amd/csrc/mechanism.hpp"

#include <cmath>
#include <cstring>
#include <stdexcept>
#include <vector>

using namespace micm_hip;

namespace
{
  // the head's level schedule; false where two tasks of a level touch one position
  bool run_lu(const LevelSchedule& s, std::vector<double>& A)
  {
    for (int32_t l = 0; l < s.n_levels(); ++l)
    {
      const std::vector<double> A0 = A;
      std::vector<char> written(A.size(), 0);
      if (s.offsets[l + 1] - s.offsets[l] > 256)
        return false;
      for (int32_t t = s.offsets[l]; t < s.offsets[l + 1]; ++t)
      {
        const uint32_t o = s.tasks[2 * t] & 0xffffu;
        if (written.at(o)++)
          return false;
      }
      for (int32_t t = s.offsets[l]; t < s.offsets[l + 1]; ++t)
      {
        const uint32_t o = s.tasks[2 * t] & 0xffffu, d = s.tasks[2 * t] >> 16;
        double v = A0.at(o);
        for (uint32_t q = s.tasks[2 * t + 1]; q < s.tasks[2 * t + 3]; ++q)
        {
          const uint32_t a = s.terms[q] & 0xffffu, b = s.terms[q] >> 16;
          if (written.at(a) || written.at(b))
            return false;
          v -= A0[a] * A0[b];
        }
        if (d < kUnitDivisor)
        {
          if (written.at(d))
            return false;
          v /= A0[d];
        }
        A[o] = v;
      }
    }
    return true;
  }

  bool run_rows(const RowLevels& r, int32_t first, int32_t last, const std::vector<double>& A, std::vector<double>& x,
                uint32_t zero_x)
  {
    for (int32_t l = first; l < last; ++l)
    {
      const std::vector<double> x0 = x;
      std::vector<char> written(x.size(), 0);
      for (int s = 0; s < kRowSlots; ++s)
      {
        const uint32_t o = r.heads.at(l * kRowSlots + s) & 0xffffu;
        if (o != zero_x && written.at(o)++)
          return false;
      }
      for (int s = 0; s < kRowSlots; ++s)
      {
        const size_t slot = static_cast<size_t>(l) * kRowSlots + s;
        const uint32_t o = r.heads[slot] & 0xffffu, d = r.heads[slot] >> 16;
        double v = x0.at(o);
        for (int q = 0; q < 64; ++q)
        {
          const uint32_t tr = r.terms.at(slot * 64 + 4 * (q % 16) + q / 16);
          const bool pad = (tr >> 16) == zero_x;
          if (!pad && written.at(tr >> 16))
            return false;
          v -= A.at(tr & 0xffffu) * x0.at(tr >> 16);
        }
        if (d < kUnitDivisor)
          v /= A.at(d);
        x[o] = v;
      }
    }
    return true;
  }
}  // namespace

extern "C"
{
  // One cell as harness_factor_solve of schedule_harness.cpp, through the block: `lower` and
  // `upper` in the reference's storage, b solved.  masked: the block's products tested
  // against the fill pattern.  Returns the block's size, 0 where there is none, -1 where a
  // table breaks its own rules.
  int tail_factor_solve(const micm_hip_mechanism_desc* desc, const double* jac, double alpha, int masked, double* lower,
                        double* upper, double* b)
  {
    const MechanismTables t = compile_mechanism(*desc);
    const TailTables& T = t.tail;
    if (T.size == 0)
      return 0;
    const int32_t n = static_cast<int32_t>(t.n_species), d = T.size, stride = d + 1;
    if (d % kTailBlock != 0 || d > kTailMax || T.first != n - d || T.nnz != T.head + d * stride)
      return -1;
    std::vector<double> A(static_cast<size_t>(T.nnz) + 1, 0.0);
    for (size_t e = 0; e < T.jac_pos.size(); ++e)
      A.at(T.jac_pos[e]) = jac[e];
    for (int32_t i = 0; i < n; ++i)
      A.at(T.diag_pos[i]) += alpha;
    if (!run_lu(T.lu, A))
      return -1;
    double* B = A.data() + T.head;
    auto in = [&](int i, int j) { return (T.row_mask[i] >> j) & 1u; };
    for (int k = 0; k < d; ++k)
    {
      for (int i = k + 1; i < d; ++i)
        if (!masked || in(i, k))
          B[i * stride + k] = B[i * stride + k] / B[k * stride + k];
      for (int i = k + 1; i < d; ++i)
        for (int j = k + 1; j < d; ++j)
          if (!masked || (in(i, k) && in(k, j)))
            B[i * stride + j] -= B[i * stride + k] * B[k * stride + j];
    }
    // positions of the factor's elements
    std::vector<int32_t> pos;
    int32_t head = 0;
    for (int32_t i = 0; i < n; ++i)
      for (int32_t p = t.alu_row_ptr[i]; p < t.alu_row_ptr[i + 1]; ++p)
        pos.push_back(i >= T.first && t.alu_col[p] >= T.first ? T.head + (i - T.first) * stride + t.alu_col[p] - T.first
                                                              : head++);
    if (head != T.head)
      return -1;
    for (size_t p = 0; p < t.alu_lower.size(); ++p)
      lower[p] = t.alu_lower[p] >= 0 ? A.at(pos[t.alu_lower[p]]) : 1.0;
    for (size_t p = 0; p < t.alu_upper.size(); ++p)
      upper[p] = A.at(pos[t.alu_upper[p]]);
    std::vector<double> x(b, b + n);
    x.push_back(0.0);
    const uint32_t zero_x = static_cast<uint32_t>(n);
    if (T.fwd_padded % kRowPadding != 0 || T.rows.n_levels() % kRowPadding != 0 || T.rows.n_levels() < kRowPadding || T.fwd_levels > T.fwd_padded ||
        T.bwd_end > T.rows.n_levels() ||
        T.rows.heads.size() != static_cast<size_t>(T.rows.n_levels() + 2) * kRowSlots ||
        T.rows.terms.size() != T.rows.heads.size() * 64)
      return -1;
    if (!run_rows(T.rows, 0, T.fwd_levels, A, x, zero_x))
      return -1;
    double* xt = x.data() + T.first;
    for (int c = 0; c < d; ++c)
      for (int r = c + 1; r < d; ++r)
        if (!masked || in(r, c))
          xt[r] -= B[r * stride + c] * xt[c];
    for (int i = d - 1; i >= 0; --i)
    {
      double v = xt[i];
      for (int j = i + 1; j < d; ++j)
        if (!masked || in(i, j))
          v -= B[i * stride + j] * xt[j];
      xt[i] = v / B[i * stride + i];
    }
    if (!run_rows(T.rows, T.fwd_padded, T.bwd_end, A, x, zero_x) || x[n] != 0.0)
      return -1;
    std::memcpy(b, x.data(), sizeof(double) * n);
    return d;
  }

  // Tasks, levels: LU, forward, back.
  void tail_shape(const micm_hip_mechanism_desc* desc, int64_t* out)
  {
    const MechanismTables t = compile_mechanism(*desc);
    out[0] = t.tail.size;
    out[1] = t.tail.lu.n_levels();
    out[2] = t.tail.fwd_levels;
    out[3] = t.tail.rows.n_levels();
    out[4] = t.tail.nnz;
    out[5] = static_cast<int64_t>(t.term_process.size());
    out[6] = t.tail.lu.max_terms;
  }
}
