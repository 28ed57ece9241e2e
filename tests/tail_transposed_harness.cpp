// tail_transposed_harness.cpp -- CPU execution of the transposed substitutions' tables
// (TailTables::t_rows), for tests/test_tail_transposed.py.
#include "../micm_amd/csrc/mechanism.hpp"

#include <cstring>
#include <vector>

using namespace micm_hip;

namespace
{
  // false where a level's tasks touch one position
  bool run_rows(const RowLevels& r, int32_t first, int32_t last, const std::vector<double>& A, std::vector<double>& x,
                uint32_t zero_x)
  {
    for (int32_t l = first; l < last; ++l)
    {
      const std::vector<double> x0 = x;
      std::vector<char> written(x.size(), 0);
      for (int s = 0; s < kRowSlots; ++s)
      {
        const uint32_t o = r.heads.at(static_cast<size_t>(l) * kRowSlots + s) & 0xffffu;
        if (o != zero_x && written.at(o)++)
          return false;
      }
      for (int s = 0; s < kRowSlots; ++s)
      {
        const size_t slot = static_cast<size_t>(l) * kRowSlots + s;
        const uint32_t o = r.heads[slot] & 0xffffu, d = r.heads[slot] >> 16;
        double v = x0.at(o);
        for (int q = 0; q < kRowTerms; ++q)
        {
          const uint32_t tr = r.terms.at(slot * kRowTerms + 4 * (q % 16) + q / 16);
          if ((tr >> 16) != zero_x && written.at(tr >> 16))
            return false;
          v -= A.at(tr & 0xffffu) * x0.at(tr >> 16);
        }
        x[o] = d < kUnitDivisor ? v / A.at(d) : v;
      }
    }
    return true;
  }
}  // namespace

extern "C"
{
  // Solves U^T z = b, L^T x = z with the factor `alu` (its combined row storage), by the block's
  // tables (`x`) and row by row over the storage (`ref`).  Returns the block's size, 0 where there
  // is none, -1 where a table breaks its own rules.
  int tail_transposed(const micm_hip_mechanism_desc* desc, const double* alu, int64_t capacity, const double* b, double* x,
                      double* ref)
  {
    const MechanismTables t = compile_mechanism(*desc);
    const TailTables& T = t.tail;
    const int32_t n = static_cast<int32_t>(t.n_species);
    if (static_cast<int64_t>(t.alu_col.size()) > capacity)
      return -1;
    std::vector<std::vector<std::pair<int32_t, int32_t>>> column(n);  // (row, position), ascending rows
    for (int32_t i = 0; i < n; ++i)
      for (int32_t p = t.alu_row_ptr[i]; p < t.alu_row_ptr[i + 1]; ++p)
        column[t.alu_col[p]].emplace_back(i, p);
    std::memcpy(ref, b, sizeof(double) * n);
    for (int32_t i = 0; i < n; ++i)
    {
      for (auto [j, p] : column[i])
        if (j < i)
          ref[i] -= alu[p] * ref[j];
      ref[i] /= alu[t.alu_diag[i]];
    }
    for (int32_t i = n - 1; i >= 0; --i)
      for (auto [j, p] : column[i])
        if (j > i)
          ref[i] -= alu[p] * ref[j];
    if (T.size == 0)
      return 0;
    const int32_t d = T.size, stride = d + 1;
    std::vector<double> A(static_cast<size_t>(T.nnz) + 1, 0.0);
    int32_t head = 0;
    for (int32_t i = 0; i < n; ++i)
      for (int32_t p = t.alu_row_ptr[i]; p < t.alu_row_ptr[i + 1]; ++p)
        A.at(i >= T.first && t.alu_col[p] >= T.first
                 ? T.head + (i - T.first) * stride + t.alu_col[p] - T.first
                 : head++) = alu[p];
    const RowLevels& r = T.t_rows;
    if (head != T.head || T.t_fwd_padded % kRowPadding != 0 || r.n_levels() % kRowPadding != 0 ||
        r.n_levels() < kRowPadding || T.t_fwd_levels > T.t_fwd_padded || T.t_bwd_end > r.n_levels() ||
        r.heads.size() != static_cast<size_t>(r.n_levels() + 2) * kRowSlots || r.terms.size() != r.heads.size() * kRowTerms)
      return -1;
    std::vector<double> v(b, b + n);
    v.push_back(0.0);
    if (!run_rows(r, 0, T.t_fwd_levels, A, v, static_cast<uint32_t>(n)))
      return -1;
    const double* B = A.data() + T.head;
    double* xt = v.data() + T.first;
    for (int32_t c = 0; c < d; ++c)
    {
      xt[c] /= B[c * stride + c];
      for (int32_t q = c + 1; q < d; ++q)
        xt[q] -= B[c * stride + q] * xt[c];
    }
    for (int32_t i = d - 1; i >= 0; --i)
      for (int32_t j = i + 1; j < d; ++j)
        xt[i] -= B[j * stride + i] * xt[j];
    if (!run_rows(r, T.t_fwd_padded, T.t_bwd_end, A, v, static_cast<uint32_t>(n)) || v[n] != 0.0)
      return -1;
    std::memcpy(x, v.data(), sizeof(double) * n);
    return d;
  }
}
