// product_rows.hpp -- rows of a sparse product on the host.
#pragma once

#include <algorithm>
#include <cstdint>
#include <vector>

#include "../../include/lace.h"

namespace lace {

// Rows of A B (CSR), one after another: f(i, cnt, list, acc) is given row
// i's cnt columns in ascending order and their sums acc[column].  Each sum
// runs over A's row in order.
//
// A bit per column (and one per 64 of them) marks the columns of the row and
// then gives them in order, without a sort and without a test per product
// (host part of a ParILU call on a mesh of 13800 rows: 13.5 -> 6.0 ms).
template <typename F>
void product_rows(const data_d_matrix& A, const data_d_matrix& B, F f) {
  const int m = A.num_rows, n = B.num_cols;
  const int *ar = A.row, *ac = A.col, *br = B.row, *bc = B.col;
  const dataType *av = A.val, *bv = B.val;
  std::vector<int> list_(n);
  std::vector<double> acc_(n, 0.0);
  std::vector<uint64_t> bits_(n / 64 + 1, 0), sum_(n / 4096 + 1, 0);
  int* list = list_.data();
  double* acc = acc_.data();
  uint64_t *bits = bits_.data(), *sum = sum_.data();
  for (int i = 0; i < m; i++) {
    int lo = n, hi = -1;
    for (int p = ar[i]; p < ar[i + 1]; p++) {
      const double a = av[p];
      const int k = ac[p], q1 = br[k + 1];
      for (int q = br[k]; q < q1; q++) {
        const int j = bc[q];
        bits[j >> 6] |= 1ull << (j & 63);
        sum[j >> 12] |= 1ull << (j >> 6 & 63);
        lo = std::min(lo, j);
        hi = std::max(hi, j);
        acc[j] += a * bv[q];
      }
    }
    int cnt = 0;
    for (int s = lo >> 12; s <= hi >> 12; s++)
      for (; sum[s]; sum[s] &= sum[s] - 1) {
        const int w = s * 64 + __builtin_ctzll(sum[s]);
        for (; bits[w]; bits[w] &= bits[w] - 1) list[cnt++] = w * 64 + __builtin_ctzll(bits[w]);
      }
    f(i, cnt, list, acc);
    for (int t = 0; t < cnt; t++) acc[list[t]] = 0.0;
  }
}

}  // namespace lace
