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
// Rows of kManyProducts or more, whose products fall on the same columns
// again and again, mark a column the first time only, and rows whose columns
// lie more than kWide apart are sorted, since finding the bits would pass over
// every word in between.  Against a marker array and a sort for every row:
// dense 400 x 400 25.5 -> 22.5 ms (marking every product: 54), rows whose
// columns lie 500000 apart 75 -> 67 ms (passing over the words: 112), a mesh
// 105 -> 57 ms, 7 diagonals 39 -> 24 ms.
constexpr long kManyProducts = 128;
constexpr int kWide = 4096 * 64;

template <typename F>
void product_rows(const data_d_matrix& A, const data_d_matrix& B, F f) {
  const int m = A.num_rows, n = B.num_cols;
  if (m <= 0) return;  // an empty matrix may have no arrays
  const int *ar = A.row, *ac = A.col, *br = B.row, *bc = B.col;
  const dataType *av = A.val, *bv = B.val;
  std::vector<int> list_(n), mark_;
  std::vector<double> acc_(n, 0.0);
  std::vector<uint64_t> bits_(n / 64 + 1, 0), sum_(n / 4096 + 1, 0);
  int* list = list_.data();
  double* acc = acc_.data();
  uint64_t *bits = bits_.data(), *sum = sum_.data();
  long longest = 0;
  for (int k = 0; k < B.num_rows; k++) longest = std::max(longest, (long)br[k + 1] - br[k]);
  for (int i = 0; i < m; i++) {
    const int p0 = ar[i], p1 = ar[i + 1];
    long products = (p1 - p0) * longest;  // at most
    if (products >= kManyProducts) {
      products = 0;
      for (int p = p0; p < p1; p++) products += br[ac[p] + 1] - br[ac[p]];
    }
    int lo = n, hi = -1;
    const auto set = [&](int j) {
      bits[j >> 6] |= 1ull << (j & 63);
      sum[j >> 12] |= 1ull << (j >> 6 & 63);
      lo = std::min(lo, j);
      hi = std::max(hi, j);
    };
    if (products < kManyProducts) {
      for (int p = p0; p < p1; p++) {
        const double a = av[p];
        const int k = ac[p], q1 = br[k + 1];
        for (int q = br[k]; q < q1; q++) {
          const int j = bc[q];
          set(j);
          acc[j] += a * bv[q];
        }
      }
    } else {
      if (mark_.empty()) mark_.assign(n, -1);
      int* mark = mark_.data();
      for (int p = p0; p < p1; p++) {
        const double a = av[p];
        const int k = ac[p], q1 = br[k + 1];
        for (int q = br[k]; q < q1; q++) {
          const int j = bc[q];
          if (mark[j] != i) {
            mark[j] = i;
            set(j);
          }
          acc[j] += a * bv[q];
        }
      }
    }
    int cnt = 0;
    if (hi - lo < kWide) {
      for (int s = lo >> 12; s <= hi >> 12; s++)
        for (; sum[s]; sum[s] &= sum[s] - 1) {
          const int w = s * 64 + __builtin_ctzll(sum[s]);
          for (; bits[w]; bits[w] &= bits[w] - 1) list[cnt++] = w * 64 + __builtin_ctzll(bits[w]);
        }
    } else {
      for (int p = p0; p < p1; p++)
        for (int q = br[ac[p]]; q < br[ac[p] + 1]; q++) {
          const int j = bc[q];
          const uint64_t bit = 1ull << (j & 63);
          if (!(bits[j >> 6] & bit)) continue;
          bits[j >> 6] &= ~bit;
          sum[j >> 12] = 0;
          list[cnt++] = j;
        }
      std::sort(list, list + cnt);
    }
    f(i, cnt, list, acc);
    for (int t = 0; t < cnt; t++) acc[list[t]] = 0.0;
  }
}

// Places of a row's columns in an ascending list of columns: forwards from
// one column to the next, by binary search from the first column that is out
// of order.
struct RowPlaces {
  const int *list, *end, *at;
  int before = -1;
  bool ordered = true;
  RowPlaces(const int* list_, int cnt) : list(list_), end(list_ + cnt), at(list_) {}
  // The index in the list of the row's next column, -1 where it is not there.
  int next(int c) {
    if (c < before) ordered = false;
    before = c;
    if (ordered)
      while (at < end && *at < c) at++;
    else
      at = std::lower_bound(list, end, c);
    return at < end && *at == c ? (int)(at - list) : -1;
  }
};

}  // namespace lace
