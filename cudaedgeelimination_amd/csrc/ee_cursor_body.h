// The row of one deletion set, shared by the row producer (ee_cursor.hip) and
// the cost kernel that makes its own rows (ee_kopt.hip).
#pragma once

#include <cmath>
#include <cstdint>
#include <limits>

#include "ee_internal.h"

namespace ee {

// C(n, j) for j in 1..4 and n < 2^16, exact in 64 bits.
__host__ __device__ inline uint64_t Binom(uint64_t n, uint32_t j) {
  if (n < j) return 0;
  switch (j) {
    case 1:
      return n;
    case 2:
      return n * (n - 1) / 2;
    case 3:
      return n * (n - 1) / 2 * (n - 2) / 3;
    default:
      return (n * (n - 1) / 2) * ((n - 2) * (n - 3) / 2) / 6;
  }
}

// The smallest m with C(m, j) >= r, for 1 <= r <= C(2^16 - 1, j): from the
// estimate m^j / j! ~ r (shifted by the mean of its j factors), corrected
// with exact binomials: about two of them instead of one per step of a
// binary search (a block of 4,096 k = 5 sets evaluated as masks, 16 sets to a
// wavefront: 31.6 -> 28 us).
__host__ __device__ inline uint32_t SmallestWithBinom(uint64_t r, uint32_t j) {
  if (j == 1) return static_cast<uint32_t>(r);
  const float factorial = j == 2 ? 2.0f : (j == 3 ? 6.0f : 24.0f);
  const float root = exp2f(log2f(static_cast<float>(r) * factorial) / static_cast<float>(j));
  uint32_t m = static_cast<uint32_t>(root) + j / 2;
  while (m > j && Binom(m - 1, j) >= r) --m;
  while (Binom(m, j) < r) ++m;
  return m;
}

// The row of deletion set `rank` (BuildKOptCostTask's ports and summed deleted
// cost) and its sorted positions in pos; false where the cost overflows int64
// (the row's cost is then 0).  The set is unranked in the combinatorial
// number system: the index of slot s is the largest v whose preceding choices
// (indices prev+1 .. v-1, each followed by C(labels - u, rem) completions)
// number at most the remaining rank; by the hockey-stick identity those
// number C(labels - prev, rem + 1) - C(labels - v + 1, rem + 1).
__device__ inline bool CursorRow(const KoptCursor& c, uint32_t k, uint64_t rank, uint64_t (&pos)[kMaxK],
                                 ee_kopt_task* row) {
  pos[0] = c.selectable[0];
  uint32_t prev = 0;
  for (uint32_t s = 1; s < k; ++s) {
    const uint32_t j = k - s;
    const uint64_t total = Binom(c.labels - prev, j);
    const uint32_t m = SmallestWithBinom(total - rank, j);
    rank -= total - Binom(m, j);
    prev = c.labels - m + 1;
    pos[s] = c.selectable[prev];
  }
  for (uint32_t s = 1; s < k; ++s) {  // insertion sort, k <= 5
    const uint64_t v = pos[s];
    uint32_t t = s;
    while (t > 0 && pos[t - 1] > v) {
      pos[t] = pos[t - 1];
      --t;
    }
    pos[t] = v;
  }
  uint64_t sum = 0;
  bool overflow = false;
  for (uint32_t e = 0; e < k; ++e) {
    const uint64_t p = pos[e];
    const uint64_t next = p + 1 == c.tour_length ? 0 : p + 1;
    row->port_nodes[2 * e] = c.tour[p];
    row->port_nodes[2 * e + 1] = c.tour[next];
    overflow |= __builtin_add_overflow(sum, static_cast<uint64_t>(c.edge_costs[p]), &sum);
  }
  overflow |= sum > static_cast<uint64_t>(std::numeric_limits<int64_t>::max());
  row->deleted_cost = overflow ? 0 : static_cast<int64_t>(sum);
  return !overflow;
}

}  // namespace ee
