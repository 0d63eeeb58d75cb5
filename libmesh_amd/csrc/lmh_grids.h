// lmh_grids.h -- grid sizes of the solvers' products.  Host arithmetic only.
#pragma once

#include <algorithm>
#include <cstdint>

namespace lmh {

// MI355X dispatches workgroups round-robin over its 8 XCDs
constexpr int NXCD = 8;

// Workgroups of a product over `blocks` row blocks on a GPU of `cus` CUs: `per_cu`
// on every CU at most, of which `resident` are there at once (0: no rounds, see
// below).
//
// Each publishes up to three partial sums (k_refresh, k_refresh16) into the
// second half of the partial buffer, 2 n_part doubles: no more than fit there,
// in whole rounds over the XCDs.
//
// At most one workgroup per row block.  Up to four rounds of what a GPU holds at
// once, a workgroup takes as many blocks as there are rounds: it loads one while
// it sums the last, and its consumers read fewer partial sums.  Q2 20^3 (4,050
// blocks) BiCGSTAB 6.8 -> 6.4 ms a solve, Q2 24^3 CG 7.69 -> 7.32, mixed 7.68 ->
// 7.37, Q1 50^3 CG 4.82 -> 4.63, TET4 40^3 products 49 -> 43 us; one round (Q2
// 12^3) 2.6 ms either way, and two rounds for it 2.8; beyond four rounds (Q2
// 30^3 and up) the full grid measures the same.
inline int product_grid(int cus, int per_cu, int resident, int n_part, int64_t blocks) {
  const int64_t fit = 2 * (int64_t)n_part / 3 / NXCD * NXCD;
  const int64_t most = std::min<int64_t>((int64_t)cus * per_cu, fit), held = (int64_t)cus * resident;
  int64_t want = blocks;
  if (blocks <= 4 * held) {
    const int64_t rounds = std::max<int64_t>(1, (blocks + held - 1) / held);
    want = (blocks + rounds - 1) / rounds;
  }
  return (int)std::min<int64_t>(most, (want + NXCD - 1) / NXCD * NXCD);
}

}  // namespace lmh
