// rp_multisect.h -- how the search for a chain's lowest eigenvalue places its shifts
// (ring_lowest_eigen).  Plain C++ on the host.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstddef>

namespace rp {

// Shifts per chain of a multisection round: seven, and more where few chains are left open.  A
// round of up to kShiftTasks tasks takes as long as its longest chain, so a few chains get that
// many between them, up to kShiftMost each: on 256 chains of the 27-dof EVB the last two rounds,
// 12 chains and one, took 1.65 ms each with seven.
constexpr int kShifts = 7, kShiftTasks = 512, kShiftMost = 63;
inline int multisect_shifts(int chains_left) {
  return std::max(kShifts, std::min(kShiftMost, kShiftTasks / std::max(chains_left, 1)));
}

// Tasks of a round of at most `chains` chains
inline size_t multisect_tasks(int chains) { return std::max((size_t)kShifts * chains, (size_t)kShiftTasks); }

// Shift k = 1..m of a round, strictly inside (lo, hi) and rising with k.  The first round's
// crowd toward hi, down to 2^-7 of the bracket: eta_1 is usually within a few per cent of the
// Rayleigh quotient.  Later rounds split the bracket evenly.
inline double multisect_shift(double lo, double hi, bool first, int k, int m) {
  const double f = first ? 1.0 - std::exp2(-(double)(k * kShifts) / m) : (double)k / (m + 1);
  return lo + (hi - lo) * f;
}

}  // namespace rp
