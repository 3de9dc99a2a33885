// Host rules of the WCSPH passes' lists and launches (no GPU types, so that
// they can be checked at sizes no test could run).
#pragma once

#include <algorithm>
#include <cmath>

namespace sphx {

// Particles of one launch: a grid holds fewer than 2^32 threads, and a
// particle takes up to 32 of them.
constexpr int WC_LAUNCH = 1 << 26;

// f(first, m) for the launches of n particles.
template <class F>
inline void wc_launches(int n, F&& f) {
  for (int left = n; left > 0; left -= WC_LAUNCH) f(n - left, std::min(left, WC_LAUNCH));
}

// Particles up to which the list routes address the 16-byte records with
// 32-bit byte offsets.
constexpr int WC_LIST_PARTICLES = 1 << 28;

// Entries per particle of the neighbour list: 1.6x the neighbours of a
// lattice of the particles' spacing within the support, plus slack (a
// particle with more scans the cells), a multiple of 8, at most 512 so that a
// workgroup's lists fit in LDS, and at most `most` (0: no such limit, < 0: no
// list).  0: no list, every particle scans.
inline int wc_entries(int n, double spacing, double reach, int most) {
  if (n > WC_LIST_PARTICLES || most < 0) return 0;
  const double ratio = spacing > 0 ? std::min(reach / spacing, 8.0) : 4.0;
  const int cap = (int)(1.6 * 4.18879 * ratio * ratio * ratio + 8.0);
  const int fit = std::max(16, std::min(512, (cap + 7) & ~7));
  return most ? std::min(fit, most & ~7) : fit;
}

}  // namespace sphx
