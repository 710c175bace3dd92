// Work split of the shared-activation kernels (wq_mid.hip: 5 to 64 rows;
// wq_w8a8.hip: up to 255 rows), host only.
#pragma once

#include "wq_common.h"

namespace wq {

constexpr int kMidTilesPerWave = 2;   // 16-row tiles per wave

// Tile groups of 2 P tiles (P wave pairs per workgroup), S k splits; us is
// mid_split's estimate, which leaves out a constant of about 4 us (launch,
// first loads, parity sum; over 140 shapes x 20 row counts measured times lie
// within 12 % of estimate + 4.2).
struct MidSplit {
  int p, s;
  int64_t groups;
  double us = 0;
};

inline int64_t mid_groups(int64_t ntile, int p) {
  return (ntile + p * kMidTilesPerWave - 1) / (p * kMidTilesPerWave);
}

// Split partials: one 1 KiB unit per tile, 16-row chunk and split, behind the
// counter region (which other split kernels keep at zero in a shared
// workspace).
inline size_t mid_partial_bytes(const MidSplit& m, int64_t nz, int mc) {
  return m.s <= 1 ? 0 : kSplitCounterBytes + (size_t)(m.groups * nz * m.s) * m.p * kMidTilesPerWave * mc * 1024;
}

// The (P, S) of least estimated time.  Timing-only copies of the kernels
// showed what bounds them: leaving out the MFMAs or the LDS reads changes
// nothing, leaving out the x copies their share of the bytes, so a compute
// unit takes in about 35 KB/us whatever it holds (16 B per cycle; one
// workgroup of 72 or 128 KiB in flight or two alike), and all of them
// together what memory gives, about 5.5 MB/us.  Hence
//   rounds of workgroups over 256 compute units x bytes per workgroup / 35 KB
//   (at least the whole weight / 5.5 MB; a tenth of it on top, so that of two
//   splits at that bound the finer one wins)
//   + the partial sums: their launch 1.5 us, a second round of loads beyond
//   six splits 1 us, their bytes out and back at 4 MB/us.
// P = 4 or 5: eight or ten tiles a workgroup.  Ten is for grids of more than
// 128 groups of eight, whose rounds it can even out: 5120->34816 (2176 tiles)
// takes 218 workgroups in one round instead of 272 in two (us, eight -> ten:
// W8A8 M = 48 51.5 -> 39.2, INT8 M = 40 55.7 -> 41.0, W4 M = 40 43 -> 36.5),
// 5120->17408 in two splits the same (W8A8 M = 48 28.7 -> 26.0, INT8 M = 24 27.8
// -> 24.1, W4 M = 56 30.7 -> 27.1; W4 M = 24 20.4 -> 20.7).  On narrow N ten waves
// lost to eight at the same bytes (W4 17408->5120 M = 8 18.5 us against 15.8).
// Beyond 64 rows ten waves' registers would spill.
// w_tile / x_stage: bytes of one tile's weights and of the workgroup's x in one
// stage; nst stages; nz row blocks; mc 16-row chunks.
inline MidSplit mid_split(int64_t ntile, int64_t nst, double w_tile, double x_stage, int64_t nz, int mc) {
  MidSplit best{4, 1, mid_groups(ntile, 4)};
  double best_us = 1e30;
  const int most = mc <= 4 && mid_groups(ntile, 4) * nz > 128 ? 5 : 4;
  for (int p = 4; p <= most; ++p) {
    MidSplit m{p, 1, mid_groups(ntile, p)};
    for (m.s = 1; m.s <= 16 && m.s * 5 <= nst * 3; ++m.s) {
      if (mid_partial_bytes(m, nz, mc) > kSplitWorkspaceMaxBytes) break;
      const double rounds = (double)((m.groups * nz * m.s + 255) / 256);
      const double stages = (double)((nst + m.s - 1) / m.s);
      const double fill = rounds * stages * (p * kMidTilesPerWave * w_tile + x_stage) / 35e3;
      const double stream = (double)ntile * (double)nst * w_tile / 5.5e6;
      double us = (fill > stream ? fill : stream) + 0.1 * fill;
      if (m.s > 1) us += (m.s > 6 ? 2.5 : 1.5) + 2.0 * (double)mid_partial_bytes(m, nz, mc) / 4e6;
      if (us < best_us) {
        best_us = us;
        best = m;
        best.us = us;
      }
    }
    if (nst * 3 < 5) {   // a single stage: the loop above has no S to try
      m.s = 1;
      const double us = (double)((m.groups * nz + 255) / 256) * (p * kMidTilesPerWave * w_tile + x_stage) / 35e3;
      if (p == 4 || us < best_us) {
        best_us = us;
        best = m;
        best.us = us;
      }
    }
  }
  return best;
}

// wq_batch.hip's plan: R blocks per workgroup in flight, S splits, groups of
// eight tiles; r == 0 for the shapes it has none for.  us is its time, fitted to
// 256 shapes of 12 to 32 rows (10 % at most off): a chain of R blocks per 16-row
// chunk, the partial sums of two splits, and the tiles.
constexpr int64_t kW4BatchMaxTiles = 1152;
struct W4BatchPlan {
  int mc, r, s, groups;
  double us;
};
inline W4BatchPlan w4_batch_plan(int64_t m, int64_t n, int64_t k) {
  const int64_t ntile = (n + 15) / 16, nblk = k / kW4BlockK;
  if (m < 12 || m > 32 || k % kW4BlockK != 0 || ntile <= 512 || ntile > kW4BatchMaxTiles || nblk > 20) return {};
  const int mc = (int)((m + 15) / 16), groups = (int)((ntile + 7) / 8);
  for (int r : {10, 8, 5, 4}) {
    const int s = (int)(nblk / r);
    if (nblk % r != 0 || r * mc * 4 % 8 != 0) continue;   // the x copies split evenly over eight waves
    if (s > 2 || s * groups > 256) return {};             // more than one round of workgroups
    return {mc, r, s, groups,
            1.6 + 0.5 * mc + (0.40 + 0.07 * mc) * r + (s > 1 ? 1.3 + 0.5 * mc : 0.0) + 0.5 * (double)ntile / 1152};
  }
  return {};
}

// The plan where that kernel is estimated the fastest, else r == 0 (wq_mid.hip).
W4BatchPlan w4_batch_route(int64_t m, int64_t n, int64_t k);

}  // namespace wq
