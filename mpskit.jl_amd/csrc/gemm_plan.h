// Host choice of the tile and of the K split of a plain (non-grouped) GEMM
// launch, from a model of the time each choice takes.
//
// A CU works on the workgroups it holds at the matrix cores' rate times an
// efficiency that grows with their number, because the wavefronts of one
// workgroup wait together at each K step (for operands and at the barrier) and
// only another workgroup's fill that time.  A launch whose tiles do not give
// every CU the same number of workgroups therefore loses twice, in idle CUs and
// in waiting; cutting the tiles of the last round along K (in the extreme all
// of them) repairs both for one write and one read of the partial tiles.
//
// And the host's check of what the FP64 LDS-DMA kernel takes (f64_fit).
#pragma once
#include <algorithm>

#include "gemm.h"

namespace mk {

// One tile kernel: its K step, the time of a step at the matrix cores' rate
// (us, one workgroup alone on a CU), the efficiency with 1, 2, 3, >= 4
// workgroups on the CU, how many a CU holds, and the bytes of a partial tile.
struct TileModel {
  struct Eff { double v[4]; };
  int bm, bn, bk;
  double step_us;
  Eff eff;
  int occ;
  int part_bytes;
};

struct TileChoice {
  SplitPlan split;
  double us = 1e30;
};

constexpr int PLAN_CUS = 256;
constexpr int MAX_KSPLIT = 16;
// The least K steps of a slice: below that the first loads' latency dominates.
constexpr int MIN_SLICE_STEPS = 4;

inline double tile_rounds_us(const TileModel& m, int64_t units, double steps) {
  if (units <= 0) return 0.0;
  const int64_t n = cdiv(units, PLAN_CUS);
  const int r = (int)std::min<int64_t>(std::min<int64_t>(n, m.occ), 4);
  return (double)n * steps * m.step_us / m.eff.v[r - 1];
}

// The best split of `tiles` tiles of `nsteps` K steps under model m; `ws` tells
// whether a workspace is there.  Launch and first-load time count the same for
// every choice, except the 4 us of the second launch of a split one.
inline TileChoice plan_tile(const TileModel& m, int64_t tiles, int64_t nsteps, bool ws) {
  TileChoice best;
  best.split.full = (int)tiles;
  best.us = tile_rounds_us(m, tiles, (double)nsteps);
  if (!ws || tiles <= 0) return best;
  const int64_t round = (int64_t)PLAN_CUS * m.occ;
  const int64_t fulls[3] = {0, tiles / PLAN_CUS * PLAN_CUS, tiles / round * round};
  for (int64_t full : fulls) {
    const int64_t tail = tiles - full;
    if (tail <= 0) continue;
    const double base = tile_rounds_us(m, full, (double)nsteps);
    for (int s = 2; s <= MAX_KSPLIT && nsteps / s >= MIN_SLICE_STEPS; ++s) {
      // past one round of workgroups a finer cut gains nothing
      if (tail * (s - 1) >= round || (size_t)tail * s * m.part_bytes > GEMM_WS_BYTES) break;
      // partial tiles written and read back at about 6 TB/s (partly out of the Infinity Cache)
      const double us = base + tile_rounds_us(m, tail * s, (double)cdiv(nsteps, s)) + 4.0 +
                        2.0 * (double)tail * s * m.part_bytes / 6.0e6;
      if (us < best.us) {
        best.us = us;
        best.split.full = (int)full;
        best.split.ksplit = s;
      }
    }
  }
  return best;
}

// Tiles of a launch and the fewest K steps of its problems, for tile m.
inline void tile_counts(const TileModel& m, const ProbSpec* probs, int nprob, int64_t& tiles, int64_t& nsteps) {
  tiles = 0;
  nsteps = 1ll << 40;
  for (int i = 0; i < nprob; ++i) {
    const int64_t t = cdiv(probs[i].M, m.bm) * cdiv(probs[i].N, m.bn);
    if (t == 0) continue;
    int64_t n = 0;
    for (int s = 0; s < probs[i].nseg; ++s) n += cdiv(probs[i].seg[s].K, m.bk);
    tiles += t;
    nsteps = std::min(nsteps, n);
  }
  if (tiles == 0) nsteps = 0;
}

inline TileChoice plan_launch(const TileModel& m, const ProbSpec* probs, int nprob, bool ws) {
  int64_t tiles, nsteps;
  tile_counts(m, probs, nprob, tiles, nsteps);
  return plan_tile(m, tiles, nsteps, ws);
}

// What gemm_f64_dma_kernel with bm x bn tiles makes of one problem: BUF_NO, or its
// form for odd sizes and 8-byte alignment, or the one for whole pairs.  Its byte
// offsets within a tile are 32 bits wide and a load's scalar part is not masked, so
// the bound counts K up to the end of the last K step, not to the last element: an
// operand stored along its rows has loads for those k too, whose lanes are masked.
enum BufFit { BUF_NO = 0, BUF_ODD = 1, BUF_EVEN = 2 };
constexpr int64_t F64_BK = 16;
inline BufFit f64_fit(const ProbSpec& ps, GemmShape sh, int bm, int bn) {
  BufFit fit = BUF_EVEN;
  for (int s = 0; s < ps.nseg; ++s) {
    const SegSpec& g = ps.seg[s];
    if (g.K <= 0) continue;
    const int64_t K = cdiv(g.K, F64_BK) * F64_BK;
    // one past the largest offset, with the 16 bytes of a load
    const int64_t endA = (sh.ta ? K + (bm - 1) * g.lda : bm + (K - 1) * g.lda) * 8 + 16;
    const int64_t endB = (!sh.tb ? K + (bn - 1) * g.ldb : bn + (K - 1) * g.ldb) * 8 + 16;
    if (endA >= (1ll << 31) || endB >= (1ll << 31)) return BUF_NO;
    if ((uintptr_t)g.A % 8 || (uintptr_t)g.B % 8) return BUF_NO;
    if ((uintptr_t)g.A % 16 || (uintptr_t)g.B % 16 || g.lda % 2 || g.ldb % 2 || g.K % 2 || (!sh.ta && ps.M % 2) ||
        (sh.tb && ps.N % 2))
      fit = BUF_ODD;
  }
  return fit;
}

}  // namespace mk
