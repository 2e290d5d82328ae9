// Device-side tile sources shared by the GEMM kernel families: a kernel runs
// `for (t = first(); t < total_tiles; t += stride())` and fetches the problem
// owning tile t.  GemmBatch launches one workgroup per tile (the loop runs once,
// tiles remapped so that each XCD gets a contiguous range); GemmGroup launches a
// persistent grid over a device-resident problem array (remapped the same way
// within every round of gridDim.x tiles).
#pragma once
#include "gemm.h"

namespace mk {

constexpr int NXCD = 8;

// Workgroups are dispatched round-robin over the XCDs.  Give XCD x a
// contiguous range of tile ids so that neighbouring tiles (which share A row
// panels / B column panels) are resident in the same L2.
__device__ __forceinline__ int xcd_remap(int t, int total) {
  const int q = total / NXCD, r = total % NXCD;
  const int x = t % NXCD, local = t / NXCD;
  return x * q + min(x, r) + local;
}

// Whole tiles and split tiles are remapped apart, so that every XCD gets its
// share of both.  Consecutive units of the split part are neighbouring tiles of
// one K slice, which share operand panels.
__device__ __forceinline__ int src_first(const GemmBatch& b) {
  const int u = blockIdx.x;
  if (u < b.full_tiles) return xcd_remap(u, b.full_tiles);
  return b.full_tiles + xcd_remap(u - b.full_tiles, (b.total_tiles - b.full_tiles) * b.ksplit);
}
__device__ __forceinline__ int src_stride(const GemmBatch&) { return 1 << 30; }
__device__ __forceinline__ int src_units(const GemmBatch& b) {
  return b.full_tiles + (b.total_tiles - b.full_tiles) * b.ksplit;
}
// Tile, K slice (-1: the whole range) and slice count of a unit.
__device__ __forceinline__ void src_unit(const GemmBatch& b, int u, int& tile, int& slice, int& nslice) {
  tile = u;
  slice = -1;
  nslice = 1;
  if (u >= b.full_tiles) {
    const int tail = b.total_tiles - b.full_tiles, v = u - b.full_tiles;
    tile = b.full_tiles + v % tail;
    slice = v / tail;
    nslice = b.ksplit;
  }
}
// Where a unit's partial tile of `elems` elements of type T goes.
template <class T>
__device__ __forceinline__ T* src_partial(const GemmBatch& b, int tile, int slice, int elems) {
  return static_cast<T*>(b.ws) + ((int64_t)(tile - b.full_tiles) * b.ksplit + slice) * elems;
}
__device__ __forceinline__ const GemmProb& src_prob(const GemmBatch& b, int t) {
  int pi = 0;
  while (pi + 1 < b.nprob && t >= b.p[pi + 1].tile_start) ++pi;
  return b.p[pi];
}

// Persistent grid: round r covers tiles [r G, r G + G) (G = gridDim.x); the
// remap gives each XCD a contiguous range of every round.
__device__ __forceinline__ int src_first(const GemmGroup&) { return xcd_remap(blockIdx.x, gridDim.x); }
__device__ __forceinline__ int src_stride(const GemmGroup&) { return gridDim.x; }
__device__ __forceinline__ int src_units(const GemmGroup& g) { return g.total_tiles; }
__device__ __forceinline__ void src_unit(const GemmGroup&, int u, int& tile, int& slice, int& nslice) {
  tile = u;
  slice = -1;
  nslice = 1;
}
template <class T>
__device__ __forceinline__ T* src_partial(const GemmGroup&, int, int, int) { return nullptr; }
__device__ __forceinline__ const GemmProb& src_prob(const GemmGroup& g, int t) {
  int lo = 0, hi = g.nprob - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (g.probs[mid].tile_start <= t) lo = mid;
    else hi = mid - 1;
  }
  return g.probs[lo];
}

// Resolve a descriptor pointer: absolute for GemmBatch, (slot, offset) for GemmGroup.
template <class T>
__device__ __forceinline__ T* resolve(const GemmBatch&, T* p) { return p; }
// Every operand lives in device (global) memory.  A pointer rebuilt from an
// integer loses that fact and would be accessed with flat instructions, whose
// completion counts on both the memory and the LDS counters; the round trip
// through the global address space lets the compiler emit global loads and
// stores again.
template <class T>
__device__ __forceinline__ T* as_global(T* p) {
  return (T*)((__attribute__((address_space(1))) T*)p);
}
// The same pointer typed in the global address space, for the access sites.
template <class T>
using gptr_t = __attribute__((address_space(1))) T*;
template <class T>
__device__ __forceinline__ gptr_t<T> gptr(T* p) {
  return (gptr_t<T>)p;
}
template <class T>
__device__ __forceinline__ T* resolve(const GemmGroup& g, T* p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const int slot = (int)(v >> 62);
  T* r = slot == 0 ? p : reinterpret_cast<T*>(const_cast<char*>(g.base[slot]) + (v & REL_MASK));
  return as_global(r);
}

// Epilogue C = alpha * acc + beta * C of an FM x FN grid of 16 x 16 accumulator
// blocks, item r of lane (li, lq) at C[row0 + 16 i + li][col0 + 16 j + cq(lq, r)]
// with cq = lq + 4 r (QMAJOR = false: the fp64 MFMA layout) or 4 lq + r
// (QMAJOR = true: the fp32-accumulating MFMA layouts).  With beta != 0 the
// 4 JB values of C of JB consecutive blocks of a row block are all fetched
// before any of them is stored, so their reads overlap (one round trip per
// batch instead of one per element; JB = 2 keeps the batch within the
// registers the main loop leaves free); out-of-range items read a clamped
// in-range address (branch-free) and are not stored.  beta == 0 never reads C.
template <bool QMAJOR, int FM, int FN, class V, int JB = 2>
__device__ __forceinline__ void epilogue_c(const V (&acc)[FM][FN], double* C, int64_t ldc, int M, int N, int row0,
                                           int col0, int li, int lq, double alpha, double beta) {
  static_assert(FN % JB == 0, "batch must divide the block columns");
  gptr_t<double> Cg = gptr(C);
  auto col_of = [&](int j, int r) { return col0 + j * 16 + (QMAJOR ? 4 * lq + r : lq + 4 * r); };
  const bool rd = beta != 0.0;
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int row = row0 + i * 16 + li;
#pragma unroll
    for (int j0 = 0; j0 < FN; j0 += JB) {
      double cin[JB * 4];
      if (rd) {
        const int64_t rc = min(row, M - 1);
#pragma unroll
        for (int j = 0; j < JB; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) cin[j * 4 + r] = Cg[rc + (int64_t)min(col_of(j0 + j, r), N - 1) * ldc];
      }
      if (row >= M) continue;
#pragma unroll
      for (int j = 0; j < JB; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int col = col_of(j0 + j, r);
          if (col >= N) continue;
          double v = alpha * (double)acc[i][j0 + j][r];
          if (rd) v += beta * cin[j * 4 + r];
          Cg[(int64_t)row + (int64_t)col * ldc] = v;
        }
    }
  }
  // Drain the stores here.  Their data registers are reused inside the next
  // tile's K loop, and without this wait the compiler's wait-count analysis
  // carries the pending stores around the tile loop and inserts a full
  // vmcnt(0) wait (on the K step's own global loads) into every K step.
  __builtin_amdgcn_s_waitcnt(0);
}

// Position of tile u of a problem: tile rows are grouped GROUP_M at a time so
// that consecutive tiles reuse the same A row panels.
constexpr int GROUP_M = 8;
__device__ __forceinline__ void tile_coords(const GemmProb& P, int u, int& tm, int& tn) {
  const int per_group = GROUP_M * P.tiles_n;
  const int g = u / per_group;
  const int first_m = g * GROUP_M;
  const int gsize = min(GROUP_M, P.tiles_m - first_m);
  tm = first_m + (u % per_group) % gsize;
  tn = (u % per_group) / gsize;
}

// K steps [s0, s1) of a slice, and the segment and depth where they start.
template <int BK>
__device__ __forceinline__ void slice_range(const GemmProb& P, int nsteps, int slice, int nslice, int& s0, int& s1,
                                            int& seg, int& k0) {
  s0 = 0;
  s1 = nsteps;
  seg = 0;
  k0 = 0;
  if (slice < 0) return;
  s0 = (int)((int64_t)slice * nsteps / nslice);
  s1 = (int)((int64_t)(slice + 1) * nsteps / nslice);
  int r = s0;
  for (; seg + 1 < P.nseg; ++seg) {
    const int n = (P.seg[seg].K + BK - 1) / BK;
    if (r < n) break;
    r -= n;
  }
  k0 = r * BK;
}

// A wave's accumulators to its part of a partial tile: 16 x 16 block (i, j) of
// wave w at block index (w FM + i) FN + j, four consecutive items a lane.
template <int FM, int FN, class V, class T>
__device__ __forceinline__ void store_partial(const V (&acc)[FM][FN], T* out, int wave, int lane) {
  typedef __attribute__((address_space(1))) V gV;
  gV* o = (gV*)out + (int64_t)wave * FM * FN * 64 + lane;
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) o[(i * FN + j) * 64] = acc[i][j];
  __builtin_amdgcn_s_waitcnt(0);   // as in epilogue_c
}

// Adds the partial tiles of the split tiles slice by slice (always in the same
// order, in float64) and writes C = alpha * sum + beta * C.  One wave per 16 x 16
// block: it reads ksplit contiguous runs of 64 lanes x 4 items, so the pass runs
// at the memory rate of its ksplit reads and one write of C.  Block layout as
// written by store_partial; WGM x WGN waves of FM x FN blocks make a tile.
template <bool QMAJOR, int WGM, int FM, int FN, int WGN, class V>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(GemmBatch b) {
  constexpr int NBLK = WGM * WGN * FM * FN;
  const int tail = b.total_tiles - b.full_tiles;
  const int g = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (g >= tail * NBLK) return;
  const int lane = threadIdx.x & 63, li = lane & 15, lq = lane >> 4;
  const int tile = b.full_tiles + g / NBLK, blk = g % NBLK;
  const GemmProb& P = src_prob(b, tile);
  int tm, tn;
  tile_coords(P, tile - P.tile_start, tm, tn);
  const int wave = blk / (FM * FN), i = blk / FN % FM, j = blk % FN;
  const int row = tm * (WGM * FM * 16) + (wave % WGM) * FM * 16 + i * 16 + li;
  const int col0 = tn * (WGN * FN * 16) + (wave / WGM) * FN * 16 + j * 16;
  typedef const __attribute__((address_space(1))) V gV;
  gV* p = (gV*)b.ws + ((int64_t)(tile - b.full_tiles) * b.ksplit * NBLK + blk) * 64 + lane;
  double s[4] = {0.0, 0.0, 0.0, 0.0};
  for (int k0 = 0; k0 < b.ksplit; k0 += 4) {
    V v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = p[(int64_t)min(k0 + k, b.ksplit - 1) * NBLK * 64];
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int r = 0; r < 4; ++r) s[r] += k0 + k < b.ksplit ? (double)v[k][r] : 0.0;
  }
  if (row >= P.M) return;
  gptr_t<double> C = gptr(P.C);
  double cin[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int col = col0 + (QMAJOR ? 4 * lq + r : lq + 4 * r);
    if (P.beta != 0.0 && col < P.N) cin[r] = C[row + (int64_t)col * P.ldc];
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int col = col0 + (QMAJOR ? 4 * lq + r : lq + 4 * r);
    double v = P.alpha * s[r];
    if (P.beta != 0.0) v += P.beta * cin[r];
    if (col < P.N) C[row + (int64_t)col * P.ldc] = v;
  }
}

}  // namespace mk
