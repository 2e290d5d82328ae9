// FP64 MFMA GEMM for CDNA4 (gfx950): v_mfma_f64_16x16x4_f64, LDS-staged
// BK = 16 deep tiles, double-buffered (straight to LDS in gemm_f64_dma_kernel, the
// usual one, or through registers), 256 threads = 4 waves of 64 lanes in a 2x2
// arrangement.  One workgroup computes one BM x BN output tile of one problem, summing every segment of that problem into the same
// accumulators before a single fused epilogue (alpha/beta and optional CB term).
#include "gemm_dev.h"
#include "gemm_plan.h"
#include "prof.h"

#include <algorithm>
#include <cstdlib>
#include <cstring>

namespace mk {
namespace {

typedef double dx4 __attribute__((ext_vector_type(4)));
typedef double dx2 __attribute__((ext_vector_type(2)));

constexpr int NT = 256;
constexpr int PAD = 16;     // LDS row padding (doubles): alternates 128-B bank halves

// Stage a tile whose contiguous memory direction is the LDS fast direction.
// element (r, k) lives at p[(r0 + r) + (k0 + k) * ld]; LDS tile S[k][r].
template <int R, int LDR, int BK, class Ptr>
__device__ __forceinline__ void load_fastdir(Ptr __restrict__ p, int64_t ld, int r0,
                                             int k0, int Rlim, int Klim, bool vec,
                                             dx2 (&reg)[R * BK / 2 / NT]) {
  constexpr int CH = R * BK / 2 / NT;
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int id = threadIdx.x + c * NT;
    const int k = id / (R / 2);
    const int r = (id % (R / 2)) * 2;
    const int gr = r0 + r, gk = k0 + k;
    dx2 v = {0.0, 0.0};
    if (gk < Klim) {
      const auto q = p + (int64_t)gr + (int64_t)gk * ld;
      if (vec && gr + 1 < Rlim) {
        v = *(const __attribute__((address_space(1))) dx2*)q;
      } else {
        if (gr < Rlim) v.x = q[0];
        if (gr + 1 < Rlim) v.y = q[1];
      }
    }
    reg[c] = v;
  }
}

template <int R, int LDR, int BK>
__device__ __forceinline__ void store_fastdir(double (*S)[LDR], const dx2 (&reg)[R * BK / 2 / NT]) {
  constexpr int CH = R * BK / 2 / NT;
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int id = threadIdx.x + c * NT;
    const int k = id / (R / 2);
    const int r = (id % (R / 2)) * 2;
    *reinterpret_cast<dx2*>(&S[k][r]) = reg[c];
  }
}

// Stage a tile whose contiguous memory direction is k.
// element (r, k) lives at p[(k0 + k) + (r0 + r) * ld]; LDS tile S[k][r ^ kswz(k)].
// The 16 lanes that share a column write rows k = 0, 2, ..., 30; with a row
// length that is a multiple of 32 doubles they would all hit one bank pair, so
// the column index is XORed with bits 1..4 of k (a permutation inside each
// aligned 32-column group, undone by the fragment reads).
__device__ __forceinline__ int kswz(int k) { return k & 30; }

template <int R, int LDR, int BK, class Ptr>
__device__ __forceinline__ void load_kdir(Ptr __restrict__ p, int64_t ld, int r0, int k0,
                                          int Rlim, int Klim, bool vec,
                                          dx2 (&reg)[R * BK / 2 / NT]) {
  constexpr int CH = R * BK / 2 / NT;
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int id = threadIdx.x + c * NT;
    const int r = id / (BK / 2);
    const int k = (id % (BK / 2)) * 2;
    const int gr = r0 + r, gk = k0 + k;
    dx2 v = {0.0, 0.0};
    if (gr < Rlim) {
      const auto q = p + (int64_t)gk + (int64_t)gr * ld;
      if (vec && gk + 1 < Klim) {
        v = *(const __attribute__((address_space(1))) dx2*)q;
      } else {
        if (gk < Klim) v.x = q[0];
        if (gk + 1 < Klim) v.y = q[1];
      }
    }
    reg[c] = v;
  }
}

template <int R, int LDR, int BK>
__device__ __forceinline__ void store_kdir(double (*S)[LDR], const dx2 (&reg)[R * BK / 2 / NT]) {
  constexpr int CH = R * BK / 2 / NT;
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int id = threadIdx.x + c * NT;
    const int r = id / (BK / 2);
    const int k = (id % (BK / 2)) * 2;
    S[k][r ^ kswz(k)] = reg[c].x;
    S[k + 1][r ^ kswz(k)] = reg[c].y;
  }
}

template <int BM, int BN, bool TA, bool TB, class Src>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(2)))
void gemm_f64_kernel(Src src) {
  constexpr int BK = 16;
  constexpr int LDA_S = BM + PAD;
  constexpr int LDB_S = BN + PAD;
  constexpr int WM = BM / 2, WN = BN / 2;
  constexpr int FM = WM / 16, FN = WN / 16;
  constexpr int CHA = BM * BK / 2 / NT;
  constexpr int CHB = BN * BK / 2 / NT;
  static_assert(CHA >= 1 && CHB >= 1, "tile too small for 256 threads");

  __shared__ double As[2][BK][LDA_S];
  __shared__ double Bs[2][BK][LDB_S];

  for (int un = src_first(src); un < src_units(src); un += src_stride(src)) {
  int t, slice, nslice;
  src_unit(src, un, t, slice, nslice);
  const GemmProb& P = src_prob(src, t);
  int tm, tn;
  tile_coords(P, t - P.tile_start, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm0 = (wave & 1) * WM;
  const int wn0 = (wave >> 1) * WN;
  const int li = lane & 15;   // row (A) / column (B, D) inside a 16x16 block
  const int lk = lane >> 4;   // k slot (A, B) / row quad (D)

  dx4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = dx4{0.0, 0.0, 0.0, 0.0};

  int nsteps = 0;
  for (int s = 0; s < P.nseg; ++s) nsteps += (P.seg[s].K + BK - 1) / BK;

  dx2 ra[CHA], rb[CHB];
  // descriptor of the segment being loaded, read from the problem array once
  // per segment rather than once per K step
  typedef const __attribute__((address_space(1))) double* gptr;   // operands are in device memory
  struct Cur {
    gptr A;
    gptr B;
    int64_t lda, ldb;
    int K;
    bool vec;
  } cur{};
  int cur_s = -1;
  const int M = P.M, N = P.N;
  auto load = [&](int s, int k0) {
    if (s != cur_s) {
      const GemmSeg& S = P.seg[s];
      cur.A = (gptr)static_cast<const double*>(resolve(src, S.A));
      cur.B = (gptr)static_cast<const double*>(resolve(src, S.B));
      cur.lda = S.lda;
      cur.ldb = S.ldb;
      cur.K = S.K;
      cur.vec = S.vec != 0;
      cur_s = s;
    }
    if (!TA) load_fastdir<BM, LDA_S, BK>(cur.A, cur.lda, m0, k0, M, cur.K, cur.vec, ra);
    else     load_kdir<BM, LDA_S, BK>(cur.A, cur.lda, m0, k0, M, cur.K, cur.vec, ra);
    if (!TB) load_kdir<BN, LDB_S, BK>(cur.B, cur.ldb, n0, k0, N, cur.K, cur.vec, rb);
    else     load_fastdir<BN, LDB_S, BK>(cur.B, cur.ldb, n0, k0, N, cur.K, cur.vec, rb);
  };
  auto store = [&](int buf) {
    if (!TA) store_fastdir<BM, LDA_S, BK>(As[buf], ra);
    else     store_kdir<BM, LDA_S, BK>(As[buf], ra);
    if (!TB) store_kdir<BN, LDB_S, BK>(Bs[buf], rb);
    else     store_fastdir<BN, LDB_S, BK>(Bs[buf], rb);
  };

  int s, k0, step0, step1;
  slice_range<BK>(P, nsteps, slice, nslice, step0, step1, s, k0);
  if (step1 > step0) {
    load(s, k0);
    store(0);
  }
  __syncthreads();
  int buf = 0;
  int kcur = step1 > step0 ? P.seg[s].K : 0;
  for (int step = step0; step < step1; ++step) {
    int ns = s, nk0 = k0 + BK;
    if (nk0 >= kcur) {
      ns = s + 1;
      nk0 = 0;
      kcur = ns < P.nseg ? P.seg[ns].K : 0;
    }
    const bool has_next = step + 1 < step1;
    if (has_next) load(ns, nk0);
#pragma unroll
    for (int kk = 0; kk < BK / 4; ++kk) {
      double a[FM], b[FN];
      const int kr = kk * 4 + lk;
      const int sa = TA ? kswz(kr) : 0;    // K-contiguous operands were stored swizzled
      const int sb = TB ? 0 : kswz(kr);
#pragma unroll
      for (int i = 0; i < FM; ++i) a[i] = As[buf][kr][(wm0 + i * 16 + li) ^ sa];
#pragma unroll
      for (int j = 0; j < FN; ++j) b[j] = Bs[buf][kr][(wn0 + j * 16 + li) ^ sb];
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(b[j], a[i], acc[i][j], 0, 0, 0);
    }
    if (has_next) store(buf ^ 1);
    __syncthreads();
    buf ^= 1;
    s = ns;
    k0 = nk0;
  }

  // epilogue.  The v_mfma_f64_16x16x4f64 D layout puts item r of lane (li, lk)
  // at block row lk + 4 r, column li; with the B fragment as first operand the
  // block is C^T, so the lane holds C[row li][col lk + 4 r]: the 16 lanes of a
  // quarter-wave store 16 consecutive rows (128 B) of one column.
  if (slice < 0)
    epilogue_c<false, FM, FN, dx4, 1>(acc, resolve(src, P.C), P.ldc, P.M, P.N, m0 + wm0, n0 + wn0, li, lk, P.alpha, P.beta);
  else
    store_partial(acc, src_partial<double>(src, t, slice, BM * BN), wave, lane);
  }  // units
}

// ---------------------------------------------------------------------------
// Operands straight to LDS (buffer_load ... lds, 16 bytes a lane): no staging
// registers and no LDS stores, so a K step is 8 DMA loads, the fragment reads and
// the MFMAs.  A load needs its address aligned to 4 bytes only, so odd leading
// dimensions and 8-byte aligned operands will do.  ODD is for those and for odd
// sizes: the pair that straddles the end of an odd row range or of an odd K is left
// out of the DMA (the hardware writes zeros) and its one element goes through a
// register of the same lane, before the step's barrier; no load leaves the operand,
// and only the workgroups at the edge or in the last step do this.  Scalar offsets
// run over whole K steps, past K in the last one, and stay below 2 GiB (f64_fit):
// a masked lane's vector offset is then past num_records whichever way the
// hardware counts the scalar one.
//
// A DMA load writes 1 KB of LDS in lane order, so every swizzle is in which
// element a lane loads:
//   rows contiguous in memory: S[k][R] (R = 128: one k a load; 64: two), the row
//     XORed by 16 for k with bit 1 set;
//   k contiguous: S[row][16] as eight 16-byte chunks, chunk XORed by row % 8
//     (eight rows a load).
// An MFMA takes four k, one per lane quarter lq; quarter lq of slice s (8 deep)
// owns k = 8 s + 2 lq and the next, which a 16-byte read of a k-contiguous
// operand returns together and which lie in rows 2 lq, 2 lq + 1 of the other
// kind.  Both read patterns hit every bank once per pass.
//
// Two stages.  The loads of step s + 1 go out at the start of step s, its barrier
// sits before the last quarter of the MFMAs, which cover the latency of the
// next step's first fragment reads; two workgroups a CU fill the rest.
// Against the kernel that stages through registers (same tiles; MFMA busy 0.86
// there at 4096 x 4096 x 8192): 4094 -> 3924 us at that shape, 1024 x 8192 x 1024
// with 64 x 64 tiles 289 -> 261, 1024 x 5120 x 2048 with A transposed 562 -> 507.
// ODD (us, through registers before): 777 x 4000 x 3885 492 -> 437, with A transposed
// 496 -> 419; 1023 x 8184 x 1023 292 -> 276; 2047 x 2047 x 4095 592 -> 557.
// ---------------------------------------------------------------------------
constexpr unsigned OOB = 0x80000000u;   // past every num_records: the hardware returns zeros
typedef __attribute__((address_space(3))) void lds_void;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t raw_rsrc(const void* p) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, 0x7fffffff, 0x00020000);
}

template <int BM, int BN, bool TA, bool TB, bool ODD, class Src>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(2)))
void gemm_f64_dma_kernel(Src src) {
  constexpr int BK = (int)F64_BK;
  constexpr int WM = BM / 2, WN = BN / 2;
  constexpr int FM = WM / 16, FN = WN / 16;
  constexpr int CHA = BM * BK * 8 / 1024 / 4, CHB = BN * BK * 8 / 1024 / 4;   // DMA loads a wave
  constexpr bool AK = TA, BKD = !TB;

  __shared__ __attribute__((aligned(1024))) double As0[BM * BK];
  __shared__ __attribute__((aligned(1024))) double As1[BM * BK];
  __shared__ __attribute__((aligned(1024))) double Bs0[BN * BK];
  __shared__ __attribute__((aligned(1024))) double Bs1[BN * BK];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm0 = (wave & 1) * WM;
  const int wn0 = (wave >> 1) * WN;
  const int li = lane & 15;
  const int lq = lane >> 4;

  for (int un = src_first(src); un < src_units(src); un += src_stride(src)) {
  int t, slice, nslice;
  src_unit(src, un, t, slice, nslice);
  const GemmProb& P = src_prob(src, t);
  int tm, tn;
  tile_coords(P, t - P.tile_start, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int M = P.M, N = P.N;

  dx4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = dx4{0.0, 0.0, 0.0, 0.0};

  int nsteps = 0;
  for (int s = 0; s < P.nseg; ++s) nsteps += (P.seg[s].K + BK - 1) / BK;

  // Load c of this wave (c < CH): byte offset v[c] of the lane (OOB where its row
  // is outside the operand) plus the uniform (c cs + k0 ks)
  __amdgpu_buffer_rsrc_t rA, rB;
  unsigned vA[AK ? CHA : 1], vB[BKD ? CHB : 1];
  unsigned csA = 0, csB = 0, ksA = 0, ksB = 0, w0A = 0, w0B = 0;
  int K = 0;
  // ODD: element offset of the pair cut by the end of an odd row range, the elements
  // themselves, and whether this step has any on either side
  unsigned eA = OOB, eB = OOB;
  double xA[CHA], xB[CHB];
  bool fixA = false, fixB = false;
  auto set_side = [&](bool kdir, int R, int CH, const char* p, int64_t ld, int r0, int lim, __amdgpu_buffer_rsrc_t& rs,
                      unsigned* v, unsigned& cs, unsigned& ks, unsigned& w0, unsigned& e) {
    if (kdir) {
      rs = raw_rsrc(p + (int64_t)r0 * ld * 8);
      ks = 8u;
      cs = (unsigned)(32 * ld * 8);          // loads wave + 4 c: 8 rows each
      w0 = (unsigned)(8 * wave * ld * 8);
      const unsigned o = (unsigned)((lane >> 3) * ld * 8 + (((lane & 7) ^ (lane >> 3)) << 4));
#pragma unroll
      for (int c = 0; c < CH; ++c) v[c] = r0 + 8 * (wave + 4 * c) + (lane >> 3) < lim ? o : OOB;
    } else {
      rs = raw_rsrc(p + (int64_t)r0 * 8);
      ks = (unsigned)(ld * 8);
      const int kpl = 128 / R;               // k rows a load
      cs = (unsigned)(4 * kpl * ld * 8);
      w0 = (unsigned)(kpl * wave * ld * 8);
      const int pairs = R / 2, kl = lane / pairs;
      const int kw = kpl * wave;             // (k >> 1) & 1 is that of the wave's first load
      const int row = (2 * (lane % pairs)) ^ (16 * ((kw >> 1) & 1));
      v[0] = r0 + row < lim ? (unsigned)(row * 8 + kl * ld * 8) : OOB;
      if (ODD) {
        e = r0 + row == lim - 1 ? v[0] : OOB;
        v[0] = r0 + row == lim - 1 ? OOB : v[0];
      }
    }
  };
  auto set_seg = [&](int s) {
    const GemmSeg& S = P.seg[s];
    set_side(AK, BM, CHA, static_cast<const char*>(resolve(src, S.A)), S.lda, m0, M, rA, vA, csA, ksA, w0A, eA);
    set_side(BKD, BN, CHB, static_cast<const char*>(resolve(src, S.B)), S.ldb, n0, N, rB, vB, csB, ksB, w0B, eB);
    K = S.K;
  };
  auto fetch_side = [&](bool kdir, int R, int CH, __amdgpu_buffer_rsrc_t rs, const unsigned* v, unsigned cs, unsigned ks,
                        unsigned w0, int k0, double* S, int r0, int lim, unsigned e, double* x, bool& fix) {
    const bool tail = k0 + BK > K;
    if (ODD) fix = kdir ? tail && (K & 1) : r0 + R > lim && (lim & 1);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      unsigned o = v[kdir ? c : 0], oe = ODD ? kdir ? o : e : OOB;
      const unsigned so = w0 + c * cs + (unsigned)k0 * ks;
      if (tail) {
        // with an even K, so are the k of a chunk or of a load's first row
        const int k = kdir ? 2 * ((lane & 7) ^ (lane >> 3)) : (128 / R) * (wave + 4 * c) + (ODD ? lane / (R / 2) : 0);
        if (ODD) oe = (kdir ? k0 + k == K - 1 : k0 + k < K) ? oe : OOB;
        o = k0 + k + (ODD && kdir ? 1 : 0) < K ? o : OOB;
      }
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void*)(S + (wave + 4 * c) * 128), 16, (int)o, (int)so, 0, 0);
      if (ODD && fix) x[c] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rs, (int)oe, (int)so, 0));
    }
  };
  // ODD: the elements into the places that their own lane's DMA loads left zero
  auto mend_side = [&](bool kdir, int CH, double* S, unsigned e, const double* x, int k0) {
    const bool mine = kdir ? k0 + 2 * ((lane & 7) ^ (lane >> 3)) == K - 1 : e != OOB;
    if (mine) {
#pragma unroll
      for (int c = 0; c < CH; ++c) S[(wave + 4 * c) * 128 + 2 * lane] = x[c];
    }
  };

  // fragments of slice s (8 deep): items m = 0, 1
  auto read_side = [&](bool kdir, int R, int F, const double* S, int w0, int s, double (*f)[2]) {
    if (kdir) {
      const double* p = S + (w0 + li) * BK + (((4 * s + lq) ^ (li & 7)) << 1);
#pragma unroll
      for (int i = 0; i < F; ++i) {
        const dx2 v = *reinterpret_cast<const dx2*>(p + i * 16 * BK);
        f[i][0] = v.x;
        f[i][1] = v.y;
      }
    } else {
      // rows XORed by 16 in the odd quarters: blocks i and i ^ 1 change places
      const int x = lq & 1;
      const double* pe = S + (8 * s + 2 * lq) * R + w0 + li + 16 * x;
      const double* po = S + (8 * s + 2 * lq) * R + w0 + li + 16 - 16 * x;
#pragma unroll
      for (int i = 0; i < F; ++i)
#pragma unroll
        for (int m = 0; m < 2; ++m) f[i][m] = (i & 1 ? po : pe)[m * R + (i >> 1) * 32];
    }
  };
  double fa[2][FM][2], fb[2][FN][2];

  int s, k0, step0, step1;
  slice_range<BK>(P, nsteps, slice, nslice, step0, step1, s, k0);
  auto fetch = [&](double* A, double* B) {
    fetch_side(AK, BM, CHA, rA, vA, csA, ksA, w0A, k0, A, m0, M, eA, xA, fixA);
    fetch_side(BKD, BN, CHB, rB, vB, csB, ksB, w0B, k0, B, n0, N, eB, xB, fixB);
  };
  auto mend = [&](double* A, double* B) {
    if (!ODD || !(fixA | fixB)) return;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (fixA) mend_side(AK, CHA, A, eA, xA, k0);
    if (fixB) mend_side(BKD, CHB, B, eB, xB, k0);
  };
  auto mfma = [&](int f, int m) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fb[f][j][m], fa[f][i][m], acc[i][j], 0, 0, 0);
  };
  auto body = [&](const double* A, const double* B, double* An, double* Bn, bool has_next) {
    if (has_next) {
      k0 += BK;
      while (k0 >= K && s + 1 < P.nseg) {
        ++s;
        k0 = 0;
        set_seg(s);
      }
      fetch(An, Bn);
    }
    read_side(AK, BM, FM, A, wm0, 1, fa[1]);
    read_side(BKD, BN, FN, B, wn0, 1, fb[1]);
    mfma(0, 0);
    mfma(0, 1);
    mfma(1, 0);
    __builtin_amdgcn_sched_barrier(0);
    if (has_next) mend(An, Bn);
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    if (has_next) {
      read_side(AK, BM, FM, An, wm0, 0, fa[0]);
      read_side(BKD, BN, FN, Bn, wn0, 0, fb[0]);
    }
    mfma(1, 1);
  };
  if (step1 > step0) {
    set_seg(s);
    fetch(As0, Bs0);
    mend(As0, Bs0);
    __syncthreads();
    read_side(AK, BM, FM, As0, wm0, 0, fa[0]);
    read_side(BKD, BN, FN, Bs0, wn0, 0, fb[0]);
  }
  for (int step = step0; step < step1; step += 2) {
    body(As0, Bs0, As1, Bs1, step + 1 < step1);
    if (step + 1 < step1) body(As1, Bs1, As0, Bs0, step + 2 < step1);
  }

  // epilogue: as in gemm_f64_kernel
  if (slice < 0)
    epilogue_c<false, FM, FN, dx4, 1>(acc, resolve(src, P.C), P.ldc, M, N, m0 + wm0, n0 + wn0, li, lq, P.alpha, P.beta);
  else
    store_partial(acc, src_partial<double>(src, t, slice, BM * BN), wave, lane);
  }  // units
}

// ---------------------------------------------------------------------------
// Small launches.  With a handful of 64 x 64 tiles the K loop is one serial chain
// of load latencies.  Here a workgroup takes a 32 x 32 tile and its eight waves an
// eighth of K each, straight from memory to the MFMA operands (no LDS stage, no
// barrier until the sums are added), two groups of four slices of four k in flight.
// Loads are single elements from clamped addresses, zeroed outside the operand,
// so any size, stride and alignment will do.  The epilogue may add the physical
// term (GemmPhys), which saves a launch.
// ---------------------------------------------------------------------------
constexpr int ST = 32, SW = 8, SG = 4;   // tile, waves, slices loaded together

template <bool TA, bool TB>
__global__ __launch_bounds__(64 * SW) void gemm_f64_small_kernel(GemmBatch src) {
  __shared__ double red[SW][ST * (ST + 1)];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, lk = lane >> 4;
  const int t = blockIdx.x;
  const GemmProb& P = src_prob(src, t);
  const int u = t - P.tile_start;
  const int m0 = (u % P.tiles_m) * ST, n0 = (u / P.tiles_m) * ST;
  const int M = P.M, N = P.N;
  dx4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = dx4{0.0, 0.0, 0.0, 0.0};

  int total = 0;
  for (int s = 0; s < P.nseg; ++s) total += (P.seg[s].K + 3) / 4;
  int g0 = (int)((int64_t)wave * total / SW);
  const int g1 = (int)((int64_t)(wave + 1) * total / SW);
  typedef const __attribute__((address_space(1))) double gd;
  int first = 0;   // slice the segment starts at
  for (int s = 0; s < P.nseg && g0 < g1; ++s) {
    const GemmSeg& S = P.seg[s];
    const int K = S.K, ns = (K + 3) / 4;
    const int e = min(g1, first + ns) - first;
    const int64_t sak = TA ? 1 : S.lda, sbk = TB ? S.ldb : 1;
    gd *pa[2], *pb[2];
    bool oka[2], okb[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = m0 + 16 * i + li, c = n0 + 16 * i + li;
      oka[i] = r < M;
      okb[i] = c < N;
      pa[i] = (gd*)static_cast<const double*>(S.A) + (int64_t)min(r, M - 1) * (TA ? S.lda : 1);
      pb[i] = (gd*)static_cast<const double*>(S.B) + (int64_t)min(c, N - 1) * (TB ? 1 : S.ldb);
    }
    auto load = [&](int g, double (&a)[SG][2], double (&b)[SG][2]) {
#pragma unroll
      for (int q = 0; q < SG; ++q) {
        const int k = 4 * (g + q) + lk, kc = min(k, K - 1);
        const bool ok = g + q < e && k < K;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const double av = pa[i][kc * sak], bv = pb[i][kc * sbk];
          a[q][i] = ok && oka[i] ? av : 0.0;
          b[q][i] = ok && okb[i] ? bv : 0.0;
        }
      }
    };
    int g = g0 - first;
    if (g < e) {
      double a[2][SG][2], b[2][SG][2];
      load(g, a[0], b[0]);
      for (int it = 0; g < e; ++it) {
        auto step = [&](double (&ac)[SG][2], double (&bc)[SG][2], double (&an)[SG][2], double (&bn)[SG][2]) {
          if (g + SG < e) load(g + SG, an, bn);
#pragma unroll
          for (int q = 0; q < SG; ++q)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
              for (int j = 0; j < 2; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bc[q][j], ac[q][i], acc[i][j], 0, 0, 0);
          g += SG;
        };
        step(a[0], b[0], a[1], b[1]);
        if (g < e) step(a[1], b[1], a[0], b[0]);
      }
      g0 = first + e;
    }
    first += ns;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[wave][(16 * j + lk + 4 * r) * (ST + 1) + 16 * i + li] = acc[i][j][r];
  __syncthreads();
  gptr_t<double> C = gptr(P.C);
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int r = threadIdx.x % ST, c = threadIdx.x / ST + 16 * q;
    const int row = m0 + r, col = n0 + c;
    if (row >= M || col >= N) continue;
    double v = 0.0;
#pragma unroll
    for (int w = 0; w < SW; ++w) v += red[w][c * (ST + 1) + r];
    if (P.phys.P) {
      gd* x = (gd*)P.phys.x + row + (int64_t)col * P.phys.ldx;
      gd* pp = (gd*)P.phys.P + P.phys.b + P.phys.d1 * P.phys.e;
      double pv = 0.0;
      for (int j = 0; j < P.phys.d2; ++j)
        for (int h = 0; h < P.phys.d1; ++h)
          pv += pp[P.phys.d1 * P.phys.d2 * (h + P.phys.d1 * j)] * x[P.phys.sh * h + P.phys.sj * j];
      v += pv;
    }
    v *= P.alpha;
    const int64_t o = row + (int64_t)col * P.ldc;
    if (P.beta != 0.0) v += P.beta * C[o];
    C[o] = v;
  }
}

// Load path of the FP64 kernels, read once from MK_F64_VARIANT ("dma" or "branch";
// default "dma"): lets benchmarks and tests pin one of them.
bool f64_direct() {
  static const bool v = [] {
    const char* e = getenv("MK_F64_VARIANT");
    return !(e && !strcmp(e, "branch"));
  }();
  return v;
}

template <int BM, int BN, bool ODD, class Src>
void launch4_dma(GemmShape sh, dim3 grid, dim3 block, hipStream_t stream, const Src& b) {
  if (!sh.ta && !sh.tb) hipLaunchKernelGGL((gemm_f64_dma_kernel<BM, BN, false, false, ODD, Src>), grid, block, 0, stream, b);
  else if (sh.ta && !sh.tb) hipLaunchKernelGGL((gemm_f64_dma_kernel<BM, BN, true, false, ODD, Src>), grid, block, 0, stream, b);
  else if (!sh.ta && sh.tb) hipLaunchKernelGGL((gemm_f64_dma_kernel<BM, BN, false, true, ODD, Src>), grid, block, 0, stream, b);
  else hipLaunchKernelGGL((gemm_f64_dma_kernel<BM, BN, true, true, ODD, Src>), grid, block, 0, stream, b);
}

template <int BM, int BN, class Src>
void launch4(GemmShape sh, dim3 grid, dim3 block, hipStream_t stream, const Src& b) {
  if (!sh.ta && !sh.tb) hipLaunchKernelGGL((gemm_f64_kernel<BM, BN, false, false, Src>), grid, block, 0, stream, b);
  else if (sh.ta && !sh.tb) hipLaunchKernelGGL((gemm_f64_kernel<BM, BN, true, false, Src>), grid, block, 0, stream, b);
  else if (!sh.ta && sh.tb) hipLaunchKernelGGL((gemm_f64_kernel<BM, BN, false, true, Src>), grid, block, 0, stream, b);
  else hipLaunchKernelGGL((gemm_f64_kernel<BM, BN, true, true, Src>), grid, block, 0, stream, b);
}

template <int BM, int BN, class Src>
void launch_path(int fit, GemmShape sh, dim3 grid, dim3 block, hipStream_t stream, const Src& b) {
  if (f64_direct() && fit == BUF_EVEN) launch4_dma<BM, BN, false, Src>(sh, grid, block, stream, b);
  else if (f64_direct() && fit == BUF_ODD) launch4_dma<BM, BN, true, Src>(sh, grid, block, stream, b);
  else launch4<BM, BN, Src>(sh, grid, block, stream, b);
}

// One output-tile grid of `BM` x `BN` tiles over the problems.
template <int BM, int BN>
int fill_batch(const ProbSpec* probs, int nprob, GemmBatch& b) {
  int total = 0;
  for (int i = 0; i < nprob; ++i) {
    const ProbSpec& ps = probs[i];
    GemmProb& P = b.p[i];
    P.M = (int32_t)ps.M;
    P.N = (int32_t)ps.N;
    P.nseg = 0;
    for (int s = 0; s < ps.nseg; ++s) {
      if (ps.seg[s].K <= 0) continue;
      GemmSeg& g = P.seg[P.nseg++];
      g.A = ps.seg[s].A;
      g.B = ps.seg[s].B;
      g.Alo = g.Blo = nullptr;
      g.lda = ps.seg[s].lda;
      g.ldb = ps.seg[s].ldb;
      g.K = (int32_t)ps.seg[s].K;
      const bool al = ((uintptr_t)g.A % 16 == 0) && ((uintptr_t)g.B % 16 == 0) &&
                      (g.lda % 2 == 0) && (g.ldb % 2 == 0);
      g.vec = al ? 1 : 0;
    }
    P.tiles_m = (int32_t)cdiv(ps.M, BM);
    P.tiles_n = (int32_t)cdiv(ps.N, BN);
    P.tile_start = total;
    total += P.tiles_m * P.tiles_n;
    P.C = ps.C;
    P.ldc = ps.ldc;
    P.alpha = ps.alpha;
    P.beta = ps.beta;
    P.phys = ps.phys;
  }
  b.nprob = nprob;
  b.total_tiles = total;
  return total;
}

mk_status launch_small(const ProbSpec* probs, int nprob, GemmShape sh, hipStream_t stream) {
  GemmBatch b{};
  const int total = fill_batch<ST, ST>(probs, nprob, b);
  if (total == 0) return MK_OK;
  b.full_tiles = total;
  b.ksplit = 1;
  ProfScope prof("gemm_f64", stream);
  const dim3 grid(total), block(64 * SW);
  if (!sh.ta && !sh.tb) hipLaunchKernelGGL((gemm_f64_small_kernel<false, false>), grid, block, 0, stream, b);
  else if (sh.ta && !sh.tb) hipLaunchKernelGGL((gemm_f64_small_kernel<true, false>), grid, block, 0, stream, b);
  else if (!sh.ta && sh.tb) hipLaunchKernelGGL((gemm_f64_small_kernel<false, true>), grid, block, 0, stream, b);
  else hipLaunchKernelGGL((gemm_f64_small_kernel<true, true>), grid, block, 0, stream, b);
  MK_CHECK_HIP(hipGetLastError());
  return MK_OK;
}

template <int BM, int BN>
mk_status launch_cfg(const ProbSpec* probs, int nprob, GemmShape sh, hipStream_t stream, SplitPlan sp, void* ws) {
  GemmBatch b{};
  const int total = fill_batch<BM, BN>(probs, nprob, b);
  if (total == 0) return MK_OK;
  b.full_tiles = sp.ksplit > 1 ? sp.full : total;
  b.ksplit = sp.ksplit;
  b.ws = ws;
  const int tail = total - b.full_tiles;
  MK_REQUIRE(tail == 0 || (ws != nullptr && (size_t)tail * sp.ksplit * BM * BN * 8 <= GEMM_WS_BYTES), MK_BAD_ARG,
             "gemm_f64: %d tiles split %d ways exceed the workspace", tail, sp.ksplit);
  int fit = BUF_EVEN;
  for (int i = 0; i < nprob && fit != BUF_NO; ++i) fit = std::min<int>(fit, f64_fit(probs[i], sh, BM, BN));
  dim3 grid(b.full_tiles + tail * b.ksplit), block(NT);
  ProfScope prof("gemm_f64", stream);
  launch_path<BM, BN>(fit, sh, grid, block, stream, b);
  MK_CHECK_HIP(hipGetLastError());
  if (tail > 0) {
    constexpr int NBLK = BM * BN / 256;
    hipLaunchKernelGGL((splitk_reduce_kernel<false, 2, BM / 32, BN / 32, 2, dx4>), dim3((unsigned)cdiv((int64_t)tail * NBLK, 4)),
                       dim3(256), 0, stream, b);
    MK_CHECK_HIP(hipGetLastError());
  }
  return MK_OK;
}

template <int BM, int BN>
mk_status launch_group(const GemmGroup& g, GemmShape sh, int grid, hipStream_t stream) {
  if (g.total_tiles == 0) return MK_OK;
  dim3 gr(grid), block(NT);
  ProfScope prof("gemm_f64", stream);
  launch_path<BM, BN>(g.f64_buf, sh, gr, block, stream, g);
  MK_CHECK_HIP(hipGetLastError());
  return MK_OK;
}

// Workgroups of the grouped kernel for `fit` (launch_path) that a CU holds, taken of
// one storage order.
template <int BM, int BN>
int occupancy(int fit) {
  auto of = [](auto kern) {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kern, NT, 0) != hipSuccess) n = 1;
    return n > 0 ? n : 1;
  };
  static const int occ[3] = {of(gemm_f64_kernel<BM, BN, false, false, GemmGroup>),
                             of(gemm_f64_dma_kernel<BM, BN, false, false, true, GemmGroup>),
                             of(gemm_f64_dma_kernel<BM, BN, false, false, false, GemmGroup>)};
  return occ[f64_direct() ? fit : BUF_NO];
}

}  // namespace

int f64_group_grid(int kind, int fit, int total_tiles, int cus) {
  const int occ = kind == TK_128 ? occupancy<128, 128>(fit) : occupancy<64, 64>(fit);
  return (int)std::min<int64_t>(total_tiles, (int64_t)occ * cus);
}

int f64_buf_ok(const ProbSpec* probs, int n, GemmShape sh, int kind) {
  int fit = BUF_EVEN;
  for (int i = 0; i < n && fit != BUF_NO; ++i)
    fit = std::min<int>(fit, f64_fit(probs[i], sh, tile_m(kind), tile_n(kind)));
  return fit;
}

mk_status gemm_f64_group(const GemmGroup& g, int kind, GemmShape sh, int grid, hipStream_t st) {
  if (kind == TK_128) return launch_group<128, 128>(g, sh, grid, st);
  MK_REQUIRE(kind == TK_64, MK_BAD_ARG, "gemm_f64_group: tile kind %d", kind);
  return launch_group<64, 64>(g, sh, grid, st);
}

namespace {

struct F64Plan {
  bool small = false;
  TileChoice c128, c64;
};

F64Plan plan_f64(const ProbSpec* probs, int nprob, GemmShape shape, bool ws) {
  // One step is 64 (128 tile) or 16 v_mfma_f64_16x16x4 of 64 cycles a wave.
  // Straight to LDS, measured (us): 1024 x 1024 x 2048 with 64 x 64 tiles, 1 and 3
  // workgroups a CU 83 and 83 (split 3 ways, reduction included), 1024 x 8192 x
  // 1024 8 rounds of 64 tiles 261, 2 of 128 tiles 255; 1024 x 5120 x 2048 with A
  // transposed 374 (64 tiles) and 331 (256 tiles of 128, 64 split 8 ways).  Odd
  // sizes: 1023 x 1023 x 8191, 64 tiles 1, 2, 3, 4 a CU 431, 337, 306, 295, 128 tiles
  // 1, 2 a CU 312, 291; 2047 x 2047 x 4095, 64 tiles 562, 128 tiles 600 (split 561).
  static const TileModel d128{128, 128, 16, 1.74, {0.88, 0.90, 0.90, 0.90}, 2, 128 * 128 * 8};
  static const TileModel d64{64, 64, 16, 0.436, {0.70, 0.83, 0.87, 0.88}, 4, 64 * 64 * 8};
  static const TileModel d64t{64, 64, 16, 0.436, {0.62, 0.73, 0.77, 0.78}, 4, 64 * 64 * 8};
  static const TileModel b128{128, 128, 16, 1.74, {0.74, 0.82, 0.82, 0.82}, 2, 128 * 128 * 8};
  static const TileModel b64{64, 64, 16, 0.436, {0.52, 0.68, 0.75, 0.79}, 4, 64 * 64 * 8};
  const bool direct = f64_direct() && f64_buf_ok(probs, nprob, shape, TK_128) == BUF_EVEN;
  const TileModel& m64 = !direct ? b64 : shape.ta || shape.tb ? d64t : d64;
  F64Plan pl;
  pl.c128 = plan_launch(direct ? d128 : b128, probs, nprob, ws);
  pl.c64 = plan_launch(m64, probs, nprob, ws);
  // The small kernel, on at most one 32 x 32 tile per CU.  Where it saves the launch
  // of a physical term, up to 12 slices a wave (K = 384): measured with launches (us,
  // the tile kernels beside it, which split) 128 x 128 x 256 10.8 and 14.3, 192 x 192
  // x 384 12.4 and 13.6, past the line 256 x 256 x 512 15.2 and 13.6.  Without one it
  // gains at odd sizes, whose tile kernel is the slower (up to 8 slices a wave: one-
  // site apply w = 5 D = 33 9.4 and 12.6, bond apply D = 33 15.4 and 19.2); elsewhere
  // the two are even up to 4 and it falls behind after (transfer w = 5 D = 150 36 and
  // 33, bond apply D = 64 20 and 17), so 4 is the line.
  int64_t tiles = 0, slices = 0;
  bool phys = false;
  for (int i = 0; i < nprob; ++i) {
    int64_t n = 0;
    for (int s = 0; s < probs[i].nseg; ++s) n += cdiv(std::max<int64_t>(probs[i].seg[s].K, 0), 4);
    const int64_t t = cdiv(probs[i].M, ST) * cdiv(probs[i].N, ST);
    tiles += t;
    if (t > 0) slices = std::max(slices, n);
    phys = phys || probs[i].phys.P != nullptr;
  }
  const bool split = (pl.c128.us <= pl.c64.us ? pl.c128 : pl.c64).split.ksplit > 1;
  pl.small = f64_direct() && tiles <= PLAN_CUS &&
             slices <= (phys ? 96 : direct ? 32 : 64) && (split || phys);
  return pl;
}

}  // namespace

bool gemm_f64_small(const ProbSpec* probs, int nprob, GemmShape shape, bool ws) {
  return plan_f64(probs, nprob, shape, ws).small;
}

mk_status gemm_f64(const ProbSpec* probs, int nprob, GemmShape shape, hipStream_t stream, void* ws) {
  MK_REQUIRE(nprob >= 0 && nprob <= MAX_PROB, MK_BAD_ARG, "gemm_f64: %d problems (max %d)", nprob, MAX_PROB);
  for (int i = 0; i < nprob; ++i) {
    MK_REQUIRE(!probs[i].full, MK_BAD_ARG, "gemm_f64: more than %d segments", MAX_SEG);
    MK_REQUIRE(probs[i].M >= 0 && probs[i].N >= 0 && probs[i].M < (1ll << 31) && probs[i].N < (1ll << 31),
               MK_BAD_SHAPE, "gemm_f64: bad M/N");
    for (int s = 0; s < probs[i].nseg; ++s)
      MK_REQUIRE(probs[i].seg[s].K >= 0 && probs[i].seg[s].K < (1ll << 31), MK_BAD_SHAPE, "gemm_f64: bad K");
  }
  const F64Plan pl = plan_f64(probs, nprob, shape, ws != nullptr);
  if (pl.small) return launch_small(probs, nprob, shape, stream);
  for (int i = 0; i < nprob; ++i)
    MK_REQUIRE(probs[i].phys.P == nullptr, MK_BAD_ARG, "gemm_f64: a physical term in a launch that is not small");
  const TileChoice &c128 = pl.c128, &c64 = pl.c64;
  if (c128.us <= c64.us) return launch_cfg<128, 128>(probs, nprob, shape, stream, c128.split, ws);
  return launch_cfg<64, 64>(probs, nprob, shape, stream, c64.split, ws);
}

}  // namespace mk
