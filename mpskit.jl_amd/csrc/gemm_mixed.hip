// Mixed-precision MFMA GEMMs for CDNA4 (gfx950) with float64 output.
//
//  BF16X3: each float64 operand is pre-split into bf16 hi + lo; the kernel
//          issues hi*hi + hi*lo + lo*hi on v_mfma_f32_16x16x32_bf16 and
//          accumulates in fp32 (relative error ~2^-16 per product).
//  F32   : operands pre-rounded to fp32, v_mfma_f32_16x16x4_f32.
//
// Operands are K-contiguous: A(i,k) = A[i*lda + k], B(k,j) = B[j*ldb + k], with
// 16-byte aligned rows whose length lda/ldb is padded (with zeros) to a
// multiple of 8 elements.  One LDS row per tile row holds 64 bytes of K
// (32 bf16 or 16 fp32); lane (row r = lane%16, group g = lane/16) reads the 16
// bytes at offset 16*g, which is the bf16 MFMA k-slot layout and, for fp32,
// the k-permutation "group g owns k = 4g..4g+3 across the 4 sub-steps" shared
// by A and B.
#include <hip/hip_bf16.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>

#include "gemm_dev.h"
#include "gemm_plan.h"
#include "prof.h"

namespace mk {
namespace {

typedef float fx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bfx8 __attribute__((ext_vector_type(8)));
typedef unsigned int ux4 __attribute__((ext_vector_type(4)));

constexpr int NT = 256;
constexpr int ROWB = 64;          // bytes of K per LDS row per step

// Place of 16-byte chunk q of tile row r in an LDS slab of 64-byte rows.  A
// 64-lane ds_read_b128 goes through the 256 B / cycle LDS in four groups of 16
// lanes, {0-3, 12-15, 20-27} and its like, so a fragment read (row lane % 16,
// chunk lane / 16) mixes rows of two chunks: with the chunks of rows 4 t .. 4 t + 3
// XORed by -t (mod 4) the 16 lanes of every group hit distinct banks.  (XORed by
// t, or in rows padded to 80 bytes, every read took two passes.)  The stores of
// 16 consecutive lanes fill 256 contiguous bytes in any order.
__device__ __forceinline__ int swz(int r, int q) { return r * ROWB + ((q ^ (-(r >> 2) & 3)) << 4); }

enum Mode { M_BF16X3 = 0, M_F32 = 1 };

// Load path of the kernels, read once from MK_GEMM_VARIANT ("dma" or "tile";
// default "dma"): lets benchmarks and tests pin the register-staged kernel.
enum Variant { V_TILE = 0, V_DMA = 1 };
int variant() {
  static const int v = [] {
    const char* e = getenv("MK_GEMM_VARIANT");
    return e && !strcmp(e, "tile") ? (int)V_TILE : (int)V_DMA;
  }();
  return v;
}

// Epilogue of an FM x FN grid of 16x16 fp32 accumulator blocks.  The MFMAs run
// with the B fragment as first operand, so block (i, j) is C^T and item r of
// lane (li, lg) is C[row0 + 16 i + li][col0 + 16 j + 4 lg + r]: the 16 lanes of
// a quarter-wave store 16 consecutive rows (128 B) of one column.
template <int FM, int FN>
__device__ __forceinline__ void store_tile(const fx4 (&acc)[FM][FN], double* __restrict__ C, int64_t ldc, int M,
                                           int N, int row0, int col0, int li, int lg, double alpha, double beta) {
  epilogue_c<true>(acc, C, ldc, M, N, row0, col0, li, lg, alpha, beta);
}

// Load a (R rows x 64 B) slab of a K-contiguous operand into registers.
// elem_bytes = 2 (bf16) or 4 (fp32); Klim = padded row length in elements.
template <int R>
__device__ __forceinline__ void load_slab(const char* __restrict__ base, int64_t ld_bytes, int r0,
                                          int64_t kbyte0, int Rlim, int64_t Kbytes,
                                          ux4 (&reg)[R * ROWB / 16 / NT]) {
  constexpr int CH = R * ROWB / 16 / NT;
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int id = threadIdx.x + c * NT;
    const int r = id / (ROWB / 16);
    const int q = id % (ROWB / 16);
    const int gr = r0 + r;
    const int64_t kb = kbyte0 + q * 16;
    ux4 v = {0u, 0u, 0u, 0u};
    if (gr < Rlim && kb < Kbytes) v = *gptr(reinterpret_cast<const ux4*>(base + (int64_t)gr * ld_bytes + kb));
    reg[c] = v;
  }
}

template <int R>
__device__ __forceinline__ void store_slab(char* S, const ux4 (&reg)[R * ROWB / 16 / NT]) {
  constexpr int CH = R * ROWB / 16 / NT;
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int id = threadIdx.x + c * NT;
    const int r = id / (ROWB / 16);
    const int q = id % (ROWB / 16);
    *reinterpret_cast<ux4*>(S + swz(r, q)) = reg[c];
  }
}

template <int BM, int BN, int MODE, class Src>
__global__ __launch_bounds__(NT) void gemm_mixed_kernel(Src src) {
  constexpr int NPART = MODE == M_BF16X3 ? 2 : 1;   // hi/lo arrays per operand
  constexpr int EB = MODE == M_BF16X3 ? 2 : 4;      // element bytes
  constexpr int WM = BM / 2, WN = BN / 2;
  constexpr int FM = WM / 16, FN = WN / 16;
  constexpr int CHA = BM * ROWB / 16 / NT;
  constexpr int CHB = BN * ROWB / 16 / NT;

  __shared__ __attribute__((aligned(16))) char As[2][NPART][BM * ROWB];
  __shared__ __attribute__((aligned(16))) char Bs[2][NPART][BN * ROWB];

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
  const int li = lane & 15;
  const int lg = lane >> 4;

  fx4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = fx4{0.f, 0.f, 0.f, 0.f};

  constexpr int KSTEP = ROWB / EB;  // elements of K per step
  int nsteps = 0;
  for (int s = 0; s < P.nseg; ++s) nsteps += (P.seg[s].K + KSTEP - 1) / KSTEP;

  ux4 ra[NPART][CHA], rb[NPART][CHB];
  auto load = [&](int s, int k0) {
    const GemmSeg& S = P.seg[s];
    const int64_t ldab = S.lda * EB, ldbb = S.ldb * EB;
    const int64_t kb0 = (int64_t)k0 * EB, Kb = (int64_t)S.K * EB;
    load_slab<BM>(static_cast<const char*>(resolve(src, S.A)), ldab, m0, kb0, P.M, Kb, ra[0]);
    load_slab<BN>(static_cast<const char*>(resolve(src, S.B)), ldbb, n0, kb0, P.N, Kb, rb[0]);
    if (NPART == 2) {
      load_slab<BM>(static_cast<const char*>(resolve(src, S.Alo)), ldab, m0, kb0, P.M, Kb, ra[NPART - 1]);
      load_slab<BN>(static_cast<const char*>(resolve(src, S.Blo)), ldbb, n0, kb0, P.N, Kb, rb[NPART - 1]);
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int p = 0; p < NPART; ++p) {
      store_slab<BM>(As[buf][p], ra[p]);
      store_slab<BN>(Bs[buf][p], rb[p]);
    }
  };

  int s, k0, step0, step1;
  slice_range<KSTEP>(P, nsteps, slice, nslice, step0, step1, s, k0);
  if (step1 > step0) {
    load(s, k0);
    store(0);
  }
  __syncthreads();
  int buf = 0;
  for (int step = step0; step < step1; ++step) {
    int ns = s, nk0 = k0 + KSTEP;
    if (nk0 >= P.seg[s].K) { ns = s + 1; nk0 = 0; }
    const bool has_next = step + 1 < step1;
    if (has_next) load(ns, nk0);

    ux4 fa[NPART][FM], fb[NPART][FN];
#pragma unroll
    for (int p = 0; p < NPART; ++p) {
#pragma unroll
      for (int i = 0; i < FM; ++i)
        fa[p][i] = *reinterpret_cast<const ux4*>(As[buf][p] + swz(wm0 + li, lg) + i * 16 * ROWB);
#pragma unroll
      for (int j = 0; j < FN; ++j)
        fb[p][j] = *reinterpret_cast<const ux4*>(Bs[buf][p] + swz(wn0 + li, lg) + j * 16 * ROWB);
    }
    if constexpr (MODE == M_BF16X3) {
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          const bfx8 ah = __builtin_bit_cast(bfx8, fa[0][i]);
          const bfx8 al = __builtin_bit_cast(bfx8, fa[1][i]);
          const bfx8 bh = __builtin_bit_cast(bfx8, fb[0][j]);
          const bfx8 bl = __builtin_bit_cast(bfx8, fb[1][j]);
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bh, al, acc[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bl, ah, acc[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bh, ah, acc[i][j], 0, 0, 0);
        }
    } else {
#pragma unroll
      for (int sub = 0; sub < 4; ++sub)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j) {
            // extract the element to a scalar first: bit-casting a vector-element
            // lvalue reads element 0
            const unsigned int ua = fa[0][i][sub], ub = fb[0][j][sub];
            const float a = __uint_as_float(ua);
            const float b = __uint_as_float(ub);
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b, a, acc[i][j], 0, 0, 0);
          }
    }
    if (has_next) store(buf ^ 1);
    __syncthreads();
    buf ^= 1;
    s = ns;
    k0 = nk0;
  }

  if (slice < 0)
    store_tile<FM, FN>(acc, resolve(src, P.C), P.ldc, P.M, P.N, m0 + wm0, n0 + wn0, li, lg, P.alpha, P.beta);
  else
    store_partial(acc, src_partial<float>(src, t, slice, BM * BN), wave, lane);
  }  // units
}

// Raw (stride 0) buffer resource over p with num_records = 2^31 - 1 bytes and
// the gfx9 data-format word; offsets at or past num_records load zeros.
constexpr unsigned OOB = 0x80000000u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t raw_rsrc(const void* p) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, 0x7fffffff, 0x00020000);
}

typedef __attribute__((address_space(3))) void lds_void;

// ---------------------------------------------------------------------------
// Operands straight to LDS (buffer_load ... lds, 16 bytes a lane).  A K step is
// 64 bytes of every row; a load instruction fills 16 rows of the slab in lane
// order, and lane l takes the chunk of row l / 4 that swz puts at slot l % 4.
// Packed operands (256-row panels of contiguous 16 KB K steps) are read the same
// way with rows of 64 bytes.  Two stages; the loads of step s + 1 go out at the
// start of step s, and its barrier sits before the last MFMAs, which cover the
// latency of the next step's first fragment reads.  Rows and K chunks outside an
// operand get a buffer offset past num_records, which loads zeros.  Needs 256
// rows of every operand within 2 GiB of the row base (checked on the host).
//
// 128 x 128 and 64 x 64 tiles: 4 waves (2 x 2), two or more workgroups a CU, both
// fragment sets in registers.  256 x 256: 8 waves (2 x 4) of 128 x 64, one
// workgroup a CU; the next step's B fragments and first A fragment are read
// ahead, the other A fragments one block ahead of their MFMAs.
// ---------------------------------------------------------------------------
template <int BM, int BN, int WGM, int WGN, int MODE, class Src>
__global__ __launch_bounds__(64 * WGM * WGN) __attribute__((amdgpu_waves_per_eu(2)))
void gemm_mixed_dma_kernel(Src src) {
  constexpr int NPART = MODE == M_BF16X3 ? 2 : 1;
  constexpr int EB = MODE == M_BF16X3 ? 2 : 4;
  constexpr int NW = WGM * WGN;
  constexpr int WM = BM / WGM, WN = BN / WGN;
  constexpr int FM = WM / 16, FN = WN / 16;
  constexpr int CHA = BM / 16 / NW, CHB = BN / 16 / NW;   // load instructions a wave and part
  constexpr int KSTEP = ROWB / EB;
  constexpr bool BIGT = FM > 4;                           // A fragments streamed

  __shared__ __attribute__((aligned(1024))) char As0[NPART * BM * ROWB];
  __shared__ __attribute__((aligned(1024))) char As1[NPART * BM * ROWB];
  __shared__ __attribute__((aligned(1024))) char Bs0[NPART * BN * ROWB];
  __shared__ __attribute__((aligned(1024))) char Bs1[NPART * BN * ROWB];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm0 = (wave % WGM) * WM;
  const int wn0 = (wave / WGM) * WN;
  const int li = lane & 15;
  const int lg = lane >> 4;
  const int cq = (lane & 3) ^ (-(lane >> 4) & 3);         // chunk this lane loads (row lane / 4)
  const int aoff = swz(wm0 + li, lg), boff = swz(wn0 + li, lg);

  for (int un = src_first(src); un < src_units(src); un += src_stride(src)) {
  int t, slice, nslice;
  src_unit(src, un, t, slice, nslice);
  const GemmProb& P = src_prob(src, t);
  int tm, tn;
  tile_coords(P, t - P.tile_start, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;

  fx4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = fx4{0.f, 0.f, 0.f, 0.f};

  int nsteps = 0;
  for (int s = 0; s < P.nseg; ++s) nsteps += (P.seg[s].K + KSTEP - 1) / KSTEP;

  __amdgpu_buffer_rsrc_t rA[NPART], rB[NPART];
  unsigned vA[CHA], vB[CHB];               // the lane's offset in load c (OOB: row outside)
  unsigned csA = 0, csB = 0, w0A = 0, w0B = 0, kmA = 1, kmB = 1;
  int Kb = 0, kend = 0;
  auto set_side = [&](bool packed, const char* hi, const char* lo, int64_t ld, int64_t Kbytes, int r0, int lim, int CH,
                      __amdgpu_buffer_rsrc_t* rs, unsigned* v, unsigned& cs, unsigned& w0, unsigned& km) {
    const int64_t pitch = packed ? ROWB : ld * EB;
    const int64_t off = packed ? (int64_t)(r0 / 256) * Kbytes * 256 : (int64_t)r0 * pitch;
    rs[0] = raw_rsrc(hi + off);
    if constexpr (NPART == 2) rs[1] = raw_rsrc(lo + off);
    km = packed ? 256u : 1u;
    cs = (unsigned)(16 * NW * pitch);
    w0 = (unsigned)(16 * wave * pitch);
    const unsigned o = (unsigned)((lane >> 2) * pitch + cq * 16);
#pragma unroll
    for (int c = 0; c < CH; ++c) v[c] = r0 + 16 * (wave + NW * c) + (lane >> 2) < lim ? o : OOB;
  };
  auto set_seg = [&](int s) {
    const GemmSeg& S = P.seg[s];
    const int64_t kb = (int64_t)S.K * EB;
    set_side((S.vec & 2) != 0, static_cast<const char*>(resolve(src, S.A)),
             NPART == 2 ? static_cast<const char*>(resolve(src, S.Alo)) : nullptr, S.lda, kb, m0, P.M, CHA, rA, vA, csA,
             w0A, kmA);
    set_side((S.vec & 4) != 0, static_cast<const char*>(resolve(src, S.B)),
             NPART == 2 ? static_cast<const char*>(resolve(src, S.Blo)) : nullptr, S.ldb, kb, n0, P.N, CHB, rB, vB, csB,
             w0B, kmB);
    Kb = (int)kb;
    kend = S.K;
  };
  auto fetch_side = [&](int R, int CH, const __amdgpu_buffer_rsrc_t* rs, const unsigned* v, unsigned cs, unsigned w0,
                        unsigned km, int kb0, char* S) {
    const bool tail = kb0 + ROWB > Kb;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      unsigned o = v[c];
      if (tail) o = kb0 + cq * 16 < Kb ? o : OOB;
      const int so = (int)(w0 + c * cs + (unsigned)kb0 * km);
#pragma unroll
      for (int p = 0; p < NPART; ++p)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs[p], (lds_void*)(S + p * R * ROWB + (wave + NW * c) * 1024), 16,
                                                 (int)o, so, 0, 0);
    }
  };
  int s, k0, step0, step1;
  slice_range<KSTEP>(P, nsteps, slice, nslice, step0, step1, s, k0);
  auto fetch = [&](char* A, char* B) {
    fetch_side(BM, CHA, rA, vA, csA, w0A, kmA, k0 * EB, A);
    fetch_side(BN, CHB, rB, vB, csB, w0B, kmB, k0 * EB, B);
  };
  auto read_a = [&](const char* A, int i, ux4 (&f)[NPART]) {
#pragma unroll
    for (int p = 0; p < NPART; ++p) f[p] = *reinterpret_cast<const ux4*>(A + p * BM * ROWB + aoff + i * 16 * ROWB);
  };
  auto read_b = [&](const char* B, ux4 (&f)[NPART][FN]) {
#pragma unroll
    for (int p = 0; p < NPART; ++p)
#pragma unroll
      for (int j = 0; j < FN; ++j) f[p][j] = *reinterpret_cast<const ux4*>(B + p * BN * ROWB + boff + j * 16 * ROWB);
  };
  // one product (MODE F32: one of the four k of a chunk) of row block i
  auto mfma1 = [&](int i, const ux4 (&a)[NPART], const ux4 (&b)[NPART][FN], int part) {
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      if constexpr (MODE == M_BF16X3) {
        // hi*lo, lo*hi, then hi*hi
        const bfx8 av = __builtin_bit_cast(bfx8, part == 0 ? a[NPART - 1] : a[0]);
        const bfx8 bv = __builtin_bit_cast(bfx8, part == 1 ? b[NPART - 1][j] : b[0][j]);
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bv, av, acc[i][j], 0, 0, 0);
      } else {
        const unsigned int ua = a[0][part], ub = b[0][j][part];
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(ub), __uint_as_float(ua), acc[i][j], 0, 0, 0);
      }
    }
  };
  constexpr int NPROD = MODE == M_BF16X3 ? 3 : 4;
  ux4 fa[BIGT ? 2 : FM][NPART], fb[NPART][FN];
  auto body = [&](const char* A, const char* B, char* An, char* Bn, bool has_next) {
    if (has_next) {
      k0 += KSTEP;
      while (k0 >= kend && s + 1 < P.nseg) {
        ++s;
        k0 = 0;
        set_seg(s);
      }
      fetch(An, Bn);
    }
    if constexpr (!BIGT) {
      ux4 na[FM][NPART], nb[NPART][FN];
#pragma unroll
      for (int q = 0; q + 1 < NPROD; ++q)
#pragma unroll
        for (int i = 0; i < FM; ++i) mfma1(i, fa[i], fb, q);
      __builtin_amdgcn_sched_barrier(0);
      __syncthreads();
      __builtin_amdgcn_sched_barrier(0);
      if (has_next) {
        read_b(Bn, nb);
#pragma unroll
        for (int i = 0; i < FM; ++i) read_a(An, i, na[i]);
      }
#pragma unroll
      for (int i = 0; i < FM; ++i) mfma1(i, fa[i], fb, NPROD - 1);
#pragma unroll
      for (int p = 0; p < NPART; ++p) {
#pragma unroll
        for (int j = 0; j < FN; ++j) fb[p][j] = nb[p][j];
#pragma unroll
        for (int i = 0; i < FM; ++i) fa[i][p] = na[i][p];
      }
    } else {
      ux4 nb[NPART][FN];
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        if (i + 1 < FM) {
          read_a(A, i + 1, fa[(i + 1) & 1]);
        } else {
          __builtin_amdgcn_sched_barrier(0);
          __syncthreads();
          __builtin_amdgcn_sched_barrier(0);
          if (has_next) {
            read_b(Bn, nb);
            read_a(An, 0, fa[0]);
          }
        }
#pragma unroll
        for (int q = 0; q < NPROD; ++q) mfma1(i, fa[i & 1], fb, q);
      }
#pragma unroll
      for (int p = 0; p < NPART; ++p)
#pragma unroll
        for (int j = 0; j < FN; ++j) fb[p][j] = nb[p][j];
    }
  };
  if (step1 > step0) {
    set_seg(s);
    fetch(As0, Bs0);
    __syncthreads();
    read_b(Bs0, fb);
    if constexpr (BIGT) {
      read_a(As0, 0, fa[0]);
    } else {
#pragma unroll
      for (int i = 0; i < FM; ++i) read_a(As0, i, fa[i]);
    }
  }
  for (int step = step0; step < step1; step += 2) {
    body(As0, Bs0, As1, Bs1, step + 1 < step1);
    if (step + 1 < step1) body(As1, Bs1, As0, Bs0, step + 2 < step1);
  }

  if (slice < 0)
    store_tile<FM, FN>(acc, resolve(src, P.C), P.ldc, P.M, P.N, m0 + wm0, n0 + wn0, li, lg, P.alpha, P.beta);
  else
    store_partial(acc, src_partial<float>(src, t, slice, BM * BN), wave, lane);
  }  // units
}

template <int BM, int BN, int MODE, int VAR>
mk_status launch_mixed(const ProbSpec* probs, int nprob, hipStream_t stream, SplitPlan sp, void* ws) {
  constexpr int EB = MODE == M_BF16X3 ? 2 : 4;
  GemmBatch b{};
  int total = 0;
  for (int i = 0; i < nprob; ++i) {
    const ProbSpec& ps = probs[i];
    GemmProb& P = b.p[i];
    P.M = (int32_t)ps.M;
    P.N = (int32_t)ps.N;
    P.nseg = 0;
    for (int s = 0; s < ps.nseg; ++s) {
      if (ps.seg[s].K <= 0) continue;
      const SegSpec& q = ps.seg[s];
      MK_REQUIRE(q.lda % 8 == 0 && q.ldb % 8 == 0 && q.K <= q.lda && q.K <= q.ldb, MK_BAD_ARG,
                 "mixed gemm: K-contiguous operands need row length padded to 8 (lda=%lld ldb=%lld K=%lld)",
                 (long long)q.lda, (long long)q.ldb, (long long)q.K);
      const void* ptrs[4] = {q.A, q.B, q.Alo, q.Blo};
      for (int z = 0; z < (MODE == M_BF16X3 ? 4 : 2); ++z)
        MK_REQUIRE(ptrs[z] != nullptr && (uintptr_t)ptrs[z] % 16 == 0, MK_BAD_ARG,
                   "mixed gemm: operands must be non-null and 16-byte aligned");
      GemmSeg& gs = P.seg[P.nseg++];
      gs.A = q.A; gs.B = q.B; gs.Alo = q.Alo; gs.Blo = q.Blo;
      gs.lda = q.lda; gs.ldb = q.ldb;
      // K rounded up to the padded row: the padding is zero
      gs.K = (int32_t)((q.K + 7) / 8 * 8);
      // bit 0: vector loads; bits 1, 2: A, B in the packed panel layout
      gs.vec = 1 | (q.packA ? 2 : 0) | (q.packB ? 4 : 0);
      if (q.packA || q.packB)
        MK_REQUIRE(VAR == V_DMA && BM == 256 && ps.M % 256 == 0 && ps.N % 256 == 0 && q.K % 32 == 0, MK_BAD_ARG,
                   "mixed gemm: packed operands need the 256 x 256 kernel, M, N multiples of 256 and K of 32");
    }
    P.tiles_m = (int32_t)cdiv(ps.M, BM);
    P.tiles_n = (int32_t)cdiv(ps.N, BN);
    P.tile_start = total;
    total += P.tiles_m * P.tiles_n;
    P.C = ps.C; P.ldc = ps.ldc; P.alpha = ps.alpha; P.beta = ps.beta;
  }
  (void)EB;
  b.nprob = nprob;
  b.total_tiles = total;
  if (total == 0) return MK_OK;
  b.full_tiles = sp.ksplit > 1 ? sp.full : total;
  b.ksplit = b.full_tiles < total ? sp.ksplit : 1;
  b.ws = ws;
  const int tail = total - b.full_tiles, units = b.full_tiles + tail * b.ksplit;
  MK_REQUIRE(tail == 0 || (ws != nullptr && (size_t)tail * b.ksplit * BM * BN * 4 <= GEMM_WS_BYTES), MK_BAD_ARG,
             "mixed gemm: %d tiles split %d ways exceed the workspace", tail, b.ksplit);
  ProfScope prof(MODE == M_BF16X3 ? "gemm_bf16x3" : "gemm_f32", stream);
  constexpr int WGN = BM == 256 ? 4 : 2;   // waves along N (two along M)
  if constexpr (VAR == V_DMA)
    hipLaunchKernelGGL((gemm_mixed_dma_kernel<BM, BN, 2, WGN, MODE, GemmBatch>), dim3(units), dim3(128 * WGN), 0, stream, b);
  else
    hipLaunchKernelGGL((gemm_mixed_kernel<BM, BN, MODE, GemmBatch>), dim3(units), dim3(NT), 0, stream, b);
  MK_CHECK_HIP(hipGetLastError());
  if (tail > 0) {
    constexpr int NBLK = BM * BN / 256;
    hipLaunchKernelGGL((splitk_reduce_kernel<true, 2, BM / 32, BN / 16 / WGN, WGN, fx4>),
                       dim3((unsigned)cdiv((int64_t)tail * NBLK, 4)), dim3(256), 0, stream, b);
    MK_CHECK_HIP(hipGetLastError());
  }
  return MK_OK;
}

// 256 rows of every operand lie within the 32-bit buffer offsets of gemm_mixed_dma_kernel
template <int MODE>
bool rows256_fit(const ProbSpec* probs, int nprob) {
  constexpr int64_t EB = MODE == M_BF16X3 ? 2 : 4;
  for (int i = 0; i < nprob; ++i)
    for (int s = 0; s < probs[i].nseg; ++s)
      if (256 * std::max(probs[i].seg[s].lda, probs[i].seg[s].ldb) * EB >= (1ll << 31)) return false;
  return true;
}

template <int MODE>
mk_status dispatch(const ProbSpec* probs, int nprob, hipStream_t stream, void* ws) {
  MK_REQUIRE(nprob >= 0 && nprob <= MAX_PROB, MK_BAD_ARG, "mixed gemm: too many problems");
  for (int i = 0; i < nprob; ++i)
    MK_REQUIRE(!probs[i].full, MK_BAD_ARG, "mixed gemm: more than %d segments", MAX_SEG);
  constexpr int EB = MODE == M_BF16X3 ? 2 : 4;
  const bool dma = variant() == V_DMA && rows256_fit<MODE>(probs, nprob);
  bool packed = false;
  for (int i = 0; i < nprob; ++i)
    for (int s = 0; s < probs[i].nseg; ++s) packed = packed || probs[i].seg[s].packA || probs[i].seg[s].packB;
  if (packed) {
    MK_REQUIRE(dma, MK_BAD_ARG, "mixed gemm: packed operands are read by the 256 x 256 kernel only");
    return launch_mixed<256, 256, MODE, V_DMA>(probs, nprob, stream, SplitPlan{}, ws);
  }
  // Measured on 2048 x 2048 x 4096, 1024 x 2048 x 2048 and 1024 x 1024 x 2048.  The
  // bf16 steps are short (48 MFMAs of 16 cycles a wave on a 128 x 128 tile), so
  // one step of prefetch covers little of the load latency, and the operand
  // traffic of a small tile (32 KB a step through the CU's 64 B / cycle) is near
  // its limit: large tiles cut along K win.  The fp32 steps are 2.7 times longer.
  static const TileModel m64{64, 64, ROWB / EB, MODE == M_BF16X3 ? 0.095 : 0.22,
                             MODE == M_BF16X3 ? TileModel::Eff{0.18, 0.33, 0.38, 0.40} : TileModel::Eff{0.47, 0.70, 0.76, 0.78},
                             4, 64 * 64 * 4};
  static const TileModel m128{128, 128, ROWB / EB, MODE == M_BF16X3 ? 0.38 : 0.87,
                              MODE == M_BF16X3 ? TileModel::Eff{0.39, 0.55, 0.55, 0.55} : TileModel::Eff{0.80, 0.84, 0.84, 0.84},
                              2, 128 * 128 * 4};
  static const TileModel m256{256, 256, ROWB / EB, MODE == M_BF16X3 ? 1.5 : 3.5,
                              MODE == M_BF16X3 ? TileModel::Eff{0.60, 0.60, 0.60, 0.60} : TileModel::Eff{0.89, 0.89, 0.89, 0.89},
                              1, 256 * 256 * 4};
  const TileChoice c64 = plan_launch(m64, probs, nprob, ws != nullptr);
  const TileChoice c128 = plan_launch(m128, probs, nprob, ws != nullptr);
  if (!dma) {
    if (c128.us <= c64.us) return launch_mixed<128, 128, MODE, V_TILE>(probs, nprob, stream, c128.split, ws);
    return launch_mixed<64, 64, MODE, V_TILE>(probs, nprob, stream, c64.split, ws);
  }
  const TileChoice c256 = plan_launch(m256, probs, nprob, ws != nullptr);
  if (c256.us <= c128.us && c256.us <= c64.us)
    return launch_mixed<256, 256, MODE, V_DMA>(probs, nprob, stream, c256.split, ws);
  if (c128.us <= c64.us) return launch_mixed<128, 128, MODE, V_DMA>(probs, nprob, stream, c128.split, ws);
  return launch_mixed<64, 64, MODE, V_DMA>(probs, nprob, stream, c64.split, ws);
}

template <int MODE>
mk_status launch_group(const GemmGroup& g, int kind, int grid, hipStream_t stream) {
  if (g.total_tiles == 0) return MK_OK;
  ProfScope prof(MODE == M_BF16X3 ? "gemm_bf16x3" : "gemm_f32", stream);
  const bool dma = variant() == V_DMA && g.rows256_fit;
  MK_REQUIRE(kind != TK_256 || dma, MK_BAD_ARG, "grouped mixed gemm: 256 x 256 tiles need operand rows within 2 GiB");
  if (kind == TK_256)
    hipLaunchKernelGGL((gemm_mixed_dma_kernel<256, 256, 2, 4, MODE, GemmGroup>), dim3(grid), dim3(512), 0, stream, g);
  else if (kind == TK_128 && dma)
    hipLaunchKernelGGL((gemm_mixed_dma_kernel<128, 128, 2, 2, MODE, GemmGroup>), dim3(grid), dim3(NT), 0, stream, g);
  else if (dma)
    hipLaunchKernelGGL((gemm_mixed_dma_kernel<64, 64, 2, 2, MODE, GemmGroup>), dim3(grid), dim3(NT), 0, stream, g);
  else if (kind == TK_128)
    hipLaunchKernelGGL((gemm_mixed_kernel<128, 128, MODE, GemmGroup>), dim3(grid), dim3(NT), 0, stream, g);
  else
    hipLaunchKernelGGL((gemm_mixed_kernel<64, 64, MODE, GemmGroup>), dim3(grid), dim3(NT), 0, stream, g);
  MK_CHECK_HIP(hipGetLastError());
  return MK_OK;
}

template <class K>
int occ_of(K kern, int threads) {
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kern, threads, 0) != hipSuccess) n = 1;
  return n > 0 ? n : 1;
}

}  // namespace

int mixed_group_grid(int prec, int kind, int total_tiles, int cus) {
  // occupancy is a property of the kernel's resources; the BF16X3 instances are the larger
  static const int occ[3] = {occ_of(gemm_mixed_dma_kernel<64, 64, 2, 2, M_BF16X3, GemmGroup>, NT),
                             occ_of(gemm_mixed_dma_kernel<128, 128, 2, 2, M_BF16X3, GemmGroup>, NT),
                             occ_of(gemm_mixed_dma_kernel<256, 256, 2, 4, M_BF16X3, GemmGroup>, 512)};
  (void)prec;
  return (int)std::min<int64_t>(total_tiles, (int64_t)occ[kind] * cus);
}

mk_status gemm_mixed_group(const GemmGroup& g, int prec, int kind, int grid, hipStream_t st) {
  MK_REQUIRE(kind >= TK_64 && kind <= TK_256, MK_BAD_ARG, "gemm_mixed_group: tile kind %d", kind);
  if (prec == MK_BF16X3) return launch_group<M_BF16X3>(g, kind, grid, st);
  return launch_group<M_F32>(g, kind, grid, st);
}

bool mixed_256_ok() { return variant() == V_DMA; }

bool mixed_packed_ok(int64_t M, int64_t N, const int64_t* Ks, int nk) {
  if (variant() != V_DMA || M % 256 || N % 256 || (M / 256) * (N / 256) < 256) return false;
  for (int i = 0; i < nk; ++i)
    // a panel (256 rows x K, fp32 the wider) must stay within 32-bit buffer offsets
    if (Ks[i] % 32 || Ks[i] * 4 * 256 >= (1ll << 31)) return false;
  return true;
}

mk_status gemm_bf16x3(const ProbSpec* probs, int nprob, hipStream_t stream, void* ws) {
  return dispatch<M_BF16X3>(probs, nprob, stream, ws);
}
mk_status gemm_f32(const ProbSpec* probs, int nprob, hipStream_t stream, void* ws) {
  return dispatch<M_F32>(probs, nprob, stream, ws);
}

}  // namespace mk
