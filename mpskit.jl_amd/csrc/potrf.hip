// Blocked Cholesky factorisation A = L L^T of a symmetric positive definite
// float64 matrix (column-major, lower triangle used), for the Cholesky QR of
// the gauge steps.  A 64-column step is one launch: the panel below the factored
// diagonal block is L21 = A21 L11^-T, the trailing update A22 -= L21 L21^T, and the
// first block of what is left is factored and inverted beside the rest of the update
// (the inverted diagonal block turns the row-serial triangular solve into a parallel
// product, as GPU Cholesky codes commonly do).
#include <algorithm>

#include "kernels.h"
#include "ops.h"

namespace mk {
namespace {

constexpr int NB = 64;        // block columns per step
constexpr int PT = 256;       // threads of the block kernels: 4 waves
constexpr int SB = 16;        // sub-block: an MFMA tile, and the columns a wave factors in registers
constexpr int LD = NB + 1;    // LDS row length

typedef __attribute__((address_space(1))) double gdouble;
typedef double dx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ double lane_value(double v, int lane) {
  const unsigned long long u = __double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_readlane((unsigned)u, lane), hi = __builtin_amdgcn_readlane((unsigned)(u >> 32), lane);
  return __longlong_as_double(((unsigned long long)hi << 32) | lo);
}

// acc += A B for 16 x 16 blocks in LDS: A(i, k) = a[i * ai + k * ak], B(k, j) = b[k * bk + j * bj].
// Lane (li, lq) then holds rows lq + 4 r, column li of the product.
__device__ __forceinline__ void mm16(dx4& acc, const double* a, int ai, int ak, const double* b, int bk, int bj, int li,
                                     int lq) {
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) {
    const int k = 4 * kk + lq;
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[li * ai + k * ak], b[k * bk + li * bj], acc, 0, 0, 0);
  }
}

// One wave's LDS writes before its own later reads of other lanes' values.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Factor the nb x nb diagonal block at (k0, k0), which the workgroup holds in S
// (lower triangle, identity outside nb), and invert the factor.  What
// bounds it is the serial chain of the 64 pivots.  The block goes through in 16
// columns at a time: wave 0 keeps a row of them per lane and factors them
// without a barrier (pivots and column entries pass between lanes by
// v_readlane), the four waves update what is to the right on the matrix cores.
// The inverse is by blocks too: the four diagonal 16 x 16 blocks by
// substitution, one wave each, then column j of blocks by wave j,
// X_ij = -X_ii sum_k L_ik X_kj.  (One column per step over the whole block, with
// a workgroup barrier each, took 94 us, all but 4 us of it waiting.)
// A non-positive or non-finite pivot sets *info = k0 + j + 1 (LAPACK's
// convention); the block then stays as it was.  Writes L11 (zeros above the
// diagonal) into A and L11^-1 into Linv (ld NB, zeros above the diagonal);
// columns nb and on are those of the identity.  S and X: S[r LD + c], X zero;
// the caller's writes to them are its own threads' (the barrier is here).
__device__ void factor_block(double* S, double* X, double (*T)[SB * (SB + 1)], int* bad, gdouble* gA, int64_t lda, int k0,
                             int nb, double* __restrict__ Linv, int* __restrict__ info) {
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63, li = lane & 15, lq = lane >> 4;
  if (t == 0) *bad = 0;
  __syncthreads();
  for (int p = 0; p < NB / SB; ++p) {
    if (wave == 0) {
      double a[SB];
#pragma unroll
      for (int c = 0; c < SB; ++c) a[c] = S[lane * LD + p * SB + c];
      int b = 0;
#pragma unroll
      for (int j = 0; j < SB; ++j) {
        const int piv = p * SB + j;
        const double d = lane_value(a[j], piv);
        if (b == 0 && (!(d > 0.0) || !isfinite(d))) b = piv + 1;
        const double inv = rsqrt(d);
        a[j] = lane > piv ? a[j] * inv : (lane == piv ? d * inv : 0.0);
#pragma unroll
        for (int c = j + 1; c < SB; ++c) a[c] -= a[j] * lane_value(a[j], p * SB + c);
      }
#pragma unroll
      for (int c = 0; c < SB; ++c) S[lane * LD + p * SB + c] = a[c];
      if (lane == 0 && b != 0) *bad = b;
    }
    __syncthreads();
    if (*bad != 0) {
      if (t == 0) *info = k0 + *bad;
      return;
    }
    // blocks (rb, cb), p < cb <= rb, of the rest: S -= L_rb L_cb^T
    int id = 0;
    for (int cb = p + 1; cb < NB / SB; ++cb)
      for (int rb = cb; rb < NB / SB; ++rb, ++id) {
        if ((id & 3) != wave) continue;
        double* C = S + rb * SB * LD + cb * SB;
        dx4 acc;
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] = -C[(lq + 4 * r) * LD + li];
        mm16(acc, S + rb * SB * LD + p * SB, LD, 1, S + cb * SB * LD + p * SB, 1, LD, li, lq);
#pragma unroll
        for (int r = 0; r < 4; ++r) C[(lq + 4 * r) * LD + li] = -acc[r];
      }
    __syncthreads();
  }
#pragma unroll
  for (int q = 0; q < NB * NB / PT; ++q) {
    const int c = wave + 4 * q, r = lane;
    if (r < nb && c < nb) gA[(int64_t)(k0 + r) + (int64_t)(k0 + c) * lda] = r >= c ? S[r * LD + c] : 0.0;
  }
  // diagonal block `wave`: lane c < 16 solves L x = e_c
  {
    const double* L = S + wave * SB * (LD + 1);
    double x[SB];
#pragma unroll
    for (int i = 0; i < SB; ++i) {
      double s = i == li ? 1.0 : 0.0;
#pragma unroll
      for (int k = 0; k < i; ++k) s -= L[i * LD + k] * x[k];
      x[i] = s / L[i * LD + i];
    }
    if (lane < SB) {
#pragma unroll
      for (int i = 0; i < SB; ++i) X[(wave * SB + i) * LD + wave * SB + li] = x[i];
    }
  }
  __syncthreads();
  if (wave < 3) {
    double* Tw = T[wave];
    for (int i = wave + 1; i < NB / SB; ++i) {
      dx4 acc = {0.0, 0.0, 0.0, 0.0};
      for (int k = wave; k < i; ++k)
        mm16(acc, S + i * SB * LD + k * SB, LD, 1, X + k * SB * LD + wave * SB, LD, 1, li, lq);
#pragma unroll
      for (int r = 0; r < 4; ++r) Tw[(lq + 4 * r) * (SB + 1) + li] = -acc[r];
      wave_lds_fence();
      acc = dx4{0.0, 0.0, 0.0, 0.0};
      mm16(acc, X + i * SB * (LD + 1), LD, 1, Tw, SB + 1, 1, li, lq);
#pragma unroll
      for (int r = 0; r < 4; ++r) X[(i * SB + lq + 4 * r) * LD + wave * SB + li] = acc[r];
      wave_lds_fence();
    }
  }
  __syncthreads();
  gdouble* gL = (gdouble*)Linv;
#pragma unroll
  for (int q = 0; q < NB * NB / PT; ++q) {
    const int c = wave + 4 * q, r = lane;
    gL[r + c * NB] = (r >= c && r < nb && c < nb) ? X[r * LD + c] : 0.0;
  }
}

// One step of the factorisation in one launch, for the trailing matrix below and
// right of the full diagonal block at (k0, k0), whose inverted factor is Linv: a
// workgroup per 64 x 64 tile (i, j) of its lower triangle forms the panel blocks
// L_ik = A_ik Linv^T and L_jk itself (the same products in every workgroup of a row,
// on CUs that would idle) and subtracts L_ik L_jk^T; the first tile's workgroup
// goes on to factor it, so the next step's pivot chain runs beside the rest of the
// update.  As others still read A_ik, the workgroups of the first column leave L_ik
// transposed above the diagonal, whence potrf_finish_kernel takes it.  k0 < 0: only
// the first block is factored.  Bounded by the pivot chain of one workgroup, 16 of
// them at n = 1024.  Against a launch each for block, panel and update (the GEMM;
// us, with the copy of info): n = 512 340 -> 297, 1024 651 -> 557, 2048 1404 -> 1110,
// 4096 3883 -> 3822.
__global__ __launch_bounds__(PT) void potrf_step_kernel(double* __restrict__ A, int64_t lda, int64_t n, int k0,
                                                        const double* __restrict__ Linv, double* __restrict__ Lnext,
                                                        int* __restrict__ info) {
  __shared__ double Ri[NB * LD];   // Ri[k LD + r] = A_ik(r, k), then L_ik; the factor of the first tile
  __shared__ double Rj[NB * LD];
  __shared__ double Ls[NB * LD];   // Ls[j LD + k] = Linv(j, k); the inverse
  __shared__ double T[3][SB * (SB + 1)];
  __shared__ int bad;
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63, li = lane & 15, lq = lane >> 4;
  gdouble* gA = (gdouble*)A;
  const int64_t b0 = k0 < 0 ? 0 : k0 + NB, m = n - b0;   // the trailing matrix
  // an earlier block failed (a failure of the block this launch factors comes with a
  // larger *info: the other workgroups still owe their part of L)
  const int failed = *(volatile const int*)info;
  if (__syncthreads_or(failed != 0 && failed <= b0)) return;
  int i = 0, j = 0;
  if (k0 >= 0) {
    // tiles by columns of the triangle: (0, 0), (1, 0), ..., (1, 1), ...
    int u = blockIdx.x;
    for (int h = (int)((m + NB - 1) / NB); u >= h; --h, ++j) u -= h;
    i = j + u;
  }
  const int64_t ri = (int64_t)i * NB, rj = (int64_t)j * NB;
  gdouble* gC = gA + (b0 + ri) + (b0 + rj) * lda;
  dx4 acc[NB / SB];
#pragma unroll
  for (int jb = 0; jb < NB / SB; ++jb) acc[jb] = dx4{0.0, 0.0, 0.0, 0.0};
  double c[NB / SB][4];   // lane's entries: row 16 wave + li, columns 16 jb + lq + 4 r
  const int row = wave * SB + li;
#pragma unroll
  for (int jb = 0; jb < NB / SB; ++jb)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int col = jb * SB + lq + 4 * r;
      c[jb][r] = ri + row < m && rj + col < m ? gC[row + (int64_t)col * lda] : 0.0;
    }
  if (k0 >= 0) {
    const gdouble* gL = (const gdouble*)Linv;
    gdouble* gP = gA + b0 + (int64_t)k0 * lda;   // the raw panel
#pragma unroll
    for (int q = 0; q < NB * NB / PT; ++q) {
      const int k = wave + 4 * q;
      Ri[k * LD + lane] = ri + lane < m ? gP[ri + lane + (int64_t)k * lda] : 0.0;
      if (i != j) Rj[k * LD + lane] = rj + lane < m ? gP[rj + lane + (int64_t)k * lda] : 0.0;
      Ls[lane * LD + k] = gL[lane + k * NB];
    }
    __syncthreads();
    // a wave's 16 rows of the panel block, in place
    auto panel = [&](double* R) {
      dx4 p[NB / SB];
#pragma unroll
      for (int jb = 0; jb < NB / SB; ++jb) {
        p[jb] = dx4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int kb = 0; kb <= jb; ++kb)
          mm16(p[jb], Ls + jb * SB * LD + kb * SB, LD, 1, R + kb * SB * LD + wave * SB, LD, 1, li, lq);
      }
      wave_lds_fence();
#pragma unroll
      for (int jb = 0; jb < NB / SB; ++jb)
#pragma unroll
        for (int r = 0; r < 4; ++r) R[(jb * SB + lq + 4 * r) * LD + row] = p[jb][r];
    };
    panel(Ri);
    if (i != j) panel(Rj);
    __syncthreads();
    if (j == 0) {
#pragma unroll
      for (int q = 0; q < NB * NB / PT; ++q) {
        const int r = wave + 4 * q;
        if (ri + r < m) gA[k0 + lane + (b0 + ri + r) * lda] = Ri[lane * LD + r];
      }
    }
    const double* L = i == j ? Ri : Rj;
#pragma unroll
    for (int kb = 0; kb < NB / SB; ++kb)
#pragma unroll
      for (int jb = 0; jb < NB / SB; ++jb)
        mm16(acc[jb], L + kb * SB * LD + jb * SB, 1, LD, Ri + kb * SB * LD + wave * SB, LD, 1, li, lq);
  }
  if (i + j > 0) {
#pragma unroll
    for (int jb = 0; jb < NB / SB; ++jb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int col = jb * SB + lq + 4 * r;
        if (ri + row < m && rj + col < m) gC[row + (int64_t)col * lda] = c[jb][r] - acc[jb][r];
      }
    return;
  }
  const int nb = (int)min((int64_t)NB, m);
  __syncthreads();   // Ri and Ls have been read
#pragma unroll
  for (int jb = 0; jb < NB / SB; ++jb)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int col = jb * SB + lq + 4 * r;
      Ri[row * LD + col] = row < nb && col <= row ? c[jb][r] - acc[jb][r] : (row == col ? 1.0 : 0.0);
      Ls[row * LD + col] = 0.0;
    }
  factor_block(Ri, Ls, T, &bad, gA, lda, (int)b0, nb, Lnext, info);
}

// The block row of L^T that the steps left above each diagonal block, to its place
// below it, and zeros above (a workgroup per 64 x 64 block on or below the diagonal;
// grid: first, second block index).  After a failed pivot the blocks from the failing
// one on have no such row: they are only cleared above the diagonal.
__global__ __launch_bounds__(PT) void potrf_finish_kernel(double* __restrict__ A, int64_t lda, int64_t n,
                                                          const int* __restrict__ info) {
  __shared__ double S[NB * LD];
  if (blockIdx.x < blockIdx.y) return;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t r0 = (int64_t)blockIdx.x * NB, c0 = (int64_t)blockIdx.y * NB;   // c0 <= r0 < n
  const int failed = *info;
  const bool done = failed == 0 || c0 + NB < failed;
  gdouble* gA = (gdouble*)A;
  if (r0 == c0) {
    if (done) return;
#pragma unroll
    for (int q = 0; q < NB * NB / PT; ++q) {
      const int r = wave + 4 * q;
      if (lane < r && r0 + r < n) gA[c0 + lane + (r0 + r) * lda] = 0.0;
    }
    return;
  }
#pragma unroll
  for (int q = 0; q < NB * NB / PT; ++q) {
    const int r = wave + 4 * q;
    if (r0 + r < n) {
      gdouble* p = gA + c0 + lane + (r0 + r) * lda;
      S[r * LD + lane] = *p;
      *p = 0.0;
    }
  }
  if (!done) return;
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NB * NB / PT; ++q) {
    const int c = wave + 4 * q;
    if (r0 + lane < n) gA[r0 + lane + (c0 + c) * lda] = S[lane * LD + c];
  }
}

}  // namespace

mk_status potrf_lower(double* A, int64_t n, int64_t lda, int* info_dev, double* Linv, hipStream_t st) {
  MK_REQUIRE(n >= 0 && lda >= std::max<int64_t>(n, 1), MK_BAD_SHAPE, "potrf: n %lld, lda %lld", (long long)n,
             (long long)lda);
  MK_REQUIRE(n < (1 << 30), MK_BAD_SHAPE, "potrf: n %lld too large", (long long)n);
  if (n == 0) return MK_OK;
  for (int64_t k0 = -NB; k0 + NB < n; k0 += NB) {
    const int64_t nt = k0 < 0 ? 1 : cdiv(n - k0 - NB, (int64_t)NB), odd = (k0 / NB) & 1;
    hipLaunchKernelGGL(potrf_step_kernel, dim3((unsigned)(nt * (nt + 1) / 2)), dim3(PT), 0, st, A, lda, n, (int)k0,
                       Linv + odd * NB * NB, Linv + (1 - odd) * NB * NB, info_dev);
    MK_CHECK_HIP(hipGetLastError());
  }
  const unsigned nblk = (unsigned)cdiv(n, (int64_t)NB);
  hipLaunchKernelGGL(potrf_finish_kernel, dim3(nblk, nblk), dim3(PT), 0, st, A, lda, n, info_dev);
  MK_CHECK_HIP(hipGetLastError());
  return MK_OK;
}

}  // namespace mk

using namespace mk;

extern "C" mk_status mk_potrf(mk_ctx h, double* A, int64_t n, int64_t lda, int* info) {
  MK_REQUIRE(h != nullptr && A != nullptr && info != nullptr, MK_BAD_ARG, "potrf: null argument");
  Ctx* ctx = reinterpret_cast<Ctx*>(h);
  MK_CHECK_HIP(hipSetDevice(ctx->device));
  hipStream_t st = ctx->stream;
  void* mem = nullptr;
  MK_TRY(ctx->small(256, &mem));
  int* dinfo = static_cast<int*>(mem);
  double* Linv = nullptr;   // inverted diagonal blocks, this step's and the next's
  MK_TRY(carve(ctx, {{(size_t)2 * NB * NB * 8, (void**)&Linv}}));
  MK_CHECK_HIP(hipMemsetAsync(dinfo, 0, sizeof(int), st));
  MK_TRY(potrf_lower(A, n, lda, dinfo, Linv, st));
  MK_CHECK_HIP(hipMemcpyAsync(info, dinfo, sizeof(int), hipMemcpyDeviceToHost, st));
  MK_CHECK_HIP(hipStreamSynchronize(st));
  return MK_OK;
}
