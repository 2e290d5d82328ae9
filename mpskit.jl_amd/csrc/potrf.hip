// Blocked Cholesky factorisation A = L L^T of a symmetric positive definite
// float64 matrix (column-major, lower triangle used), for the Cholesky QR of
// the gauge steps.  A 64-column step is two small kernels and an MFMA GEMM:
// the diagonal block is factored and inverted (L11^-1) by one workgroup; the
// panel below it is then the product L21 = A21 L11^-T, in place, and the
// trailing update A22 -= L21 L21^T the GEMM (the inverted diagonal block turns
// the row-serial triangular solve into a parallel product, as GPU Cholesky
// codes commonly do).
#include <algorithm>

#include "gemm.h"
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

// Factor the nb x nb diagonal block at (k0, k0) and invert the factor.  What
// bounds it is the serial chain of the 64 pivots.  The block goes through in 16
// columns at a time: wave 0 keeps a row of them per lane and factors them
// without a barrier (pivots and column entries pass between lanes by
// v_readlane), the four waves update what is to the right on the matrix cores.
// The inverse is by blocks too: the four diagonal 16 x 16 blocks by
// substitution, one wave each, then column j of blocks by wave j,
// X_ij = -X_ii sum_k L_ik X_kj.  (One column per step over the whole block, with
// a workgroup barrier each, took 94 us, all but 4 us of it waiting.)
// A non-positive or non-finite pivot sets *info = k0 + j + 1 (LAPACK's
// convention) and nothing more is written.  Writes L11 (zeros above the
// diagonal) into A and L11^-1 into Linv (ld NB, zeros above the diagonal);
// columns nb and on are those of the identity.
__global__ __launch_bounds__(PT) void potrf_diag_kernel(double* __restrict__ A, int64_t lda, int k0, int nb,
                                                        double* __restrict__ Linv, int* __restrict__ info) {
  __shared__ double S[NB * LD];    // the block, then its factor: S[r LD + c]
  __shared__ double X[NB * LD];    // the inverse
  __shared__ double T[3][SB * (SB + 1)];
  __shared__ int bad;
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63, li = lane & 15, lq = lane >> 4;
  gdouble* gA = (gdouble*)A;
  if (*(volatile int*)info != 0) return;   // an earlier block failed
  if (t == 0) bad = 0;
#pragma unroll
  for (int q = 0; q < NB * NB / PT; ++q) {
    const int c = wave + 4 * q, r = lane;
    S[r * LD + c] = (r < nb && c <= r) ? gA[(int64_t)(k0 + r) + (int64_t)(k0 + c) * lda] : (r == c ? 1.0 : 0.0);
    X[r * LD + c] = 0.0;
  }
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
      if (lane == 0 && b != 0) bad = b;
    }
    __syncthreads();
    if (bad != 0) {
      if (t == 0) *info = k0 + bad;
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

// L21 = A21 L11^-T in place for the m rows below a full (64-column) diagonal
// block: a workgroup takes 64 rows, a wave 16 of them, so every row is read by
// the workgroup that writes it.  Bounded by launch and one round trip to memory
// (10 MFMAs a 16 x 16 block at most: the zero blocks of L11^-1 are left out).
__global__ __launch_bounds__(PT) void potrf_panel_kernel(double* __restrict__ A21, int64_t lda, int64_t m,
                                                         const double* __restrict__ Linv,
                                                         const int* __restrict__ info) {
  __shared__ double Rs[NB * LD];   // Rs[k LD + r] = A21(r, k)
  __shared__ double Ls[NB * LD];   // Ls[j LD + k] = L11^-1(j, k)
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63, li = lane & 15, lq = lane >> 4;
  if (*(volatile const int*)info != 0) return;
  const int64_t r0 = (int64_t)blockIdx.x * NB;
  gdouble* gA = (gdouble*)A21;
  const gdouble* gL = (const gdouble*)Linv;
#pragma unroll
  for (int q = 0; q < NB * NB / PT; ++q) {
    const int k = wave + 4 * q;
    Rs[k * LD + lane] = r0 + lane < m ? gA[r0 + lane + (int64_t)k * lda] : 0.0;
    Ls[lane * LD + k] = gL[lane + k * NB];
  }
  __syncthreads();
  const int64_t row = r0 + wave * SB + li;
#pragma unroll
  for (int jb = 0; jb < NB / SB; ++jb) {
    dx4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int kb = 0; kb <= jb; ++kb)
      mm16(acc, Ls + jb * SB * LD + kb * SB, LD, 1, Rs + kb * SB * LD + wave * SB, LD, 1, li, lq);
    if (row < m) {
#pragma unroll
      for (int r = 0; r < 4; ++r) gA[row + (int64_t)(jb * SB + lq + 4 * r) * lda] = acc[r];
    }
  }
}

// Zero the strict upper triangle of the first n columns (the factor is L).
__global__ void zero_upper_kernel(double* __restrict__ A, int64_t lda, int64_t n) {
  gdouble* gA = (gdouble*)A;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n * n; e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = e % n, c = e / n;
    if (r < c) gA[r + c * lda] = 0.0;
  }
}

}  // namespace

mk_status potrf_lower(double* A, int64_t n, int64_t lda, int* info_dev, double* Linv, hipStream_t st) {
  MK_REQUIRE(n >= 0 && lda >= std::max<int64_t>(n, 1), MK_BAD_SHAPE, "potrf: n %lld, lda %lld", (long long)n,
             (long long)lda);
  MK_REQUIRE(n < (1 << 30), MK_BAD_SHAPE, "potrf: n %lld too large", (long long)n);
  if (n == 0) return MK_OK;
  for (int64_t k0 = 0; k0 < n; k0 += NB) {
    const int nb = (int)std::min<int64_t>(NB, n - k0);
    hipLaunchKernelGGL(potrf_diag_kernel, dim3(1), dim3(PT), 0, st, A, lda, (int)k0, nb, Linv, info_dev);
    MK_CHECK_HIP(hipGetLastError());
    const int64_t m = n - k0 - nb;
    if (m <= 0) break;
    double* A21 = A + (k0 + nb) + k0 * lda;
    hipLaunchKernelGGL(potrf_panel_kernel, dim3((unsigned)cdiv(m, (int64_t)NB)), dim3(PT), 0, st, A21, lda, m, Linv,
                       info_dev);
    MK_CHECK_HIP(hipGetLastError());
    // A22 -= L21 L21^T (full square; the strict upper part is zeroed at the end)
    ProbSpec p;
    p.M = m; p.N = m;
    p.C = A + (k0 + nb) + (k0 + nb) * lda;
    p.ldc = lda;
    p.alpha = -1.0;
    p.beta = 1.0;
    p.add(A21, lda, A21, lda, nb);
    GemmShape tb;
    tb.tb = true;   // B(k, j) = A21[j + k lda] = L21(j, k)
    MK_TRY(gemm_f64(&p, 1, tb, st, nullptr));
  }
  hipLaunchKernelGGL(zero_upper_kernel, dim3((unsigned)std::min<int64_t>(cdiv(n * n, (int64_t)256), 4096)), dim3(256),
                     0, st, A, lda, n);
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
  double* Linv = nullptr;   // inverted diagonal block
  MK_TRY(carve(ctx, {{(size_t)NB * NB * 8, (void**)&Linv}}));
  MK_CHECK_HIP(hipMemsetAsync(dinfo, 0, sizeof(int), st));
  MK_TRY(potrf_lower(A, n, lda, dinfo, Linv, st));
  MK_CHECK_HIP(hipMemcpyAsync(info, dinfo, sizeof(int), hipMemcpyDeviceToHost, st));
  MK_CHECK_HIP(hipStreamSynchronize(st));
  return MK_OK;
}
