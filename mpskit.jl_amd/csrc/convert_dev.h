// Device helpers shared by the conversion kernels of single applies and of
// grouped (batched) applies.
#pragma once
#include <hip/hip_bf16.h>

#include <cstdint>

#include "gemm.h"

namespace mk {

// bf16 hi/lo split of a float64 value: hi = bf16(v), lo = bf16(v - hi).
__device__ __forceinline__ void split2(double v, __hip_bfloat16& hi, __hip_bfloat16& lo) {
  const float f = (float)v;
  hi = __float2bfloat16(f);
  const double r = v - (double)__bfloat162float(hi);
  lo = __float2bfloat16((float)r);
}

// One pass over x for the mixed-precision Jordan applies with d1 = 2 and D2 = 2
// (two sites) or 1 (one site); x is column-major (Dl, 2, Dr, D2):
//   y = alpha * P(x) + beta * y                       (the physical term; P null: y untouched)
//   xb[(c + Dr j) * kb + r + up8(Dl) h] = conv(x[r,h,c,j])   (x as right factor, K = (h, r))
//   xa[(r + Dl h) * ka + c + up8(Dr) j] = conv(x[r,h,c,j])   (x as left factor, K = (j, c))
// with conv the bf16 hi/lo split (SPLIT) or the fp32 rounding.  Each run of K
// (one h, one j) is padded with zeros to a multiple of 8, so any Dl and Dr do,
// and a GEMM segment may cover one run or several.  A 256-thread
// block owns the (a, c) tile [a0, a0 + 32) x [c0, c0 + PC) and all (h, j)
// sub-tiles of it, so x is read once: the thread holding x[a, :, c, :] produces
// the P outputs of that pair, and the converted values pass through the LDS
// array t (33 KB for PC = 64) for the transposed xa stores.  What follows the last run of a
// row is not written (no K chunk the GEMMs read reaches into it).
constexpr int PRO_A = 32, PRO_C = 64;
template <int PC>
using ProTile = unsigned int[4][PC][PRO_A + 1];

// PACK: the two views are written in the packed panel layout of the 256 x 256
// mixed kernel (packed_offset, with ka = N and kb = M their K lengths; Dl and Dr
// are multiples of 128 then) instead of K-contiguous rows of length ka / kb.
template <bool SPLIT, bool PACK = false, int D2 = 2, int PC = PRO_C>
__device__ __forceinline__ void nn_prologue_tile(const double* __restrict__ P, const double* __restrict__ x,
                                                 int64_t Dl, int64_t Dr, double alpha, double beta,
                                                 double* __restrict__ y, void* __restrict__ xa_hi,
                                                 void* __restrict__ xa_lo, int64_t ka, void* __restrict__ xb_hi,
                                                 void* __restrict__ xb_lo, int64_t kb, int64_t a0, int64_t c0,
                                                 ProTile<PC>& t) {
  // all arrays are in device memory: access them through global-typed pointers
  typedef __attribute__((address_space(1))) double gdouble;
  const gdouble* __restrict__ gx = (const gdouble*)x;
  gdouble* __restrict__ gy = (gdouble*)y;
  typedef __attribute__((address_space(1))) float gf;
  typedef __attribute__((address_space(1))) unsigned short gus;
  typedef __attribute__((address_space(1))) unsigned int gui;
  constexpr int NQ = 2 * D2;
  const int64_t M = 2 * Dl, runl = (Dl + 7) / 8 * 8, runr = (Dr + 7) / 8 * 8;
  double p[NQ * NQ];
  if (P) {
#pragma unroll
    for (int i = 0; i < NQ * NQ; ++i) p[i] = ((const gdouble*)P)[i];
  }
  {
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;   // a offset, c phase (8)
    const int64_t a = a0 + tx;
#pragma unroll
    for (int k = 0; k < PC / 8; ++k) {
      const int cc = ty + 8 * k;
      const int64_t c = c0 + cc;
      if (a < runl && c < Dr) {
        double xv[NQ];
#pragma unroll
        for (int q = 0; q < NQ; ++q) xv[q] = a < Dl ? gx[a + Dl * (q & 1) + M * (c + Dr * (q >> 1))] : 0.0;
        if (P && a < Dl) {
#pragma unroll
          for (int o = 0; o < NQ; ++o) {
            double s = 0.0;
#pragma unroll
            for (int q = 0; q < NQ; ++q) s += p[o + NQ * q] * xv[q];
            // P[b,e,h,j]: (b, e) and (h, j) with the first index fastest, as o and q
            gdouble* yp = gy + a + Dl * (o & 1) + M * (c + Dr * (o >> 1));
            double v = alpha * s;
            if (beta != 0.0) v += beta * *yp;
            *yp = v;
          }
        }
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
          const int64_t rr = a + runl * (q & 1), cl = c + Dr * (q >> 1);
          const int64_t ob = PACK ? packed_offset(cl, rr, kb, SPLIT ? 32 : 16) : cl * kb + rr;
          unsigned int packed;
          if constexpr (SPLIT) {
            __hip_bfloat16 h, l;
            split2(xv[q], h, l);
            ((gus*)xb_hi)[ob] = __builtin_bit_cast(unsigned short, h);
            ((gus*)xb_lo)[ob] = __builtin_bit_cast(unsigned short, l);
            packed = (unsigned int)__builtin_bit_cast(unsigned short, h) |
                     ((unsigned int)__builtin_bit_cast(unsigned short, l) << 16);
          } else {
            const float f = (float)xv[q];
            ((gf*)xb_hi)[ob] = f;
            packed = __float_as_uint(f);
          }
          t[q][cc][tx] = packed;
        }
      }
    }
  }
  __syncthreads();
  {
    constexpr int NA = 256 / PC;                              // a phases
    const int tx = threadIdx.x % PC, ty = threadIdx.x / PC;   // c offset, a phase
    const int64_t c = c0 + tx;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
#pragma unroll
      for (int k = 0; k < PRO_A / NA; ++k) {
        const int aa = ty + NA * k;
        const int64_t ar = a0 + aa;
        if (ar >= Dl || c >= runr) continue;
        const unsigned int v = c < Dr ? t[q][tx][aa] : 0u;
        const int64_t row = ar + Dl * (q & 1), kk = c + runr * (q >> 1);
        const int64_t idx = PACK ? packed_offset(row, kk, ka, SPLIT ? 32 : 16) : row * ka + kk;
        if constexpr (SPLIT) {
          ((gus*)xa_hi)[idx] = (unsigned short)(v & 0xffffu);
          ((gus*)xa_lo)[idx] = (unsigned short)(v >> 16);
        } else {
          ((gui*)xa_hi)[idx] = v;
        }
      }
    }
  }
}

}  // namespace mk
