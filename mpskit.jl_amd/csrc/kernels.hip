// Memory-bound helper kernels; see kernels.h for the contracts.
#include "kernels.h"
#include "convert_dev.h"

#include <hip/hip_bf16.h>

#include <algorithm>

namespace mk {
namespace {

constexpr int TPB = 256;

inline dim3 grid1d(int64_t n, int per_thread = 1) {
  int64_t b = cdiv(n, (int64_t)TPB * per_thread);
  if (b < 1) b = 1;
  if (b > (1 << 30)) b = (1 << 30);
  return dim3((unsigned)b);
}

#define GRID_STRIDE(i, n) \
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < (n); i += (int64_t)gridDim.x * blockDim.x)

__device__ __forceinline__ double env_t(const double* G, int64_t D0, int w, int64_t a, int g,
                                        int64_t f, int ident) {
  // environment with channel `ident` replaced by the identity matrix
  if (g == ident) return a == f ? 1.0 : 0.0;
  return G[a + D0 * (g + (int64_t)w * f)];
}

__global__ void prep_L_kernel(const double* __restrict__ GL, const double* __restrict__ W,
                              const int* __restrict__ klist, int nk, int64_t Da, int64_t Df,
                              int wl, int d, int wr, int g_ident, double* __restrict__ L) {
  const int64_t n = Da * d * Df * d * nk;
  GRID_STRIDE(idx, n) {
    int64_t t = idx;
    const int64_t a = t % Da; t /= Da;
    const int b = (int)(t % d); t /= d;
    const int64_t f = t % Df; t /= Df;
    const int h = (int)(t % d); t /= d;
    const int kk = (int)t;
    const int k = klist[kk];
    double s = 0.0;
    for (int g = 0; g < wl; ++g) {
      const double wv = W[g + wl * (b + d * (h + d * k))];
      if (wv != 0.0) s += env_t(GL, Da, wl, a, g, f, g_ident) * wv;
    }
    L[idx] = s;
  }
}

__global__ void prep_R_kernel(const double* __restrict__ GR, const double* __restrict__ W,
                              const int* __restrict__ klist, int nk, int64_t Di, int64_t Dc,
                              int wl, int d, int wr, int l_ident, double* __restrict__ R) {
  const int64_t n = Di * d * nk * Dc * d;
  GRID_STRIDE(idx, n) {
    int64_t t = idx;
    const int64_t i = t % Di; t /= Di;
    const int j = (int)(t % d); t /= d;
    const int kk = (int)(t % nk); t /= nk;
    const int64_t c = t % Dc; t /= Dc;
    const int e = (int)t;
    const int k = klist[kk];
    double s = 0.0;
    for (int l = 0; l < wr; ++l) {
      const double wv = W[k + wl * (e + d * (j + d * l))];
      if (wv != 0.0) s += wv * env_t(GR, Di, wr, i, l, c, l_ident);
    }
    R[idx] = s;
  }
}

__global__ void prep_Cp_kernel(const double* __restrict__ GR, const double* __restrict__ W,
                               int64_t Di, int64_t Dc, int wl, int d, int wr, int l_ident,
                               double* __restrict__ Cp) {
  const int64_t n = d * Di * d * Dc;
  GRID_STRIDE(idx, n) {
    int64_t t = idx;
    const int h = (int)(t % d); t /= d;
    const int64_t i = t % Di; t /= Di;
    const int b = (int)(t % d); t /= d;
    const int64_t c = t;
    double s = 0.0;
    for (int l = 0; l < wr; ++l) {
      const double wv = W[0 + wl * (b + d * (h + d * l))];
      if (wv != 0.0) s += wv * env_t(GR, Di, wr, i, l, c, l_ident);
    }
    Cp[idx] = s;
  }
}

__global__ void prep_CA_kernel(const double* __restrict__ GR, const double* __restrict__ W1,
                               const double* __restrict__ W2, int64_t Dr, int wl, int d1, int wm,
                               int d2, int wr, int l_ident, double* __restrict__ CA) {
  const int64_t n = (int64_t)d1 * Dr * d2 * d1 * Dr * d2;
  GRID_STRIDE(idx, n) {
    int64_t t = idx;
    const int h = (int)(t % d1); t /= d1;
    const int64_t i = t % Dr; t /= Dr;
    const int j = (int)(t % d2); t /= d2;
    const int b = (int)(t % d1); t /= d1;
    const int64_t c = t % Dr; t /= Dr;
    const int e = (int)t;
    double s = 0.0;
    for (int k = 0; k < wm; ++k) {
      const double w1 = W1[0 + wl * (b + d1 * (h + d1 * k))];
      if (w1 == 0.0) continue;
      double r = 0.0;
      for (int l = 0; l < wr; ++l) {
        const double w2 = W2[k + wm * (e + d2 * (j + d2 * l))];
        if (w2 != 0.0) r += w2 * env_t(GR, Dr, wr, i, l, c, l_ident);
      }
      s += w1 * r;
    }
    CA[idx] = s;
  }
}

__global__ void prep_AB_kernel(const double* __restrict__ GL, const double* __restrict__ W1,
                               const double* __restrict__ W2, int64_t Dl, int wl, int d1, int wm,
                               int d2, int wr, int g_ident, double* __restrict__ AB) {
  const int64_t n = Dl * d1 * Dl * d1 * d2 * d2;
  GRID_STRIDE(idx, n) {
    int64_t t = idx;
    const int64_t a = t % Dl; t /= Dl;
    const int b = (int)(t % d1); t /= d1;
    const int64_t f = t % Dl; t /= Dl;
    const int h = (int)(t % d1); t /= d1;
    const int e = (int)(t % d2); t /= d2;
    const int j = (int)t;
    double s = 0.0;
    for (int k = 0; k < wm; ++k) {
      const double w2 = W2[k + wm * (e + d2 * (j + d2 * (wr - 1)))];
      if (w2 == 0.0) continue;
      double lsum = 0.0;
      for (int g = 0; g < wl; ++g) {
        const double w1 = W1[g + wl * (b + d1 * (h + d1 * k))];
        if (w1 != 0.0) lsum += env_t(GL, Dl, wl, a, g, f, g_ident) * w1;
      }
      s += lsum * w2;
    }
    AB[idx] = s;
  }
}

__global__ void swap23_kernel(const double* __restrict__ in, int64_t D0, int64_t D1, int64_t D2,
                              double* __restrict__ out) {
  const int64_t n = D0 * D1 * D2;
  GRID_STRIDE(idx, n) {
    int64_t t = idx;
    const int64_t a = t % D0; t /= D0;
    const int64_t f = t % D2; t /= D2;
    const int64_t g = t;
    out[idx] = in[a + D0 * (g + D1 * f)];
  }
}

__global__ void env_channels_kernel(const double* __restrict__ src, int64_t Di, int w, int64_t Dc,
                                    const int* __restrict__ klist, int nk, double* __restrict__ dst) {
  const int64_t n = Di * nk * Dc;
  GRID_STRIDE(idx, n) {
    int64_t t = idx;
    const int64_t i = t % Di; t /= Di;
    const int k = (int)(t % nk); t /= nk;
    const int64_t c = t;
    dst[idx] = src[i + Di * (klist[k] + (int64_t)w * c)];
  }
}

__global__ void env_channels_last_kernel(const double* __restrict__ src, int64_t Da, int w, int64_t Df,
                                         const int* __restrict__ klist, int nk, double* __restrict__ dst) {
  const int64_t n = Da * Df * nk;
  GRID_STRIDE(idx, n) {
    const int64_t a = idx % Da, q = idx / Da;
    const int64_t f = q % Df;
    const int k = (int)(q / Df);
    dst[idx] = src[a + Da * (klist[k] + (int64_t)w * f)];
  }
}

// The MPO step of the float64 transfers.  One thread per environment row and
// column (m, c) holds the NIN >= d wl inputs that meet the MPO tensor there in
// registers, so t1 is read and t2 written once (memory-bound: a thread per
// output, which re-read its inputs through the caches and divided the index
// four times, ran at 2.1 TB/s of such traffic at D = 1024, w = 5).  Where the
// threads are few the outputs are dealt out over blockIdx.y: there it is latency
// that bounds it, of an output's MPO entries, which are fetched eight at a time, and
// of the inputs (w = 8, 160 x 171: 22.5 -> 9.0 us).
//   left:  t2[m,k,b,c] = sum_{g,h} t1[m,g,h,c] O[g,k,h,b]
//   right: t2[a,b,k,o] = sum_{h,l} t1[a,h,l,o] O[b,k,h,l]
template <int NIN, bool RIGHT>
__global__ __launch_bounds__(256) void mpo_mid_kernel(const double* __restrict__ t1, const double* __restrict__ O,
                                                      int64_t D1, int wl, int d, int wr, int64_t D2,
                                                      double* __restrict__ t2) {
  typedef __attribute__((address_space(1))) double gd;
  constexpr int OC = 8;
  const int nin = RIGHT ? d * wr : wl * d, nout = RIGHT ? wl * d : d * wr;
  // input i: left (g, h), O step wl d per h; right (h, l), O step wl d per h, wl d d per l
  int off[(NIN + OC - 1) / OC * OC];
#pragma unroll
  for (int i = 0; i < (NIN + OC - 1) / OC * OC; ++i) {
    const int e = min(i, nin - 1);
    off[i] = RIGHT ? wl * d * e : e % wl + wl * d * (e / wl);
  }
  GRID_STRIDE(idx, D1 * D2) {
    const int64_t c = idx / D1, m = idx - c * D1;
    const gd* in = (const gd*)t1 + m + D1 * (int64_t)nin * c;
    gd* out = (gd*)t2 + m + D1 * (int64_t)nout * c;
    double v[NIN];
#pragma unroll
    for (int i = 0; i < NIN; ++i) v[i] = i < nin ? in[D1 * i] : 0.0;
    for (int q = blockIdx.y; q < nout; q += gridDim.y) {
      // output q: left (k, b) = (q % d, q / d), right (b, k) = (q % wl, q / wl)
      const double* w = RIGHT ? O + q % wl + wl * (q / wl) : O + wl * (q % d + d * d * (int64_t)(q / d));
      double s = 0.0;
#pragma unroll
      for (int i0 = 0; i0 < NIN; i0 += OC) {
        double ov[OC];
#pragma unroll
        for (int i = 0; i < OC; ++i) ov[i] = i0 + i < NIN ? w[off[i0 + i]] : 0.0;
#pragma unroll
        for (int i = 0; i < OC; ++i)
          if (i0 + i < NIN && i0 + i < nin && ov[i] != 0.0) s += v[i0 + i] * ov[i];
      }
      out[D1 * q] = s;
    }
  }
}

// The same with any number of inputs (a thread per output).
template <bool RIGHT>
__global__ void mpo_mid_wide_kernel(const double* __restrict__ t1, const double* __restrict__ O, int64_t D1, int wl,
                                    int d, int wr, int64_t D2, double* __restrict__ t2) {
  const int nin = RIGHT ? d * wr : wl * d, nout = RIGHT ? wl * d : d * wr;
  GRID_STRIDE(idx, D1 * nout * D2) {
    int64_t t = idx;
    const int64_t m = t % D1; t /= D1;
    const int q = (int)(t % nout);
    const int64_t c = t / nout;
    const double* w = RIGHT ? O + q % wl + wl * (q / wl) : O + wl * (q % d + d * d * (int64_t)(q / d));
    double s = 0.0;
    if constexpr (RIGHT) {
      for (int i = 0; i < nin; ++i) {
        const double ov = w[(int64_t)wl * d * i];
        if (ov != 0.0) s += t1[m + D1 * (i + (int64_t)nin * c)] * ov;
      }
    } else {
      // by (h, g): with the index of an input divided by wl instead, the left transfer
      // with w = 17 at D = 128 takes 106 us, so 86
      const double* in = t1 + m + D1 * ((int64_t)nin * c);
      for (int h = 0; h < d; ++h, w += (int64_t)wl * d)
        for (int g = 0; g < wl; ++g, in += D1) {
          const double ov = w[g];
          if (ov != 0.0) s += *in * ov;
        }
    }
    t2[idx] = s;
  }
}

// out[a,q,p,b] = in[a,p,q,b]: the two middle legs of a column-major
// n0 x n1 x n2 x n3 tensor exchanged (reads and writes run along a).
__global__ void swap_mid_kernel(const double* __restrict__ in, int64_t n0, int64_t n1, int64_t n2, int64_t n3,
                                double* __restrict__ out) {
  const int64_t n = n0 * n1 * n2 * n3;
  GRID_STRIDE(idx, n) {
    int64_t t = idx;
    const int64_t a = t % n0; t /= n0;
    const int64_t q = t % n2; t /= n2;
    const int64_t p = t % n1;
    const int64_t b = t / n1;
    out[idx] = in[a + n0 * (p + n1 * (q + n2 * b))];
  }
}

// An MPO tensor widened by identities on a virtual and a physical passenger
// leg: out[(w,e),(k,q),(h,r),(v,f)] = O[w,k,h,v] delta(e,f) delta(q,r) with
// the fused indices w + wl e, k + d q (column-major fusion of the legs).
// O == nullptr stands for the identity MPO O[w,k,h,v] = delta(w,v) delta(k,h)
// (wl == wr).
__global__ void mpo_extend_kernel(const double* __restrict__ O, int wl, int d, int wr, int ne, int nq,
                                  double* __restrict__ out) {
  const int64_t WL = (int64_t)wl * ne, DQ = (int64_t)d * nq, WR = (int64_t)wr * ne;
  const int64_t n = WL * DQ * DQ * WR;
  GRID_STRIDE(idx, n) {
    int64_t t = idx;
    const int i0 = (int)(t % WL); t /= WL;
    const int i1 = (int)(t % DQ); t /= DQ;
    const int i2 = (int)(t % DQ);
    const int i3 = (int)(t / DQ);
    const int w = i0 % wl, e = i0 / wl, k = i1 % d, q = i1 / d;
    const int h = i2 % d, r = i2 / d, v = i3 % wr, f = i3 / wr;
    double val = 0.0;
    if (e == f && q == r)
      val = O ? O[w + (int64_t)wl * (k + (int64_t)d * (h + (int64_t)d * v))] : (w == v && k == h ? 1.0 : 0.0);
    out[idx] = val;
  }
}

// The MPO step of the left transfer written straight into the K-contiguous
// mixed-precision operand of the second GEMM (one pass instead of a float64
// round trip and a conversion):
//   t2[(m,k),(b,c)] = sum_{g,h} t1[m + Dm (g + wl (h + d c))] O[g + wl (k + d (h + d b))]
// stored out[(b + wr c) * ldo + m + Dm k], zero for Dm d <= kk < ldo.
template <bool SPLIT>
__global__ void tl_mid_mixed_kernel(const double* __restrict__ t1, const double* __restrict__ O, int64_t Dm,
                                    int wl, int d, int wr, int64_t Dc, int64_t ldo, void* __restrict__ hi,
                                    void* __restrict__ lo) {
  const int64_t n = ldo * wr * Dc, K = Dm * d;
  GRID_STRIDE(idx, n) {
    const int64_t kk = idx % ldo, col = idx / ldo;
    const int b = (int)(col % wr);
    const int64_t c = col / wr;
    double s = 0.0;
    if (kk < K) {
      const int64_t m = kk % Dm;
      const int k = (int)(kk / Dm);
      for (int h = 0; h < d; ++h)
        for (int g = 0; g < wl; ++g) {
          const double ov = O[g + wl * (k + d * (h + d * b))];
          if (ov != 0.0) s += t1[m + Dm * (g + (int64_t)wl * (h + d * c))] * ov;
        }
    }
    if constexpr (SPLIT) {
      __hip_bfloat16 h, l;
      split2(s, h, l);
      static_cast<__hip_bfloat16*>(hi)[idx] = h;
      static_cast<__hip_bfloat16*>(lo)[idx] = l;
    } else {
      static_cast<float*>(hi)[idx] = (float)s;
    }
  }
}

// The MPO step of the right transfer written straight into the K-contiguous
// mixed-precision left operand of the second GEMM (64 x 64 LDS transpose tiles:
// reads run along a, writes along (k, o)):
//   t2[(a,b),(k,o)] = sum_{l,h} t1[a + Da (h + d (l + wr o))] O[b + wl (k + d (h + d l))]
// stored out[(a + Da b) * ldo + k + d o], zero for d Do <= kk < ldo.
template <bool SPLIT>
__global__ __launch_bounds__(256) void tr_mid_mixed_kernel(const double* __restrict__ t1,
                                                           const double* __restrict__ O, int64_t Da, int wl, int d,
                                                           int wr, int64_t Do, int64_t ldo, void* __restrict__ hi,
                                                           void* __restrict__ lo) {
  __shared__ double tile[64][65];
  const int64_t rows = Da * wl, K = (int64_t)d * Do;
  const int64_t r0 = (int64_t)blockIdx.x * 64, c0 = (int64_t)blockIdx.y * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  for (int cc = ty; cc < 64; cc += 4) {
    const int64_t r = r0 + tx, kk = c0 + cc;
    double s = 0.0;
    if (r < rows && kk < K) {
      const int64_t a = r % Da;
      const int b = (int)(r / Da);
      const int k = (int)(kk % d);
      const int64_t o = kk / d;
      for (int l = 0; l < wr; ++l)
        for (int h = 0; h < d; ++h) {
          const double ov = O[b + wl * (k + d * (h + d * l))];
          if (ov != 0.0) s += t1[a + Da * (h + d * (l + (int64_t)wr * o))] * ov;
        }
    }
    tile[cc][tx] = s;
  }
  __syncthreads();
  for (int rr = ty; rr < 64; rr += 4) {
    const int64_t r = r0 + rr, kk = c0 + tx;
    if (r < rows && kk < ldo) {
      const double v = tile[tx][rr];
      if constexpr (SPLIT) {
        __hip_bfloat16 h, l;
        split2(v, h, l);
        static_cast<__hip_bfloat16*>(hi)[r * ldo + kk] = h;
        static_cast<__hip_bfloat16*>(lo)[r * ldo + kk] = l;
      } else {
        static_cast<float*>(hi)[r * ldo + kk] = (float)v;
      }
    }
  }
}

__global__ void phys2_kernel(const double* __restrict__ P, const double* __restrict__ x, int64_t Dl,
                             int d1, int64_t Dr, int d2, double alpha, double beta,
                             double* __restrict__ y) {
  const int64_t n = Dl * d1 * Dr * d2;
  GRID_STRIDE(idx, n) {
    int64_t t = idx;
    const int64_t a = t % Dl; t /= Dl;
    const int b = (int)(t % d1); t /= d1;
    const int64_t c = t % Dr; t /= Dr;
    const int e = (int)t;
    double s = 0.0;
    for (int j = 0; j < d2; ++j)
      for (int h = 0; h < d1; ++h)
        s += P[b + d1 * (e + d2 * (h + d1 * j))] * x[a + Dl * (h + d1 * (c + Dr * j))];
    double v = alpha * s;
    if (beta != 0.0) v += beta * y[idx];
    y[idx] = v;
  }
}

// Same contraction with one thread per (a, c): the d1*d2 inputs x[a,:,c,:] are
// read once into registers and all d1*d2 outputs y[a,:,c,:] written from them,
// so x is read once and y written once (loads and stores coalesced along a).
template <int D12>
__global__ void phys2_reg_kernel(const double* __restrict__ P, const double* __restrict__ x, int64_t Dl,
                                 int d1, int64_t Dr, int d2, double alpha, double beta,
                                 double* __restrict__ y) {
  const int64_t n = Dl * Dr;
  const int64_t sx = Dl * d1 * Dr;   // stride of the second physical leg
  GRID_STRIDE(idx, n) {
    const int64_t a = idx % Dl, c = idx / Dl;
    const int64_t base = a + Dl * d1 * c;
    double xv[D12];
#pragma unroll
    for (int t = 0; t < D12; ++t) {
      const int h = t % d1, j = t / d1;
      xv[t] = x[base + Dl * h + sx * j];
    }
#pragma unroll
    for (int o = 0; o < D12; ++o) {
      const int b = o % d1, e = o / d1;
      double s = 0.0;
#pragma unroll
      for (int t = 0; t < D12; ++t) s += P[b + d1 * (e + d2 * t)] * xv[t];
      double* yp = y + base + Dl * b + sx * e;
      double v = alpha * s;
      if (beta != 0.0) v += beta * *yp;
      *yp = v;
    }
  }
}

// Diagonal of the nearest-neighbour two-site Jordan operator x*IC + BE*x + CB(x):
// diag[row + M col] = IC[col, col] + BE[row, row] + CB[b, e, b, e], row = a + Dl b,
// col = c + Dr e (absent terms are null).
__global__ void diag_nn_kernel(const double* __restrict__ IC, const double* __restrict__ BE,
                               const double* __restrict__ P, int64_t Dl, int64_t Dr, int d1, int d2,
                               double* __restrict__ out) {
  const int64_t M = Dl * d1, N = Dr * d2;
  GRID_STRIDE(idx, M * N) {
    const int64_t row = idx % M, col = idx / M;
    double v = 0.0;
    if (IC) v += IC[col + N * col];
    if (BE) v += BE[row + M * row];
    if (P) {
      const int b = (int)(row / Dl), e = (int)(col / Dr);
      v += P[b + d1 * (e + d2 * (b + d1 * e))];
    }
    out[idx] = v;
  }
}

__global__ void phys1_kernel(const double* __restrict__ P, const double* __restrict__ x, int64_t Dl,
                             int d, int64_t Dr, double alpha, double beta, double* __restrict__ y) {
  const int64_t n = Dl * d * Dr;
  GRID_STRIDE(idx, n) {
    int64_t t = idx;
    const int64_t a = t % Dl; t /= Dl;
    const int b = (int)(t % d); t /= d;
    const int64_t c = t;
    double s = 0.0;
    for (int h = 0; h < d; ++h) s += P[b + d * h] * x[a + Dl * (h + (int64_t)d * c)];
    double v = alpha * s;
    if (beta != 0.0) v += beta * y[idx];
    y[idx] = v;
  }
}

// ---- reductions -------------------------------------------------------------

__device__ __forceinline__ double block_sum(double v, double* sh) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) sh[wid] = v;
  __syncthreads();
  double r = 0.0;
  if (threadIdx.x == 0) {
    for (int i = 0; i < (int)(blockDim.x >> 6); ++i) r += sh[i];
  }
  __syncthreads();
  return r;  // valid in thread 0
}

// lam[g] = sum_{i<D2, j<D1} lvec[i + D2*j] * v[j + D1*(g + w*i)]
__global__ void reg_lambda_kernel(const double* __restrict__ v, const double* __restrict__ lvec,
                                  int64_t D1, int w, int64_t D2, double* __restrict__ lam) {
  __shared__ double sh[TPB / 64];
  const int g = blockIdx.x;
  double s = 0.0;
  const int64_t n = D1 * D2;
  for (int64_t idx = threadIdx.x; idx < n; idx += blockDim.x) {
    const int64_t j = idx % D1, i = idx / D1;
    s += lvec[i + D2 * j] * v[j + D1 * (g + (int64_t)w * i)];
  }
  s = block_sum(s, sh);
  if (threadIdx.x == 0) lam[g] = s;
}

__global__ void reg_apply_kernel(double* __restrict__ v, const double* __restrict__ rvec,
                                 const double* __restrict__ lam, int64_t D1, int w, int64_t D2) {
  const int64_t n = D1 * w * D2;
  GRID_STRIDE(idx, n) {
    int64_t t = idx;
    const int64_t a = t % D1; t /= D1;
    const int g = (int)(t % w); t /= w;
    const int64_t c = t;
    v[idx] -= lam[g] * rvec[a + D1 * c];
  }
}

constexpr int MD_ITEMS = 16;  // elements of w held per thread in multidot

__global__ void multidot_kernel(const double* __restrict__ V, int64_t ldv, int k,
                                const double* __restrict__ w, int64_t n, double* __restrict__ partial) {
  __shared__ double sh[TPB / 64];
  const int64_t base = (int64_t)blockIdx.x * TPB * MD_ITEMS;
  double wr[MD_ITEMS];
#pragma unroll
  for (int it = 0; it < MD_ITEMS; ++it) {
    const int64_t i = base + it * TPB + threadIdx.x;
    wr[it] = i < n ? w[i] : 0.0;
  }
  for (int j = 0; j < k; ++j) {
    const double* Vj = V + (int64_t)j * ldv;
    double s = 0.0;
#pragma unroll
    for (int it = 0; it < MD_ITEMS; ++it) {
      const int64_t i = base + it * TPB + threadIdx.x;
      if (i < n) s += Vj[i] * wr[it];
    }
    s = block_sum(s, sh);
    if (threadIdx.x == 0) partial[(int64_t)j * gridDim.x + blockIdx.x] = s;
  }
}

__global__ void reduce_rows_kernel(const double* __restrict__ partial, int nb, double* __restrict__ out) {
  __shared__ double sh[TPB / 64];
  const int j = blockIdx.x;
  double s = 0.0;
  for (int b = threadIdx.x; b < nb; b += blockDim.x) s += partial[(int64_t)j * nb + b];
  s = block_sum(s, sh);
  if (threadIdx.x == 0) out[j] = s;
}

// Fused classical Gram-Schmidt update: u <- u - V c (c = cin[0..k)) and, with
// the updated u, the partial sums of V^T u (MODE 0, k outputs) or of u^T u and
// w^T u (MODE 1, 2 outputs).  Each thread keeps its row of V in registers
// between the update and the dot products, so V is read once for both.
// k <= CGS_KMAX; partial sums go to partial[o * gridDim.x + blockIdx.x].
// KT (4, 8, 16 or 32 >= k) sizes the register arrays: the rows of V held per
// thread, and the accumulators, scale with the basis, so small bases keep
// the occupancy (and the memory parallelism) high.  MODE 2: no update, the
// partial sums of V^T u only (the first Gram-Schmidt pass).
constexpr int CGS_KMAX = 32;
template <int MODE, int KT, typename VT>
__global__ __launch_bounds__(TPB) void cgs_update_kernel(const VT* __restrict__ V, int64_t ldv, int k,
                                                         const double* __restrict__ cin, int lo, double* __restrict__ u,
                                                         const double* __restrict__ w, int64_t n,
                                                         double* __restrict__ partial) {
  __shared__ double sh[TPB / 64];
  constexpr int NO = MODE == 1 ? 2 : KT;
  double c[KT], acc[NO];
#pragma unroll
  for (int j = 0; j < KT; ++j) c[j] = (MODE != 2 && j >= lo && j < k) ? cin[j] : 0.0;
#pragma unroll
  for (int o = 0; o < NO; ++o) acc[o] = 0.0;
  GRID_STRIDE(r, n) {
    double q[KT];
#pragma unroll
    for (int j = 0; j < KT; ++j) q[j] = j < k ? (double)V[r + (int64_t)j * ldv] : 0.0;
    double v = u[r];
    if constexpr (MODE != 2) {
#pragma unroll
      for (int j = 0; j < KT; ++j) v -= c[j] * q[j];
      u[r] = v;
    }
    if constexpr (MODE != 1) {
#pragma unroll
      for (int j = 0; j < KT; ++j) acc[j] += q[j] * v;
    } else {
      acc[0] += v * v;
      acc[1] += w[r] * v;
    }
  }
  const int nout = MODE == 1 ? 2 : k;
#pragma unroll
  for (int o = 0; o < NO; ++o) {
    if (o >= nout) break;
    const double t = block_sum(acc[o], sh);
    if (threadIdx.x == 0) partial[(int64_t)o * gridDim.x + blockIdx.x] = t;
  }
}

__global__ void multiaxpy_kernel(const double* __restrict__ V, int64_t ldv, int k,
                                 const double* __restrict__ c, double* __restrict__ w, int64_t n) {
  GRID_STRIDE(i, n) {
    double s = w[i];
    for (int j = 0; j < k; ++j) s -= c[j] * V[i + (int64_t)j * ldv];
    w[i] = s;
  }
}

__global__ void gemv_kernel(const double* __restrict__ V, int64_t ldv, int k,
                            const double* __restrict__ s, double* __restrict__ x, int64_t n) {
  GRID_STRIDE(i, n) {
    double acc = 0.0;
    for (int j = 0; j < k; ++j) acc += s[j] * V[i + (int64_t)j * ldv];
    x[i] = acc;
  }
}

// a = 0 or b = 0: that operand is not read (y may hold anything before its first write)
__global__ void axpby_kernel(double a, const double* x, double b, double* y,
                             int64_t n) {
  GRID_STRIDE(i, n) {
    double v = a != 0.0 ? a * x[i] : 0.0;
    if (b != 0.0) v += b * y[i];
    y[i] = v;
  }
}

// y = x / sqrt(*s2)
__global__ void normalize_kernel(const double* __restrict__ x, const double* __restrict__ s2, double* __restrict__ y,
                                 int64_t n) {
  const double s = 1.0 / sqrt(*s2);
  GRID_STRIDE(i, n) y[i] = s * x[i];
}

__global__ void scale_dev_kernel(double* __restrict__ y, const double* __restrict__ sdev, int inv,
                                 int64_t n) {
  const double s = inv ? 1.0 / *sdev : *sdev;
  GRID_STRIDE(i, n) y[i] *= s;
}

__global__ void nonfinite_kernel(const double* __restrict__ x, int64_t n, int* flag) {
  int bad = 0;
  GRID_STRIDE(i, n) {
    if (!isfinite(x[i])) bad = 1;
  }
  if (bad) atomicOr(flag, 1);
}

// ---- precision conversion ---------------------------------------------------

// Eight consecutive elements of a converted row: bf16 hi and lo (SPLIT) or fp32.
template <bool SPLIT>
__device__ __forceinline__ void put8(const double (&v)[8], void* __restrict__ hi, void* __restrict__ lo, int64_t at) {
  typedef unsigned int u4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(1))) u4 gu4;
  if constexpr (SPLIT) {
    u4 a, b;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      __hip_bfloat16 h0, l0, h1, l1;
      split2(v[2 * q], h0, l0);
      split2(v[2 * q + 1], h1, l1);
      a[q] = (unsigned)__builtin_bit_cast(unsigned short, h0) | ((unsigned)__builtin_bit_cast(unsigned short, h1) << 16);
      b[q] = (unsigned)__builtin_bit_cast(unsigned short, l0) | ((unsigned)__builtin_bit_cast(unsigned short, l1) << 16);
    }
    *(gu4*)((char*)hi + at * 2) = a;
    *(gu4*)((char*)lo + at * 2) = b;
  } else {
    u4 a, b;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      a[q] = __float_as_uint((float)v[q]);
      b[q] = __float_as_uint((float)v[4 + q]);
    }
    *(gu4*)((char*)hi + at * 4) = a;
    *(gu4*)((char*)hi + at * 4 + 16) = b;
  }
}

// Conversions of a float64 matrix into K-contiguous rows of length ldo (a
// multiple of 8).  K may come in `nrun` runs of `run` source elements, each
// padded with zeros to `runpad` (a multiple of 8); what is left of the row is
// zero.  Both are memory-bound: a thread converts 8 elements of a row and
// writes them as 16-byte stores (2-byte stores, one element a thread, ran at
// 1.4 TB/s on a 2048 x 1024 matrix).
//
// plain (K = rows): out[c * ldo + k] = M[r + c * ld]
template <bool SPLIT>
__global__ void conv_plain_kernel(const double* __restrict__ M, int64_t run, int nrun, int64_t runpad, int64_t cols,
                                  int64_t ld, int64_t ldo, void* __restrict__ hi, void* __restrict__ lo) {
  const int64_t nch = ldo / 8, n = nch * cols;
  typedef const __attribute__((address_space(1))) double gd;
  GRID_STRIDE(idx, n) {
    const int64_t c = idx / nch, k = (idx - c * nch) * 8;
    const int64_t q = k / runpad, o = k - q * runpad;
    double v[8];
    gd* p = (gd*)M + c * ld + q * run + o;
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = (q < nrun && o + i < run) ? p[i] : 0.0;
    put8<SPLIT>(v, hi, lo, c * ldo + k);
  }
}

// transposed (K = cols): out[r * ldo + k] = M[r + c * ld], 64 x 64 LDS tiles
template <bool SPLIT>
__global__ __launch_bounds__(256) void conv_trans_kernel(const double* __restrict__ M, int64_t rows, int64_t run,
                                                         int nrun, int64_t runpad, int64_t ld, int64_t ldo,
                                                         void* __restrict__ hi, void* __restrict__ lo) {
  __shared__ double tile[64][65];
  const int64_t r0 = (int64_t)blockIdx.x * 64, k0 = (int64_t)blockIdx.y * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;  // 4 rows of threads
  typedef const __attribute__((address_space(1))) double gd;
#pragma unroll 4
  for (int cc = ty; cc < 64; cc += 4) {
    const int64_t r = r0 + tx, k = k0 + cc;
    const int64_t q = k / runpad, o = k - q * runpad;
    tile[cc][tx] = (r < rows && q < nrun && o < run) ? ((gd*)M)[r + (q * run + o) * ld] : 0.0;
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int id = threadIdx.x + it * 256, rr = id >> 3, q8 = (id & 7) * 8;
    const int64_t r = r0 + rr, k = k0 + q8;
    if (r < rows && k < ldo) {
      double v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = tile[q8 + i][rr];
      put8<SPLIT>(v, hi, lo, r * ldo + k);
    }
  }
}

// The middle step of a generic operator's apply, between x GR and GL:
//   t2[f,g,b,c,e] = sum_{h,l,j} Wc[(g,b,e)][(h,l,j)] t1[f,h,l,c,j]
// One thread per (f, c) holds its NIN >= d1 wr d2 inputs in registers, so t1
// is read once and t2 written once (memory-bound); Wc is uniform over the
// threads and zero-padded to NIN columns.  Each thread writes only the places
// it has read, so with wl == wr t2 may be t1 itself.  MODE 0: float64 t2; 1,
// 2: the K-contiguous rows (b,c,e) of length ldo of the next product's right
// factor, K = (f, g), as bf16 hi and lo or fp32, zero from K to the next
// multiple of 8.
template <int NIN, int MODE>
__global__ __launch_bounds__(256) void gen_mid_kernel(const double* t1, const double* __restrict__ Wc, int64_t Df,
                                                      int wl, int d1, int wr, int d2, int64_t nc, double* t2,
                                                      int64_t ldo, void* __restrict__ hi, void* __restrict__ lo) {
  const int nin1 = d1 * wr, nout1 = wl * d1;
  const int64_t n = Df * nc, K = Df * wl, pad = (K + 7) / 8 * 8 - K;
  GRID_STRIDE(idx, n) {
    const int64_t c = idx / Df, f = idx - c * Df;
    double v[NIN];
#pragma unroll
    for (int i = 0; i < NIN; ++i) {
      const int q = i % nin1, j = i / nin1;
      v[i] = j < d2 ? t1[f + Df * (q + (int64_t)nin1 * (c + nc * j))] : 0.0;
    }
    for (int e = 0; e < d2; ++e)
      for (int b = 0; b < d1; ++b) {
        const int64_t row = b + d1 * (c + nc * e);
        for (int g = 0; g < wl; ++g) {
          const double* w = Wc + (int64_t)(g + wl * (b + d1 * e)) * NIN;
          double s = 0.0;
#pragma unroll
          for (int i = 0; i < NIN; ++i) s += w[i] * v[i];
          if constexpr (MODE == 0) {
            t2[f + Df * (g + (int64_t)nout1 * (c + nc * e) + (int64_t)wl * b)] = s;
          } else if constexpr (MODE == 1) {
            __hip_bfloat16 h, l;
            split2(s, h, l);
            static_cast<__hip_bfloat16*>(hi)[row * ldo + f + Df * g] = h;
            static_cast<__hip_bfloat16*>(lo)[row * ldo + f + Df * g] = l;
          } else {
            static_cast<float*>(hi)[row * ldo + f + Df * g] = (float)s;
          }
        }
        if (MODE != 0) {
          for (int64_t z = f; z < pad; z += Df) {
            if constexpr (MODE == 1) {
              static_cast<__hip_bfloat16*>(hi)[row * ldo + K + z] = __float2bfloat16(0.f);
              static_cast<__hip_bfloat16*>(lo)[row * ldo + K + z] = __float2bfloat16(0.f);
            } else {
              static_cast<float*>(hi)[row * ldo + K + z] = 0.f;
            }
          }
        }
      }
  }
}

template <bool SPLIT, bool PACK, int D2, int PC>
__global__ __launch_bounds__(256) void nn_prologue_kernel(const double* __restrict__ P,
                                                          const double* __restrict__ x, int64_t Dl, int64_t Dr,
                                                          double alpha, double beta, double* __restrict__ y,
                                                          void* __restrict__ xa_hi, void* __restrict__ xa_lo,
                                                          int64_t ka, void* __restrict__ xb_hi,
                                                          void* __restrict__ xb_lo, int64_t kb) {
  __shared__ ProTile<PC> t;
  nn_prologue_tile<SPLIT, PACK, D2, PC>(P, x, Dl, Dr, alpha, beta, y, xa_hi, xa_lo, ka, xb_hi, xb_lo, kb,
                                        (int64_t)blockIdx.x * PRO_A, (int64_t)blockIdx.y * PC, t);
}

// D x D operator blocks as combinations of environment levels:
//   right (LEFT = false): out[i + D (c + D q)]      = sum_l coef[q w + l] E[i + D (l + w c)]
//   left  (LEFT = true):  out[a + D q + D nq f]     = sum_g coef[q w + g] E[a + D (g + w f)]
// One thread per (row, column) writes all nq blocks and reads every level once:
// memory-bound in its w reads and nq writes per element.
template <bool LEFT>
__global__ __launch_bounds__(256) void env_blocks_kernel(const double* __restrict__ E, const double* __restrict__ coef,
                                                         int64_t D, int w, int nq, double* __restrict__ out) {
  typedef __attribute__((address_space(1))) double gd;
  GRID_STRIDE(idx, D * D) {
    const int64_t c = idx / D, r = idx - c * D;
    const gd* e = (const gd*)E + r + D * (int64_t)w * c;
    for (int q0 = 0; q0 < nq; q0 += 4) {
      double s[4] = {0.0, 0.0, 0.0, 0.0};
      for (int l = 0; l < w; ++l) {
        const double v = e[D * l];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const double k = q0 + q < nq ? coef[(int64_t)(q0 + q) * w + l] : 0.0;
          if (k != 0.0) s[q] += k * v;
        }
      }
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (q0 + q < nq) ((gd*)out)[LEFT ? r + D * (q0 + q) + D * nq * c : r + D * (c + D * (int64_t)(q0 + q))] = s[q];
    }
  }
}

// Packed panel layout from K-contiguous rows (row length kpad >= K, element
// size eb): one 16-byte chunk per thread.
__global__ void repack_kernel(const char* __restrict__ in, int64_t MN, int64_t K, int64_t kpad, int eb,
                              char* __restrict__ out) {
  typedef unsigned int u4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(1))) u4 gu4;
  const int64_t steps = K * eb / 64;
  GRID_STRIDE(o, MN * K * eb / 16) {
    const int64_t slab = o / 1024, r = (o % 1024) / 4, q = o % 4;
    const int64_t row = (slab / steps) * 256 + r, kbyte = (slab % steps) * 64 + q * 16;
    ((gu4*)out)[o] = ((const gu4*)(in + row * kpad * eb + kbyte))[0];
  }
}

// ---- Jordan operator matrices from constructed terms (prepare_operator!! folds)
// Absent terms are null pointers; flags say which optional terms a target takes.

__global__ void asm_ic_kernel(const double* __restrict__ IC, const double* __restrict__ ID,
                              const double* __restrict__ II, int64_t Dr, int d2, double* __restrict__ out) {
  const int64_t N = Dr * d2;
  GRID_STRIDE(idx, N * N) {
    const int64_t row = idx % N, col = idx / N;
    const int64_t i = row % Dr, c = col % Dr;
    const int j = (int)(row / Dr), e = (int)(col / Dr);
    double v = IC ? IC[e + d2 * (c + Dr * (j + d2 * i))] : 0.0;
    if (ID && c == i) v += ID[e + d2 * j];
    if (II && e == j) v += II[c + Dr * i];
    out[idx] = v;
  }
}

__global__ void asm_be_kernel(const double* __restrict__ BE, const double* __restrict__ DE,
                              const double* __restrict__ EE, int64_t Dl, int d1, double* __restrict__ out) {
  const int64_t M = Dl * d1;
  GRID_STRIDE(idx, M * M) {
    const int64_t row = idx % M, col = idx / M;
    const int64_t a = row % Dl, f = col % Dl;
    const int b = (int)(row / Dl), h = (int)(col / Dl);
    double v = BE ? BE[idx] : 0.0;
    if (DE && a == f) v += DE[b + d1 * h];
    if (EE && b == h) v += EE[a + Dl * f];
    out[idx] = v;
  }
}

__global__ void asm_ca_kernel(const double* __restrict__ CA, const double* __restrict__ CB,
                              const double* __restrict__ IC, const double* __restrict__ ID,
                              const double* __restrict__ II, int64_t Dr, int d1, int d2, double* __restrict__ out) {
  const int64_t N = Dr * d2, R = d1 * N;
  GRID_STRIDE(idx, R * R) {
    int64_t t = idx % R;
    const int h = (int)(t % d1); t /= d1;
    const int64_t i = t % Dr;
    const int j = (int)(t / Dr);
    t = idx / R;
    const int b = (int)(t % d1); t /= d1;
    const int64_t c = t % Dr;
    const int e = (int)(t / Dr);
    double v = CA[b + d1 * (e + d2 * (c + Dr * (h + d1 * (j + d2 * i))))];
    if (CB && c == i) v += CB[b + d1 * (e + d2 * (h + d1 * j))];
    if (b == h) {
      if (IC) v += IC[e + d2 * (c + Dr * (j + d2 * i))];
      if (ID && c == i) v += ID[e + d2 * j];
      if (II && e == j) v += II[c + Dr * i];
    }
    out[idx] = v;
  }
}

__global__ void asm_ab_kernel(const double* __restrict__ AB, const double* __restrict__ CB,
                              const double* __restrict__ BE, const double* __restrict__ DE,
                              const double* __restrict__ EE, int64_t Dl, int d1, int d2, double* __restrict__ out) {
  const int64_t M = Dl * d1, MM = M * M;
  GRID_STRIDE(idx, MM * d2 * d2) {
    const int64_t blk = idx / MM, w = idx % MM;
    const int e = (int)(blk % d2), j = (int)(blk / d2);
    const int64_t row = w % M, col = w / M;
    const int64_t a = row % Dl, f = col % Dl;
    const int b = (int)(row / Dl), h = (int)(col / Dl);
    double v = AB[a + Dl * (b + d1 * (e + d2 * (f + Dl * (h + d1 * (int64_t)j))))];
    if (CB && a == f) v += CB[b + d1 * (e + d2 * (h + d1 * j))];
    if (e == j) {
      if (BE) v += BE[w];
      if (DE && a == f) v += DE[b + d1 * h];
      if (EE && b == h) v += EE[a + Dl * f];
    }
    out[idx] = v;
  }
}

__global__ void asm_cp_kernel(const double* __restrict__ C, const double* __restrict__ D,
                              const double* __restrict__ I, int64_t Dr, int d, double* __restrict__ out) {
  const int64_t N = Dr * d;
  GRID_STRIDE(idx, N * N) {
    const int64_t row = idx % N, col = idx / N;
    const int h = (int)(row % d), b = (int)(col % d);
    const int64_t i = row / d, c = col / d;
    double v = C ? C[b + d * (c + Dr * (h + d * i))] : 0.0;
    if (D && i == c) v += D[b + d * h];
    if (I && b == h) v += I[i + Dr * c];
    out[idx] = v;
  }
}

}  // namespace

#define LAUNCH_1D(kern, n, st, ...)                                          \
  do {                                                                        \
    if ((n) > 0) {                                                            \
      hipLaunchKernelGGL(kern, grid1d(n, 4), dim3(TPB), 0, st, __VA_ARGS__);  \
      MK_CHECK_HIP(hipGetLastError());                                        \
    }                                                                         \
    return MK_OK;                                                             \
  } while (0)

mk_status k_prep_L(const double* GL, const double* W, const int* klist, int nk, int64_t Da,
                   int64_t Df, int wl, int d, int wr, int g_ident, double* L, hipStream_t st) {
  LAUNCH_1D(prep_L_kernel, Da * d * Df * d * nk, st, GL, W, klist, nk, Da, Df, wl, d, wr, g_ident, L);
}
mk_status k_prep_R(const double* GR, const double* W, const int* klist, int nk, int64_t Di,
                   int64_t Dc, int wl, int d, int wr, int l_ident, double* R, hipStream_t st) {
  LAUNCH_1D(prep_R_kernel, Di * d * nk * Dc * d, st, GR, W, klist, nk, Di, Dc, wl, d, wr, l_ident, R);
}
mk_status k_prep_Cp(const double* GR, const double* W, int64_t Di, int64_t Dc, int wl, int d,
                    int wr, int l_ident, double* Cp, hipStream_t st) {
  LAUNCH_1D(prep_Cp_kernel, (int64_t)d * Di * d * Dc, st, GR, W, Di, Dc, wl, d, wr, l_ident, Cp);
}
mk_status k_prep_CA(const double* GR, const double* W1, const double* W2, int64_t Dr, int wl,
                    int d1, int wm, int d2, int wr, int l_ident, double* CA, hipStream_t st) {
  LAUNCH_1D(prep_CA_kernel, (int64_t)d1 * Dr * d2 * d1 * Dr * d2, st, GR, W1, W2, Dr, wl, d1, wm, d2,
            wr, l_ident, CA);
}
mk_status k_prep_AB(const double* GL, const double* W1, const double* W2, int64_t Dl, int wl,
                    int d1, int wm, int d2, int wr, int g_ident, double* AB, hipStream_t st) {
  LAUNCH_1D(prep_AB_kernel, Dl * d1 * Dl * d1 * d2 * d2, st, GL, W1, W2, Dl, wl, d1, wm, d2, wr,
            g_ident, AB);
}
mk_status k_swap23(const double* in, int64_t D0, int64_t D1, int64_t D2, double* out, hipStream_t st) {
  LAUNCH_1D(swap23_kernel, D0 * D1 * D2, st, in, D0, D1, D2, out);
}
mk_status k_env_channels(const double* src, int64_t Di, int w, int64_t Dc, const int* klist, int nk,
                         double* dst, hipStream_t st) {
  LAUNCH_1D(env_channels_kernel, Di * nk * Dc, st, src, Di, w, Dc, klist, nk, dst);
}
mk_status k_env_channels_last(const double* src, int64_t Da, int w, int64_t Df, const int* klist, int nk, double* dst,
                              hipStream_t st) {
  LAUNCH_1D(env_channels_last_kernel, Da * Df * nk, st, src, Da, w, Df, klist, nk, dst);
}
template <bool RIGHT>
static mk_status launch_mpo_mid(const double* t1, const double* O, int64_t D1, int wl, int d, int wr, int64_t D2,
                                double* t2, hipStream_t st) {
  const int nin = RIGHT ? d * wr : wl * d, nout = RIGHT ? wl * d : d * wr;
  if (D1 * D2 * nout == 0) return MK_OK;
  // four workgroups a CU, as far as the outputs go
  dim3 g = grid1d(D1 * D2, 1);
  g.y = (unsigned)std::max<int64_t>(1, std::min<int64_t>(nout, 1024 / g.x));
#define MPO_MID(N) hipLaunchKernelGGL((mpo_mid_kernel<N, RIGHT>), g, dim3(256), 0, st, t1, O, D1, wl, d, wr, D2, t2)
  // no input at all (an empty bond): a zero per output, without reading O
  if (nin == 0 || nin > 32)
    hipLaunchKernelGGL((mpo_mid_wide_kernel<RIGHT>), grid1d(D1 * nout * D2, 4), dim3(TPB), 0, st, t1, O, D1, wl, d, wr,
                       D2, t2);
  else if (nin <= 4) MPO_MID(4);
  else if (nin <= 6) MPO_MID(6);
  else if (nin <= 10) MPO_MID(10);
  else if (nin <= 16) MPO_MID(16);
  else MPO_MID(32);
#undef MPO_MID
  MK_CHECK_HIP(hipGetLastError());
  return MK_OK;
}
mk_status k_tl_mid(const double* t1, const double* O, int64_t Dm, int wl, int d, int wr, int64_t Dc, double* t2,
                   hipStream_t st) {
  return launch_mpo_mid<false>(t1, O, Dm, wl, d, wr, Dc, t2, st);
}
mk_status k_tr_mid(const double* t1, const double* O, int64_t Da, int wl, int d, int wr, int64_t Do, double* t2,
                   hipStream_t st) {
  return launch_mpo_mid<true>(t1, O, Da, wl, d, wr, Do, t2, st);
}
mk_status k_swap_mid(const double* in, int64_t n0, int64_t n1, int64_t n2, int64_t n3, double* out,
                     hipStream_t st) {
  LAUNCH_1D(swap_mid_kernel, n0 * n1 * n2 * n3, st, in, n0, n1, n2, n3, out);
}
mk_status k_mpo_extend(const double* O, int wl, int d, int wr, int ne, int nq, double* out, hipStream_t st) {
  LAUNCH_1D(mpo_extend_kernel, (int64_t)wl * ne * d * nq * d * nq * wr * ne, st, O, wl, d, wr, ne, nq, out);
}
mk_status k_tl_mid_mixed(const double* t1, const double* O, int64_t Dm, int wl, int d, int wr, int64_t Dc,
                         int64_t ldo, int split, void* hi, void* lo, hipStream_t st) {
  if (split) LAUNCH_1D(tl_mid_mixed_kernel<true>, ldo * wr * Dc, st, t1, O, Dm, wl, d, wr, Dc, ldo, hi, lo);
  LAUNCH_1D(tl_mid_mixed_kernel<false>, ldo * wr * Dc, st, t1, O, Dm, wl, d, wr, Dc, ldo, hi, lo);
}
mk_status k_tr_mid_mixed(const double* t1, const double* O, int64_t Da, int wl, int d, int wr, int64_t Do,
                         int64_t ldo, int split, void* hi, void* lo, hipStream_t st) {
  if (Da * wl * ldo == 0) return MK_OK;
  dim3 g((unsigned)cdiv(Da * wl, (int64_t)64), (unsigned)cdiv(ldo, (int64_t)64));
  if (split)
    hipLaunchKernelGGL(tr_mid_mixed_kernel<true>, g, dim3(256), 0, st, t1, O, Da, wl, d, wr, Do, ldo, hi, lo);
  else
    hipLaunchKernelGGL(tr_mid_mixed_kernel<false>, g, dim3(256), 0, st, t1, O, Da, wl, d, wr, Do, ldo, hi, lo);
  MK_CHECK_HIP(hipGetLastError());
  return MK_OK;
}
mk_status k_phys2(const double* P, const double* x, int64_t Dl, int d1, int64_t Dr, int d2,
                  double alpha, double beta, double* y, hipStream_t st) {
  switch (d1 * d2) {
    case 2: LAUNCH_1D(phys2_reg_kernel<2>, Dl * Dr, st, P, x, Dl, d1, Dr, d2, alpha, beta, y);
    case 3: LAUNCH_1D(phys2_reg_kernel<3>, Dl * Dr, st, P, x, Dl, d1, Dr, d2, alpha, beta, y);
    case 4: LAUNCH_1D(phys2_reg_kernel<4>, Dl * Dr, st, P, x, Dl, d1, Dr, d2, alpha, beta, y);
    case 9: LAUNCH_1D(phys2_reg_kernel<9>, Dl * Dr, st, P, x, Dl, d1, Dr, d2, alpha, beta, y);
    case 16: LAUNCH_1D(phys2_reg_kernel<16>, Dl * Dr, st, P, x, Dl, d1, Dr, d2, alpha, beta, y);
    default: LAUNCH_1D(phys2_kernel, Dl * d1 * Dr * d2, st, P, x, Dl, d1, Dr, d2, alpha, beta, y);
  }
}
mk_status k_diag_nn(const double* IC, const double* BE, const double* P, int64_t Dl, int64_t Dr, int d1, int d2,
                    double* out, hipStream_t st) {
  LAUNCH_1D(diag_nn_kernel, Dl * d1 * Dr * d2, st, IC, BE, P, Dl, Dr, d1, d2, out);
}
mk_status k_phys1(const double* P, const double* x, int64_t Dl, int d, int64_t Dr, double alpha,
                  double beta, double* y, hipStream_t st) {
  LAUNCH_1D(phys1_kernel, Dl * d * Dr, st, P, x, Dl, d, Dr, alpha, beta, y);
}

mk_status k_regularize(double* v, const double* lvec, const double* rvec, int64_t D1, int w, int64_t D2,
                       double* lam, hipStream_t st) {
  if (D1 * D2 * w == 0) return MK_OK;
  hipLaunchKernelGGL(reg_lambda_kernel, dim3(w), dim3(TPB), 0, st, v, lvec, D1, w, D2, lam);
  MK_CHECK_HIP(hipGetLastError());
  hipLaunchKernelGGL(reg_apply_kernel, grid1d(D1 * w * D2, 4), dim3(TPB), 0, st, v, rvec, lam, D1, w, D2);
  MK_CHECK_HIP(hipGetLastError());
  return MK_OK;
}

int multidot_blocks(int64_t n) { return (int)std::max<int64_t>(1, cdiv(n, (int64_t)TPB * MD_ITEMS)); }

int cgs_blocks(int64_t n);

template <int MODE, typename VT>
void launch_cgs(int k, int nb, hipStream_t st, const VT* V, int64_t ldv, const double* cin, int lo, double* u,
                const double* w, int64_t n, double* partial) {
  if (k <= 4)
    hipLaunchKernelGGL((cgs_update_kernel<MODE, 4, VT>), dim3(nb), dim3(TPB), 0, st, V, ldv, k, cin, lo, u, w, n,
                       partial);
  else if (k <= 8)
    hipLaunchKernelGGL((cgs_update_kernel<MODE, 8, VT>), dim3(nb), dim3(TPB), 0, st, V, ldv, k, cin, lo, u, w, n,
                       partial);
  else if (k <= 16)
    hipLaunchKernelGGL((cgs_update_kernel<MODE, 16, VT>), dim3(nb), dim3(TPB), 0, st, V, ldv, k, cin, lo, u, w, n,
                       partial);
  else
    hipLaunchKernelGGL((cgs_update_kernel<MODE, 32, VT>), dim3(nb), dim3(TPB), 0, st, V, ldv, k, cin, lo, u, w, n,
                       partial);
}

mk_status k_multidot(const double* V, int64_t ldv, int k, const double* w, int64_t n, double* out,
                     double* partial, hipStream_t st) {
  if (k <= 0) return MK_OK;
  if (k <= CGS_KMAX) {
    // one read of V with register accumulators; at most multidot_blocks(n)
    // blocks, so callers' partial buffers sized for the wide kernel suffice
    const int nb = std::min(cgs_blocks(n), multidot_blocks(n));
    launch_cgs<2, double>(k, nb, st, V, ldv, nullptr, 0, const_cast<double*>(w), nullptr, n, partial);
    MK_CHECK_HIP(hipGetLastError());
    hipLaunchKernelGGL(reduce_rows_kernel, dim3(k), dim3(TPB), 0, st, partial, nb, out);
    MK_CHECK_HIP(hipGetLastError());
    return MK_OK;
  }
  const int nb = multidot_blocks(n);
  hipLaunchKernelGGL(multidot_kernel, dim3(nb), dim3(TPB), 0, st, V, ldv, k, w, n, partial);
  MK_CHECK_HIP(hipGetLastError());
  hipLaunchKernelGGL(reduce_rows_kernel, dim3(k), dim3(TPB), 0, st, partial, nb, out);
  MK_CHECK_HIP(hipGetLastError());
  return MK_OK;
}
int cgs_blocks(int64_t n) { return (int)std::min<int64_t>(1024, std::max<int64_t>(1, cdiv(n, (int64_t)TPB * 4))); }

mk_status k_cgs_update_dot(const double* V, int64_t ldv, int k, const double* cin, int lo, double* u, int64_t n,
                           double* out, double* partial, hipStream_t st) {
  MK_REQUIRE(k >= 1 && k <= CGS_KMAX, MK_BAD_ARG, "cgs_update_dot: k = %d not in [1, %d]", k, CGS_KMAX);
  const int nb = cgs_blocks(n);
  launch_cgs<0, double>(k, nb, st, V, ldv, cin, lo, u, nullptr, n, partial);
  MK_CHECK_HIP(hipGetLastError());
  hipLaunchKernelGGL(reduce_rows_kernel, dim3(k), dim3(TPB), 0, st, partial, nb, out);
  MK_CHECK_HIP(hipGetLastError());
  return MK_OK;
}

mk_status k_cgs_update_norm(const double* V, int64_t ldv, int k, const double* cin, double* u, const double* w,
                            int64_t n, double* out, double* partial, hipStream_t st) {
  MK_REQUIRE(k >= 1 && k <= CGS_KMAX, MK_BAD_ARG, "cgs_update_norm: k = %d not in [1, %d]", k, CGS_KMAX);
  const int nb = cgs_blocks(n);
  launch_cgs<1, double>(k, nb, st, V, ldv, cin, 0, u, w, n, partial);
  MK_CHECK_HIP(hipGetLastError());
  hipLaunchKernelGGL(reduce_rows_kernel, dim3(2), dim3(TPB), 0, st, partial, nb, out);
  MK_CHECK_HIP(hipGetLastError());
  return MK_OK;
}

mk_status k_multiaxpy(const double* V, int64_t ldv, int k, const double* c, double* w, int64_t n,
                      hipStream_t st) {
  if (k <= 0) return MK_OK;
  LAUNCH_1D(multiaxpy_kernel, n, st, V, ldv, k, c, w, n);
}
mk_status k_gemv(const double* V, int64_t ldv, int k, const double* s, double* x, int64_t n,
                 hipStream_t st) {
  LAUNCH_1D(gemv_kernel, n, st, V, ldv, k, s, x, n);
}

mk_status k_axpby(double a, const double* x, double b, double* y, int64_t n, hipStream_t st) {
  LAUNCH_1D(axpby_kernel, n, st, a, x, b, y, n);
}
mk_status k_normalize(const double* x, const double* s2, double* y, int64_t n, hipStream_t st) {
  LAUNCH_1D(normalize_kernel, n, st, x, s2, y, n);
}
mk_status k_scale_dev(double* y, const double* sdev, int inv, int64_t n, hipStream_t st) {
  LAUNCH_1D(scale_dev_kernel, n, st, y, sdev, inv, n);
}
mk_status k_nonfinite(const double* x, int64_t n, int* flag, hipStream_t st) {
  LAUNCH_1D(nonfinite_kernel, n, st, x, n, flag);
}

mk_status k_convert(const double* M, int64_t MN, int64_t run, int nrun, int64_t runpad, int64_t ld, int trans,
                    int64_t ldo, int split, void* hi, void* lo, hipStream_t st) {
  if (MN * run * nrun == 0) return MK_OK;
  MK_REQUIRE(runpad % 8 == 0 && ldo % 8 == 0 && runpad >= run && runpad * nrun <= ldo, MK_BAD_ARG,
             "convert: runs of %lld padded to %lld, rows of %lld", (long long)run, (long long)runpad, (long long)ldo);
  if (trans) {
    const dim3 g = grid1d(ldo / 8 * MN, 1);
    if (split)
      hipLaunchKernelGGL((conv_plain_kernel<true>), g, dim3(TPB), 0, st, M, run, nrun, runpad, MN, ld, ldo, hi, lo);
    else
      hipLaunchKernelGGL((conv_plain_kernel<false>), g, dim3(TPB), 0, st, M, run, nrun, runpad, MN, ld, ldo, hi, lo);
  } else {
    dim3 g((unsigned)cdiv(MN, 64), (unsigned)cdiv(ldo, 64));
    if (split)
      hipLaunchKernelGGL((conv_trans_kernel<true>), g, dim3(256), 0, st, M, MN, run, nrun, runpad, ld, ldo, hi, lo);
    else
      hipLaunchKernelGGL((conv_trans_kernel<false>), g, dim3(256), 0, st, M, MN, run, nrun, runpad, ld, ldo, hi, lo);
  }
  MK_CHECK_HIP(hipGetLastError());
  return MK_OK;
}

int gen_mid_nin(int nin) { return nin <= 8 ? 8 : nin <= 16 ? 16 : nin <= 20 ? 20 : nin <= 32 ? 32 : 0; }

template <int MODE>
static mk_status launch_gen_mid(int nin, dim3 g, hipStream_t st, const double* t1, const double* Wc, int64_t Df, int wl,
                                int d1, int wr, int d2, int64_t nc, double* t2, int64_t ldo, void* hi, void* lo) {
#define GEN_MID(N) \
  hipLaunchKernelGGL((gen_mid_kernel<N, MODE>), g, dim3(256), 0, st, t1, Wc, Df, wl, d1, wr, d2, nc, t2, ldo, hi, lo)
  switch (gen_mid_nin(nin)) {
    case 8: GEN_MID(8); break;
    case 16: GEN_MID(16); break;
    case 20: GEN_MID(20); break;
    case 32: GEN_MID(32); break;
    default: MK_REQUIRE(false, MK_BAD_ARG, "gen_mid: %d inputs", nin);
  }
#undef GEN_MID
  MK_CHECK_HIP(hipGetLastError());
  return MK_OK;
}

mk_status k_gen_mid(const double* t1, const double* Wc, int64_t Df, int wl, int d1, int wr, int d2, int64_t nc,
                    int prec, double* t2, int64_t ldo, void* hi, void* lo, hipStream_t st) {
  if (Df * nc == 0) return MK_OK;
  MK_REQUIRE(prec == MK_FP64 || ldo >= Df * wl, MK_BAD_ARG, "gen_mid: rows of %lld", (long long)ldo);
  const dim3 g = grid1d(Df * nc, 1);
  const int nin = d1 * wr * d2;
  if (prec == MK_FP64) return launch_gen_mid<0>(nin, g, st, t1, Wc, Df, wl, d1, wr, d2, nc, t2, ldo, hi, lo);
  if (prec == MK_BF16X3) return launch_gen_mid<1>(nin, g, st, t1, Wc, Df, wl, d1, wr, d2, nc, t2, ldo, hi, lo);
  return launch_gen_mid<2>(nin, g, st, t1, Wc, Df, wl, d1, wr, d2, nc, t2, ldo, hi, lo);
}

mk_status k_nn_prologue(const double* P, const double* x, int64_t Dl, int64_t Dr, int d2, double alpha, double beta,
                        double* y, int split, void* xa_hi, void* xa_lo, int64_t ka, void* xb_hi, void* xb_lo,
                        int64_t kb, int packed, hipStream_t st) {
  if (Dl * Dr == 0) return MK_OK;
  MK_REQUIRE(d2 == 1 || d2 == 2, MK_BAD_ARG, "nn_prologue: d2 = %d", d2);
  if (packed)
    MK_REQUIRE(split && d2 == 2 && (2 * Dl) % 256 == 0 && (2 * Dr) % 256 == 0 && ka == 2 * Dr && kb == 2 * Dl,
               MK_BAD_ARG, "nn_prologue: packed views are bf16, with 2 Dl, 2 Dr multiples of 256 and unpadded rows");
  // 64 columns a block (128-byte runs of the bf16 left view) while that makes two
  // blocks a CU, fewer below: at D = 512 the 128 blocks of 64 columns took 14.5 us
  // and the 512 of 16 columns 7.6
  const int64_t rows = cdiv(Dl, (int64_t)PRO_A);
  const int pc = packed || rows * cdiv(Dr, (int64_t)64) >= 512 ? 64 : rows * cdiv(Dr, (int64_t)32) >= 512 ? 32 : 16;
  const dim3 g((unsigned)rows, (unsigned)cdiv(Dr, (int64_t)pc));
#define NN_PROLOGUE(S, K, N, C) \
  hipLaunchKernelGGL((nn_prologue_kernel<S, K, N, C>), g, dim3(256), 0, st, P, x, Dl, Dr, alpha, beta, y, xa_hi, \
                     S ? xa_lo : nullptr, ka, xb_hi, S ? xb_lo : nullptr, kb)
#define NN_PROLOGUE_C(S, N) \
  do { \
    if (pc == 64) NN_PROLOGUE(S, false, N, 64); \
    else if (pc == 32) NN_PROLOGUE(S, false, N, 32); \
    else NN_PROLOGUE(S, false, N, 16); \
  } while (0)
  if (packed) NN_PROLOGUE(true, true, 2, 64);
  else if (split && d2 == 2) NN_PROLOGUE_C(true, 2);
  else if (split) NN_PROLOGUE_C(true, 1);
  else if (d2 == 2) NN_PROLOGUE_C(false, 2);
  else NN_PROLOGUE_C(false, 1);
#undef NN_PROLOGUE_C
#undef NN_PROLOGUE
  MK_CHECK_HIP(hipGetLastError());
  return MK_OK;
}

mk_status k_env_blocks(const double* E, const double* coef, int64_t D, int w, int nq, int left, double* out,
                       hipStream_t st) {
  if (nq == 0) return MK_OK;
  const dim3 g = grid1d(D * D, 1);
  if (left) hipLaunchKernelGGL((env_blocks_kernel<true>), g, dim3(256), 0, st, E, coef, D, w, nq, out);
  else hipLaunchKernelGGL((env_blocks_kernel<false>), g, dim3(256), 0, st, E, coef, D, w, nq, out);
  MK_CHECK_HIP(hipGetLastError());
  return MK_OK;
}

mk_status k_repack(const void* in, int64_t MN, int64_t K, int64_t kpad, int eb, void* out, hipStream_t st) {
  MK_REQUIRE(MN % 256 == 0 && (K * eb) % 64 == 0 && kpad >= K && (kpad * eb) % 16 == 0 &&
                 (uintptr_t)in % 16 == 0 && (uintptr_t)out % 16 == 0,
             MK_BAD_ARG, "repack: rows %lld, K %lld, kpad %lld do not fit the packed layout", (long long)MN,
             (long long)K, (long long)kpad);
  if (MN * K == 0) return MK_OK;
  LAUNCH_1D(repack_kernel, MN * K * eb / 16, st, static_cast<const char*>(in), MN, K, kpad, eb,
            static_cast<char*>(out));
}


mk_status k_asm_ic(const double* IC, const double* ID, const double* II, int64_t Dr, int d2, double* out,
                   hipStream_t st) {
  LAUNCH_1D(asm_ic_kernel, Dr * d2 * Dr * d2, st, IC, ID, II, Dr, d2, out);
}
mk_status k_asm_be(const double* BE, const double* DE, const double* EE, int64_t Dl, int d1, double* out,
                   hipStream_t st) {
  LAUNCH_1D(asm_be_kernel, Dl * d1 * Dl * d1, st, BE, DE, EE, Dl, d1, out);
}
mk_status k_asm_ca(const double* CA, const double* CB, const double* IC, const double* ID, const double* II,
                   int64_t Dr, int d1, int d2, double* out, hipStream_t st) {
  const int64_t R = (int64_t)d1 * Dr * d2;
  LAUNCH_1D(asm_ca_kernel, R * R, st, CA, CB, IC, ID, II, Dr, d1, d2, out);
}
mk_status k_asm_ab(const double* AB, const double* CB, const double* BE, const double* DE, const double* EE,
                   int64_t Dl, int d1, int d2, double* out, hipStream_t st) {
  const int64_t M = Dl * d1;
  LAUNCH_1D(asm_ab_kernel, M * M * d2 * d2, st, AB, CB, BE, DE, EE, Dl, d1, d2, out);
}
mk_status k_asm_cp(const double* C, const double* D, const double* I, int64_t Dr, int d, double* out,
                   hipStream_t st) {
  LAUNCH_1D(asm_cp_kernel, Dr * d * Dr * d, st, C, D, I, Dr, d, out);
}

}  // namespace mk
