// Cholesky solve of the direct SR (cholesky_solve, sr.rs:535,
// sr_backend.rs:243-247): S = U^T U from the upper triangle of a column-major
// S, that is L L^T with L[j][k] = S[k + j n] row by row, then L y = b and
// L^T x = y.
//
// What bounds it at the orders in use (n to a few thousand: n^3 / 3 is 7 us
// of FP64 MFMA at n = 1111) is the chain of n pivots and the launches it is
// cut into, so the split keeps that chain short:
//  - one launch per panel of 64 columns.  Workgroup (I, J) of the trailing
//    tiles solves L_I and L_J itself from the panel P and the panel's diagonal
//    factor (MFMA, blocks of 16 columns with the inverses of the factor's 16 x
//    16 diagonal blocks, all tiles at once) instead of waiting for a launch
//    that solves the panel, then A_IJ -= L_I L_J^T.  (One product with the
//    inverse of all 64 columns is as fast, with residuals up to twice as large.)
//  - the tiles of the next panel go to a buffer of their own, so the
//    panel L can be written back in the launch that still reads P.
//  - workgroup (k+1, k+1) goes on to factor its tile in column blocks of 16,
//    a row per lane with the pivots by readlane, the block's inverse from
//    identity rows in further lanes, MFMA between the blocks.
//  - L y = b rides along with the diagonal tiles; L^T x = y takes a launch
//    per 256 columns, every workgroup solving that block itself and taking
//    it from its own 64 columns.
// n = 1111: 0.56 ms (24 launches; 20 us a panel, 10 of them the 64 pivots)
// where a factorisation and two triangular solves by the vendor's solver took
// 3.4; n = 5000: 4.4 ms.  Residuals are 0.6 of the vendor's.
// From CH_PRE trailing tile rows on, forming L_I per tile costs more than a
// launch (3 products a tile instead of 1): the panel is solved by a launch of
// its own first.
#pragma once
#include <hip/hip_runtime.h>

#include "pfinv_dev.h"

namespace mvmc_hip {

constexpr int CH_B = 64;    // tile order
constexpr int CH_LD = 66;   // LDS row stride: 16 rows x 2 k of an operand fetch fall in distinct banks
constexpr size_t CH_V = sizeof(double) * CH_B * 16;  // LDS of a tile's inverted diagonal blocks
constexpr int CH_BACK = 4;  // tiles per launch of the back substitution
constexpr int CH_PRE = 40;  // trailing tile rows from which the panel has its own launch

typedef double ch_v2d __attribute__((ext_vector_type(2)));
typedef double ch_v4d __attribute__((ext_vector_type(4)));

// Workspace: diagonal factors [nt][64][64] (the 16 x 16 blocks below the
// diagonal ones from L, the diagonal blocks inverted), panels [2][64 nt][64],
// right-hand side b and forward solution y [64 nt] each.
struct CholWs {
  double *F, *P, *b, *y;
  int* info;
};
inline size_t chol_ws_doubles(int n) {
  const size_t np = (size_t)((n + CH_B - 1) / CH_B) * CH_B;
  return 3 * np * CH_B + 2 * np + 1;
}
inline CholWs chol_ws(double* p, int n) {
  const size_t np = (size_t)((n + CH_B - 1) / CH_B) * CH_B;
  return {p, p + np * CH_B, p + 3 * np * CH_B, p + 3 * np * CH_B + np, (int*)(p + 3 * np * CH_B + 2 * np)};
}

// Reciprocal q of a pivot p, its square root d and the root's reciprocal r, by
// Newton's and Goldschmidt's iterations from the hardware's estimates.  The
// next pivot waits for q alone, which takes half the latency of a division.
// ANY: pivots out of the iterations' range (ch_usual) too.
__device__ __forceinline__ bool ch_usual(double p) { return p > 0x1p-900 && p < 0x1p900; }
template <bool ANY>
__device__ __forceinline__ void ch_pivot(double p, double& q, double& d, double& r) {
  if (ANY) {
    q = 1.0 / p;
    d = sqrt(p);
    r = 1.0 / d;
    return;
  }
  q = __builtin_amdgcn_rcp(p);
  q = __builtin_fma(__builtin_fma(-p, q, 1.0), q, q);
  q = __builtin_fma(__builtin_fma(-p, q, 1.0), q, q);
  const double y = __builtin_amdgcn_rsq(p);
  double g = p * y, h = 0.5 * y;
  double e = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, e, g);
  h = __builtin_fma(h, e, h);
  e = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, e, g);
  h = __builtin_fma(h, e, h);
  d = __builtin_fma(__builtin_fma(-g, g, p), h, g);
  r = h + h;
  r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
}

__device__ __forceinline__ double ch_lane(double x, int lane) {
  const long long b = __builtin_bit_cast(long long, x);
  const int lo = __builtin_amdgcn_readlane((int)b, lane), hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
}

// Step K of a 16-column block: a lane's row a[], the diagonal block's rows in
// lanes 0..15; lane K < 16 keeps pivot K.
template <bool ANY, int K = 0>
__device__ __forceinline__ void ch_steps(double (&a)[16], double& pivot) {
  if constexpr (K < 16) {
    const double p = ch_lane(a[K], K);
    const bool own = (threadIdx.x & 63) == K;
    if (own) pivot = p;
    double q, d, r;
    ch_pivot<ANY>(p, q, d, r);
    const double t = a[K] * q;
#pragma unroll
    for (int j = K + 1; j < 16; ++j) a[j] = __builtin_fma(-t, ch_lane(a[K], j), a[j]);
    // l = a r, its rounding corrected
    const double l = a[K] * r;
    a[K] = own ? d : __builtin_fma(__builtin_fma(-l, d, a[K]), r, l);
    ch_steps<ANY, K + 1>(a, pivot);
  }
}

// X Y^T over k in [k0, k1): X rows from x, Y rows from y (LDS, stride CH_LD).
// Lane l feeds X[l % 16][k + l / 16] and Y[l % 16][k + l / 16] and holds rows
// l / 16 + 4 e of column l % 16.  Products are summed from zero and taken from
// a tile by one subtraction: summed onto the tile, every one of them would
// round at the tile's magnitude (twice the residual at n = 1111).
__device__ __forceinline__ ch_v4d ch_mul(const double* x, const double* y, int k0, int k1) {
  const int lane = threadIdx.x & 63, r = lane & 15, kq = lane >> 4;
  ch_v4d acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
  for (int k = k0; k < k1; k += 4)
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(x[r * CH_LD + k + kq], y[r * CH_LD + k + kq], acc, 0, 0, 0);
  return acc;
}

__device__ __forceinline__ ch_v4d ch_get(const double* c) {
  const int lane = threadIdx.x & 63;
  ch_v4d x;
#pragma unroll
  for (int e = 0; e < 4; ++e) x[e] = c[((lane >> 4) + 4 * e) * CH_LD + (lane & 15)];
  return x;
}
__device__ __forceinline__ void ch_put(double* c, ch_v4d x) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int e = 0; e < 4; ++e) c[((lane >> 4) + 4 * e) * CH_LD + (lane & 15)] = x[e];
}

// Factors the tile T (lower triangle read) in place and leaves the inverses
// of the factor's 16 x 16 diagonal blocks in V [4][16][16]; 256 threads, all
// of them enter.  Wave 3 does `side` meanwhile.
template <class Side>
__device__ __forceinline__ void ch_factor(double* T, double* V, int first, int n, int* info, Side side) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  __syncthreads();
#pragma unroll 1
  for (int b = 0; b < 4; ++b) {
    const int c0 = 16 * b;
    // wave 0: T's rows from the diagonal block on; wave 1: the diagonal block
    // again, and the rows of an identity
    const int tr = min(c0 + lane, CH_B - 1);
    double* row = T + (wave == 0 ? tr : c0 + (lane & 15)) * CH_LD + c0;
    double a[16];
    if (wave < 2) {
      const bool ident = wave == 1 && lane >= 16;
      auto load = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < 16; ++k) {
          const double x = row[k];
          a[k] = ident ? (k == lane - 16 ? 1.0 : 0.0) : x;
        }
      };
      double pivot = 1.0;
      load();
      ch_steps<false>(a, pivot);
      if (__ballot(lane < 16 && !ch_usual(pivot)) != 0) {
        load();
        ch_steps<true>(a, pivot);
      }
      if (wave == 0) {
        const unsigned long long bad =
            __ballot(lane < 16 && first + c0 + lane < n && !(pivot > 0.0 && pivot < __builtin_inf()));
        if (bad != 0 && lane == 0) atomicCAS(info, 0, first + c0 + __ffsll(bad));
        if (lane >= 16 && c0 + lane < CH_B) {
#pragma unroll
          for (int k = 0; k < 16; ++k) row[k] = a[k];
        }
      } else if (ident && lane < 32) {
#pragma unroll
        for (int k = 0; k < 16; ++k) V[(c0 + k) * 16 + lane - 16] = a[k];
      }
    } else if (wave == 3 && b == 0) {
      side();
    }
    __syncthreads();
    // the diagonal block, which both waves read (the trailing update does not)
    if (wave == 0 && lane < 16) {
#pragma unroll
      for (int k = 0; k < 16; ++k) row[k] = a[k];
    }
    int id = 0;
    for (int c = b + 1; c < 4; ++c)
      for (int r = c; r < 4; ++r) {
        if ((id++ & 3) != wave) continue;
        double* C = T + 16 * r * CH_LD + 16 * c;
        ch_put(C, ch_get(C) - ch_mul(T + 16 * r * CH_LD, T + 16 * c * CH_LD, c0, c0 + 16));
      }
    __syncthreads();
  }
}

// Rows p[0..15] of L from those of the panel, in place: L F^T = P in column
// blocks of 16, by one wave.
__device__ __forceinline__ void ch_rows(double* p, const double* F) {
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    if (b > 0) {
      const ch_v4d x = ch_get(p + 16 * b) - ch_mul(p, F + 16 * b * CH_LD, 0, 16 * b);
      ch_put(p + 16 * b, x);
      wave_sync();
    }
    const ch_v4d l = ch_mul(p, F + 16 * b * CH_LD, 16 * b, 16 * b + 16);
    wave_sync();
    ch_put(p + 16 * b, l);
    wave_sync();
  }
}

// y = F^{-1} v over a wave, lane r holding row r; row: the lane's row of F.
__device__ __forceinline__ double ch_forward(const double* row, double v) {
  const int lane = threadIdx.x & 63, own = lane >> 4;
  double y = 0.0;
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int c = 0; c < 16; ++c) s[c & 3] = __builtin_fma(row[16 * b + c], ch_lane(v, 16 * b + c), s[c & 3]);
    if (own == b) y = (s[0] + s[1]) + (s[2] + s[3]);
    double t[4] = {0.0, 0.0, 0.0, 0.0};
    if (b < 3) {
#pragma unroll
      for (int c = 0; c < 16; ++c) t[c & 3] = __builtin_fma(row[16 * b + c], ch_lane(y, 16 * b + c), t[c & 3]);
      if (own > b) v -= (t[0] + t[1]) + (t[2] + t[3]);
    }
  }
  return y;
}

// x = F^{-T} v, lane c holding column c; col[r]: the lane's column of F.
__device__ __forceinline__ double ch_backward(const double (&col)[CH_B], double v) {
  const int lane = threadIdx.x & 63, own = lane >> 4;
  double x = 0.0;
#pragma unroll
  for (int b = 3; b >= 0; --b) {
    double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r & 3] = __builtin_fma(col[16 * b + r], ch_lane(v, 16 * b + r), s[r & 3]);
    if (own == b) x = (s[0] + s[1]) + (s[2] + s[3]);
    double t[4] = {0.0, 0.0, 0.0, 0.0};
    if (b > 0) {
#pragma unroll
      for (int r = 0; r < 16; ++r) t[r & 3] = __builtin_fma(col[16 * b + r], ch_lane(x, 16 * b + r), t[r & 3]);
      if (own < b) v -= (t[0] + t[1]) + (t[2] + t[3]);
    }
  }
  return x;
}

// (No launch looks at info before the back substitution: behind a failed
// pivot the tiles hold NaN, which nothing reads.)
// Forward solution with panel k, by one wave: F y_k = b_k (kept by the tile
// next to the diagonal), b_I -= L_I y_k.
__device__ __forceinline__ void ch_rhs(const double* L, const double* F, const CholWs& ws, int I, int k, bool keep) {
  const int lane = threadIdx.x & 63;
  const double yk = ch_forward(F + lane * CH_LD, ws.b[k * CH_B + lane]);
  if (keep) ws.y[k * CH_B + lane] = yk;
  double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
  for (int c = 0; c < CH_B; c += 4)
#pragma unroll
    for (int u = 0; u < 4; ++u) s[u] = __builtin_fma(L[lane * CH_LD + c + u], ch_lane(yk, c + u), s[u]);
  ws.b[I * CH_B + lane] -= (s[0] + s[1]) + (s[2] + s[3]);
}

// One launch of the factorisation behind panel k (k = -1: the first panel is
// taken from S and factored).  Workgroup t holds trailing tile (I, J), I >= J
// > k; PRE: the panel L of column k already stands in S (k_chol_panel).
template <bool PRE>
__global__ void __launch_bounds__(256) k_chol_step(double* S, int n, int k, CholWs ws) {
  extern __shared__ __align__(16) double ch_lds[];
  double* sA = ch_lds;
  double* sB = sA + CH_B * CH_LD;
  double* sV = sB + CH_B * CH_LD;
  double* sF = sV + CH_B * 16;  // !PRE
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int t = blockIdx.x;
  int i, j;
  if (k < 0) {
    i = t;
    j = 0;
  } else {
    i = (int)((sqrtf(8.0f * (float)t + 1.0f) - 1.0f) * 0.5f);
    while ((i + 1) * (i + 2) / 2 <= t) ++i;
    while (i * (i + 1) / 2 > t) --i;
    j = t - i * (i + 1) / 2;
  }
  const int I = k + 1 + i, J = k + 1 + j;
  const size_t panel = (size_t)((n + CH_B - 1) / CH_B) * CH_B * CH_B;
  const double* Pk = ws.P + (size_t)(k & 1) * panel;
  double* Pn = ws.P + (size_t)((k + 1) & 1) * panel;
  const bool diag = I == J;
  ch_v4d acc[4];
  auto load_tile = [&]() __attribute__((always_inline)) {
    // wave w: rows 16 w .. 16 w + 15 of the tile, columns in four blocks
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = I * CH_B + 16 * wave + (lane >> 4) + 4 * e, q = J * CH_B + 16 * c + (lane & 15);
        acc[c][e] = r < n && q <= r ? S[(size_t)r * n + q] : (r == q ? 1.0 : 0.0);
      }
  };
  if (k >= 0) {
    const int c4 = (tid & 31) * 2, r0 = tid >> 5;
    if (PRE) {
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int r = r0 + 8 * u, ra = I * CH_B + r, rb = J * CH_B + r;
        const double* a = S + (size_t)ra * n + (size_t)k * CH_B + c4;
        const double* b = S + (size_t)rb * n + (size_t)k * CH_B + c4;
#pragma unroll
        for (int z = 0; z < 2; ++z) {
          sA[r * CH_LD + c4 + z] = ra < n ? a[z] : 0.0;
          if (!diag) sB[r * CH_LD + c4 + z] = rb < n ? b[z] : 0.0;
        }
      }
      load_tile();
      __syncthreads();
    } else {
      const double* F = ws.F + (size_t)k * CH_B * CH_B;
      const double* pa = Pk + (size_t)I * CH_B * CH_B;
      const double* pb = Pk + (size_t)J * CH_B * CH_B;
      ch_v2d x[8], y[8], z[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int e = (r0 + 8 * u) * CH_B + c4;
        x[u] = *(const ch_v2d*)(pa + e);
        z[u] = *(const ch_v2d*)(F + e);
        if (!diag) y[u] = *(const ch_v2d*)(pb + e);
      }
      load_tile();  // behind the loads that are needed first
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int e = (r0 + 8 * u) * CH_LD + c4;
        *(ch_v2d*)(sA + e) = x[u];
        *(ch_v2d*)(sF + e) = z[u];
        if (!diag) *(ch_v2d*)(sB + e) = y[u];
      }
      __syncthreads();
      // a wave's rows are its own
      ch_rows(sA + 16 * wave * CH_LD, sF);
      if (!diag) ch_rows(sB + 16 * wave * CH_LD, sF);
      __syncthreads();
    }
    const double* la = sA + (16 * wave + (lane & 15)) * CH_LD + (lane >> 4);
    const double* lb = (diag ? sA : sB) + (lane & 15) * CH_LD + (lane >> 4);
    ch_v4d sum[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) sum[c] = ch_v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < CH_B; q += 4) {
      const double av = la[q];
#pragma unroll
      for (int c = 0; c < 4; ++c)
        sum[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, lb[16 * c * CH_LD + q], sum[c], 0, 0, 0);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[c] -= sum[c];
    if (!PRE) {
      if (j == 0) {  // panel k of the factor
#pragma unroll
        for (int u = 0; u < 16; ++u) {
          const int r = (tid >> 6) + 4 * u, ra = I * CH_B + r;
          if (ra < n) S[(size_t)ra * n + (size_t)k * CH_B + lane] = sA[r * CH_LD + lane];
        }
      }
      if (diag && j > 0 && wave == 0) ch_rhs(sA, sF, ws, I, k, false);
    }
  }
  if (k < 0) load_tile();
  if (j == 0) {
    if (!diag) {
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          Pn[(size_t)I * CH_B * CH_B + (16 * wave + (lane >> 4) + 4 * e) * CH_B + 16 * c + (lane & 15)] = acc[c][e];
      return;
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) sB[(16 * wave + (lane >> 4) + 4 * e) * CH_LD + 16 * c + (lane & 15)] = acc[c][e];
    ch_factor(sB, sV, I * CH_B, n, ws.info, [&] {
      if (!PRE && k >= 0) ch_rhs(sA, sF, ws, I, k, true);
    });
    double* F = ws.F + (size_t)I * CH_B * CH_B;
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const int r = (tid >> 6) + 4 * u, ra = I * CH_B + r;
      F[r * CH_B + lane] = lane > r ? 0.0 : (lane >> 4) == (r >> 4) ? sV[r * 16 + (lane & 15)] : sB[r * CH_LD + lane];
      if (ra < n && lane <= r) S[(size_t)ra * n + (size_t)I * CH_B + lane] = sB[r * CH_LD + lane];
    }
    return;
  }
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = I * CH_B + 16 * wave + (lane >> 4) + 4 * e, q = J * CH_B + 16 * c + (lane & 15);
      if (r < n && q <= r) S[(size_t)r * n + q] = acc[c][e];
    }
}

// Panel k of the factor, a tile per workgroup (tile k + 1 + blockIdx.x), and
// the right-hand side's part.
__global__ void __launch_bounds__(256) k_chol_panel(double* S, int n, int k, CholWs ws) {
  extern __shared__ __align__(16) double ch_lds[];
  double* sA = ch_lds;
  double* sF = sA + CH_B * CH_LD;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int I = k + 1 + blockIdx.x;
  const size_t panel = (size_t)((n + CH_B - 1) / CH_B) * CH_B * CH_B;
  const double* pa = ws.P + (size_t)(k & 1) * panel + (size_t)I * CH_B * CH_B;
  const double* F = ws.F + (size_t)k * CH_B * CH_B;
#pragma unroll
  for (int u = 0; u < 16; ++u) {
    const int r = (tid >> 6) + 4 * u;
    sA[r * CH_LD + lane] = pa[r * CH_B + lane];
    sF[r * CH_LD + lane] = F[r * CH_B + lane];
  }
  __syncthreads();
  ch_rows(sA + 16 * wave * CH_LD, sF);
  for (int r = 16 * wave; r < 16 * wave + 16; ++r)
    if (I * CH_B + r < n) S[(size_t)(I * CH_B + r) * n + (size_t)k * CH_B + lane] = sA[r * CH_LD + lane];
  __syncthreads();
  if (wave == 0) ch_rhs(sA, sF, ws, I, k, I == k + 1);
}

// b = rhs (padded with zeros), info = 0.
__global__ void k_chol_begin(const double* rhs, int n, int np, CholWs ws) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e < np) ws.b[e] = e < n ? rhs[e] : 0.0;
  if (e == 0) *ws.info = 0;
}

// Back substitution of tiles k1, k1 - 1, .. k0: every workgroup solves them
// (F_k^T x_k = y_k, y_j -= L_kj^T x_k below), then takes them from its tile
// blockIdx.x of y; workgroup 0 writes x.  A failed factorisation leaves x
// alone.
__global__ void __launch_bounds__(256) k_chol_back(const double* S, int n, int k0, int k1, int nt, CholWs ws,
                                                   double* x) {
  __shared__ double y[CH_BACK * CH_B];
  __shared__ double xk[CH_BACK * CH_B];
  __shared__ double part[4][CH_B];
  if (*ws.info != 0) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int cols = (k1 - k0 + 1) * CH_B;
  if (tid < cols) y[tid] = k0 * CH_B + tid >= (nt - 1) * CH_B ? ws.b[k0 * CH_B + tid] : ws.y[k0 * CH_B + tid];
  __syncthreads();
  for (int k = k1; k >= k0; --k) {
    double l[16];
    if (wave == 0) {
      const double* F = ws.F + (size_t)k * CH_B * CH_B;
      double f[CH_B];
      double v = y[(k - k0) * CH_B + lane];
      if (k == nt - 1) {  // the last tile's forward solution
#pragma unroll
        for (int c = 0; c < CH_B; ++c) f[c] = F[lane * CH_B + c];
        v = ch_forward(f, v);
      }
#pragma unroll
      for (int c = 0; c < CH_B; ++c) f[c] = F[c * CH_B + lane];
      xk[(k - k0) * CH_B + lane] = ch_backward(f, v);
    }
    __syncthreads();
    // column tid of the block's tiles below k
    if (tid < (k - k0) * CH_B) {
      double v[4] = {0.0, 0.0, 0.0, 0.0};
      for (int r0 = 0; r0 < CH_B; r0 += 16) {
#pragma unroll
        for (int u = 0; u < 16; ++u) {
          const int row = k * CH_B + r0 + u;
          l[u] = row < n ? S[(size_t)row * n + k0 * CH_B + tid] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < 16; ++u) v[u & 3] = __builtin_fma(l[u], xk[(k - k0) * CH_B + r0 + u], v[u & 3]);
      }
      y[tid] -= (v[0] + v[1]) + (v[2] + v[3]);
    }
    __syncthreads();
  }
  if (blockIdx.x == 0 && tid < cols && k0 * CH_B + tid < n) x[k0 * CH_B + tid] = xk[tid];
  if (k0 == 0) return;
  // own tile: wave w takes tile row k0 + w of the block
  double v = 0.0;
  if (k0 + wave <= k1) {
    for (int r0 = 0; r0 < CH_B; r0 += 16) {
      double l[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const int row = (k0 + wave) * CH_B + r0 + u;
        l[u] = row < n ? S[(size_t)row * n + (size_t)blockIdx.x * CH_B + lane] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < 16; ++u) v = __builtin_fma(l[u], xk[wave * CH_B + r0 + u], v);
    }
  }
  part[wave][lane] = v;
  __syncthreads();
  if (wave == 0) ws.y[blockIdx.x * CH_B + lane] -= (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
}

inline void chol_launches(double* S, double* x, int n, double* work, hipStream_t st) {
  const CholWs ws = chol_ws(work, n);
  const int nt = (n + CH_B - 1) / CH_B;
  const size_t tile = sizeof(double) * CH_B * CH_LD;
  hipLaunchKernelGGL(k_chol_begin, dim3((unsigned)((nt * CH_B + 255) / 256)), dim3(256), 0, st, x, n, nt * CH_B, ws);
  hipLaunchKernelGGL(k_chol_step<false>, dim3((unsigned)nt), dim3(256), 3 * tile + CH_V, st, S, n, -1, ws);
  for (int k = 0; k + 1 < nt; ++k) {
    const int m = nt - 1 - k;
    const unsigned tiles = (unsigned)(m * (m + 1) / 2);
    if (m >= CH_PRE) {
      hipLaunchKernelGGL(k_chol_panel, dim3((unsigned)m), dim3(256), 2 * tile, st, S, n, k, ws);
      hipLaunchKernelGGL(k_chol_step<true>, dim3(tiles), dim3(256), 2 * tile + CH_V, st, S, n, k, ws);
    } else {
      hipLaunchKernelGGL(k_chol_step<false>, dim3(tiles), dim3(256), 3 * tile + CH_V, st, S, n, k, ws);
    }
  }
  for (int k1 = nt - 1; k1 >= 0; k1 -= CH_BACK) {
    const int k0 = k1 >= CH_BACK ? k1 - CH_BACK + 1 : 0;
    hipLaunchKernelGGL(k_chol_back, dim3((unsigned)(k0 > 0 ? k0 : 1)), dim3(256), 0, st, S, n, k0, k1, nt, ws, x);
  }
}
}  // namespace mvmc_hip
