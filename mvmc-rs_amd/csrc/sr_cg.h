// SR-CG iterations with few launches (sr_cg.rs:611-880, 952-1004; the
// arithmetic and the reduction order of the k_cg_* kernels of ensemble.hip,
// element by element):
//   k_cg_small   the whole solve in one workgroup, for operators that its CU
//                streams from L2 faster than an iteration's launches take
//   k_cg_tail    everything of an iteration after the chunk partials' first
//                fold, in one workgroup
// What bounds the solver is not arithmetic: an iteration is 8 dependent
// steps over vectors of na entries around one product with the samples, and
// as kernels each step cost 2-5 us.
#pragma once
#include "ensemble.h"
#include "sr_stages.h"

namespace mvmc_hip {

constexpr int CGS_WAVES = 8;              // waves of k_cg_small
constexpr int CGS_NT = 64 * CGS_WAVES;
constexpr int CGS_M = 10;                 // columns per lane of k_cg_small: na <= 640
// Operators that k_cg_small takes.  A wave takes a chunk of 32 rows at a time
// (CGS_WAVES chunks a round), at a cost per round of about a fixed part and a
// part per column of the lane, while an iteration of launches takes 23 .. 30 us
// whatever the size in this range.  So the line lies at rounds x (columns per
// lane + 2) = CGS_COST (us an iteration, one launch / launches):
//   columns   up to the line          behind it
//        64   1280 rows 22.2 / 26.1   2560 rows 41.9 / 26.8
//       100    800 rows 19.7 / 26.4   1600 rows 35.7 / 26.8
//       200    400 rows 19.8 / 25.7    800 rows 36.2 / 26.7
//       400    200 rows 15.8 / 25.2    400 rows 27.1 / 26.6
//       500    160 rows 19.0 / 24.5    320 rows 29.9 / 26.2
//       595    256 rows 24.7 / 30.5
// (20 x 8192 in one launch took 73 us, in launches 25).  Solves that run side
// by side cost the longest of them in one launch each and their sum in
// launches, which moves the line by their number.
// A Gram of FP32 has half the bytes and no second pass: 271 columns 8.7 us
// against 15.0, 421 columns 15.3 against 13.8.  CGS_ELEMS is its line (404
// columns) and, for samples, what keeps the chunk partials in LDS.
constexpr long long CGS_ELEMS = 160 * 1024;
constexpr long long CGS_COST = 16;
constexpr int CGT_NT = 1024;              // threads of k_cg_tail
constexpr int CGT_NMAX = 8000;            // na up to which k_cg_tail keeps products in LDS
// Superchunk partials from which their fold is a launch over all CUs instead
// of k_cg_tail's one: a launch costs 1 us more than the fold it replaces at
// 4000 partials (na = 1000, 2048 rows: 33.4 us an iteration in the tail, 34.5
// apart), as much at 8000 (4000 x 600: 59.0 and 58.8), and the tail's CU
// reads the rest at its own rate (7784 x 512: 99.8 and 96.6, 4000 x 8192: 81
// and 75, 7784 x 16384: 268 and 239).
constexpr long long CG_FOLD_MIN = 8000;

// LDS doubles of k_cg_small: x, r, d, q, mean, diag, g, the chunk partials
// and the reduction buffers.
__host__ __device__ inline size_t cgs_lds_doubles(int na, int rows, bool gram) {
  const size_t nch = gram ? 0 : (size_t)(rows + CG_RCH - 1) / CG_RCH;
  return 7 * (size_t)na + nch * na + 8;
}

// Columns per lane of the k_cg_small instance for na columns.
__host__ __device__ constexpr int cgs_columns(int na) {
  const int m = (na + 63) / 64;
  return m <= 3 ? m : m <= 5 ? 5 : m <= 7 ? 7 : CGS_M;
}

// Whether one launch solves it, beside `side` - 1 other solves.
inline bool cgs_takes(int na, int rows, bool gram, int side) {
  if (na > 64 * CGS_M || rows <= 0 || (long long)na * (gram ? na : rows) > CGS_ELEMS) return false;
  const long long rounds = ((rows + CG_RCH - 1) / CG_RCH + CGS_WAVES - 1) / CGS_WAVES;
  return gram || rounds * (cgs_columns(na) + 2) <= CGS_COST * side;
}

// Exchanges between the halves of a wave (and between odd and even rows of 16
// lanes) of two registers, and rotations of a row: a step of a tree without
// the LDS round trip of a shuffle.
__device__ __forceinline__ double cg_f64(unsigned lo, unsigned hi) {
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
// a + b with a = lanes 0..31 of x, then of y; b = lanes 32..63 of x, then of y
__device__ __forceinline__ double cg_fold32(double x, double y) {
  const unsigned long long bx = __builtin_bit_cast(unsigned long long, x), by = __builtin_bit_cast(unsigned long long, y);
  const auto l = __builtin_amdgcn_permlane32_swap((unsigned)bx, (unsigned)by, false, false);
  const auto h = __builtin_amdgcn_permlane32_swap((unsigned)(bx >> 32), (unsigned)(by >> 32), false, false);
  return cg_f64(l[0], h[0]) + cg_f64(l[1], h[1]);
}
// the same for the rows 0, 2 and 1, 3 of 16 lanes: x0 + x1, y0 + y1, x2 + x3, y2 + y3
__device__ __forceinline__ double cg_fold16(double x, double y) {
  const unsigned long long bx = __builtin_bit_cast(unsigned long long, x), by = __builtin_bit_cast(unsigned long long, y);
  const auto l = __builtin_amdgcn_permlane16_swap((unsigned)bx, (unsigned)by, false, false);
  const auto h = __builtin_amdgcn_permlane16_swap((unsigned)(bx >> 32), (unsigned)(by >> 32), false, false);
  return cg_f64(l[0], h[0]) + cg_f64(l[1], h[1]);
}
// x + x rotated by H lanes within every row of 16
template <int H>
__device__ __forceinline__ double cg_ror(double x) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, x);
  const unsigned lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x120 + H, 0xf, 0xf, true);
  const unsigned hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x120 + H, 0xf, 0xf, true);
  return x + cg_f64(lo, hi);
}
__device__ __forceinline__ double cg_tree16(double v) { return cg_ror<1>(cg_ror<2>(cg_ror<4>(cg_ror<8>(v)))); }

// Pairwise tree over the 64 lanes (h = 32 .. 1; sums of two, so the sides may
// swap), result in every lane.
__device__ __forceinline__ double cg_tree64(double v) {
  v = cg_fold32(v, v);
  return cg_tree16(cg_fold16(v, v));
}

// The trees of U = 4 values at once: lanes 0..15 hold the first's, 16..31 the
// third's, 32..47 the second's, 48..63 the fourth's; of two: a half each.
template <int U>
__device__ __forceinline__ double cg_trees(const double (&v)[U]) {
  static_assert(U == 2 || U == 4);
  const double a = cg_fold32(v[0], v[1]);
  return cg_tree16(cg_fold16(a, U == 4 ? cg_fold32(v[U - 2], v[U - 1]) : a));
}

__device__ __forceinline__ double cg_lane(double x, int lane) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, x);
  return cg_f64((unsigned)__builtin_amdgcn_readlane((int)b, lane),
                (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), lane));
}

// bdot of the 256 strided lane partials that one wave holds as p[t] = partial
// lane + 64 t: the tree h = 128, 64, then 32 .. 1.
__device__ __forceinline__ double cg_tree256_wave(double p0, double p1, double p2, double p3) {
  return cg_tree64((p0 + p2) + (p1 + p3));
}

// One product of the operator with v (LDS), into out (LDS): out = S v, or
// g - S v.  M: columns per lane.
template <int M, bool GRAM, class P>
__device__ void cgs_apply(const P* op, int rows, int na, const double* v, const double* mean, const double* diag,
                          const double* g, double inv_w, double shift, double* cp, double* red, double* out) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  double xv[M];
#pragma unroll
  for (int m = 0; m < M; ++m) xv[m] = lane + 64 * m < na ? v[lane + 64 * m] : 0.0;
  if (wave == CGS_WAVES - 1) {  // coef = mean . v
    double p[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int m = 0; m < M; ++m)
      if (lane + 64 * m < na) p[m & 3] += mean[lane + 64 * m] * xv[m];
    const double c = cg_tree256_wave(p[0], p[1], p[2], p[3]);
    if (lane == 0) red[0] = c;
  }
  // Four rows at a time (two where four do not fit the registers), the loads of
  // the next ones ahead of these ones' sums:
  // with the rows alone in flight a wave waited out an L2 latency per group,
  // and a shuffle's per step of their trees.
  constexpr int U = M <= 7 ? 4 : 2;
  auto load = [&](int r, int r1, P (&o)[U][M]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const P* row = op + (size_t)min(r + u, r1 - 1) * na;
#pragma unroll
      for (int m = 0; m < M; ++m) o[u][m] = row[min(lane + 64 * m, na - 1)];
    }
  };
  if constexpr (GRAM) {
    // row i of the symmetric Gram, as k_gram_product sums it
    auto rows4 = [&](int i0, const P (&o)[U][M]) __attribute__((always_inline)) {
      double a[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        a[u] = 0.0;
#pragma unroll
        for (int m = 0; m < M; ++m)
          if (lane + 64 * m < na) a[u] += (double)o[u][m] * xv[m];
      }
      const double t = cg_trees<U>(a);
      const int i = i0 + (U == 4 ? 2 * ((lane >> 4) & 1) : 0) + (lane >> 5);
      if ((lane & (U == 4 ? 15 : 31)) == 0 && i < na) cp[i] = t;
    };
    P o0[U][M], o1[U][M];
    constexpr int STEP = CGS_WAVES * U;
    int i0 = wave * U;
    if (i0 < na) load(i0, na, o0);
    for (; i0 < na; i0 += 2 * STEP) {
      if (i0 + STEP < na) load(i0 + STEP, na, o1);
      rows4(i0, o0);
      if (i0 + 2 * STEP < na) load(i0 + 2 * STEP, na, o0);
      if (i0 + STEP < na) rows4(i0 + STEP, o1);
    }
  } else {
    // a wave per chunk of CG_RCH rows: the row's dot, then its axpy from the
    // same registers
    const int nch = (rows + CG_RCH - 1) / CG_RCH;
    for (int c = wave; c < nch; c += CGS_WAVES) {
      const int r0 = c * CG_RCH, r1 = min(rows, r0 + CG_RCH);
      double acc[M];
#pragma unroll
      for (int m = 0; m < M; ++m) acc[m] = 0.0;
      auto rows4 = [&](int r, const P (&o)[U][M]) __attribute__((always_inline)) {
        double y[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          double p[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
          for (int m = 0; m < M; ++m)
            if (lane + 64 * m < na) p[m & 3] += (double)o[u][m] * xv[m];
          y[u] = (p[0] + p[2]) + (p[1] + p[3]);
        }
        const double t = cg_trees<U>(y);
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (r + u < r1) {
            const double yu = cg_lane(t, u == 0 ? 0 : u == 1 ? 32 : u == 2 ? 16 : 48);
#pragma unroll
            for (int m = 0; m < M; ++m) acc[m] += (double)o[u][m] * yu;
          }
      };
      P o0[U][M], o1[U][M];
      load(r0, r1, o0);
      for (int r = r0; r < r1; r += 2 * U) {
        if (r + U < r1) load(r + U, r1, o1);
        rows4(r, o0);
        if (r + 2 * U < r1) load(r + 2 * U, r1, o0);
        if (r + U < r1) rows4(r + U, o1);
      }
#pragma unroll
      for (int m = 0; m < M; ++m)
        if (lane + 64 * m < na) cp[(size_t)c * na + lane + 64 * m] = acc[m];
    }
  }
  __syncthreads();
  const double coef = red[0];
  for (int i = tid; i < na; i += CGS_NT) {
    double tot = 0.0;
    if constexpr (GRAM) {
      tot = cp[i];
    } else {
      const int nch = (rows + CG_RCH - 1) / CG_RCH;
      for (int b0 = 0; b0 < nch; b0 += CG_SCH) {
        double a = cp[(size_t)b0 * na + i];
        for (int b = b0 + 1; b < min(nch, b0 + CG_SCH); ++b) a += cp[(size_t)b * na + i];
        tot = b0 == 0 ? a : tot + a;
      }
    }
    const double z = inv_w * tot - coef * mean[i] + shift * diag[i] * v[i];
    out[i] = g ? g[i] - z : z;
  }
  __syncthreads();
}

// sum of a[i] * b[i], bdot's order, in every thread (by the first wave).
__device__ inline double cgs_bdot(const double* a, const double* b, int na, double* red) {
  const int lane = threadIdx.x & 63;
  if (threadIdx.x < 64) {
    double p[4] = {0.0, 0.0, 0.0, 0.0};
    for (int i0 = 0; i0 < na; i0 += 256) {
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int i = i0 + 64 * t + lane;
        if (i < na) p[t] += a[i] * b[i];
      }
    }
    const double s = cg_tree256_wave(p[0], p[1], p[2], p[3]);
    if (lane == 0) red[1] = s;
  }
  __syncthreads();
  const double s = red[1];
  __syncthreads();
  return s;
}

// The whole solve; x_out [na], ctl[1..2] the status (as cg_finish).
template <int M, bool GRAM, class P>
__global__ void __launch_bounds__(CGS_NT) k_cg_small(const P* op, int rows, int na, const double* mean_g,
                                                     const double* diag_g, const double* g_g, double inv_w,
                                                     double shift, double threshold, double pfac, int max_it,
                                                     int diag_scale, double* x_out, int* ctl) {
  extern __shared__ __align__(16) double cgs_lds[];
  double* x = cgs_lds;
  double* r = x + na;
  double* d = r + na;
  double* q = d + na;
  double* mean = q + na;
  double* diag = mean + na;
  double* g = diag + na;
  double* red = g + na;
  double* cp = GRAM ? q : red + 8;  // a Gram product's rows land where its result does
  const int tid = threadIdx.x;
  for (int i = tid; i < na; i += CGS_NT) {
    mean[i] = mean_g[i];
    diag[i] = diag_g[i];
    g[i] = g_g[i];
    x[i] = 0.0;
    r[i] = g[i];
    d[i] = g[i];
  }
  __syncthreads();
  auto apply = [&](const double* v, const double* gv, double* out) {
    cgs_apply<M, GRAM>(op, rows, na, v, mean, diag, gv, inv_w, shift, GRAM ? out : cp, red, out);
  };
  if (diag_scale) {
    apply(x, g, r);
    for (int i = tid; i < na; i += CGS_NT) d[i] = cg_precond(pfac, diag[i], r[i]);
    __syncthreads();
  }
  double delta = cgs_bdot(r, diag_scale ? d : r, na, red);
  long long status = 0;
  for (int iter = 0;; ++iter) {
    if (iter == 0 && !(delta - delta == 0.0)) {
      status = -1;
      break;
    }
    if (iter >= max_it) {
      status = fabs(delta) >= threshold ? -(long long)(max_it + 1) : (long long)iter;
      break;
    }
    if (!(delta - delta == 0.0)) {
      status = -(long long)(iter + 1);
      break;
    }
    if (fabs(delta) < threshold) {
      status = iter;
      break;
    }
    apply(d, nullptr, q);
    const double dq = cgs_bdot(d, q, na, red);
    const double alpha = delta / dq;
    if (!(dq - dq == 0.0) || fabs(dq) < 1.0e-20 || !(alpha - alpha == 0.0)) {
      status = -(long long)(iter + 1);
      break;
    }
    const bool refresh = (iter + 1) % 20 == 0;
    for (int i = tid; i < na; i += CGS_NT) {
      x[i] += alpha * d[i];
      if (!refresh) r[i] -= alpha * q[i];
    }
    __syncthreads();
    if (refresh) apply(x, g, r);
    if (diag_scale) {
      for (int i = tid; i < na; i += CGS_NT) q[i] = cg_precond(pfac, diag[i], r[i]);
      __syncthreads();
    }
    const double* src = diag_scale ? q : r;
    const double dn = cgs_bdot(r, src, na, red);
    const double b = dn / delta;
    if (!(dn - dn == 0.0) || fabs(delta) < 1.0e-20 || !(b - b == 0.0)) {
      status = -(long long)(iter + 1);
      break;
    }
    for (int i = tid; i < na; i += CGS_NT) d[i] = src[i] + b * d[i];
    __syncthreads();
    delta = diag_scale ? dn : delta * b;
  }
  for (int i = tid; i < na; i += CGS_NT) x_out[i] = x[i];
  if (tid == 0) cg_finish(ctl, status);
}

// sum_i prod[i] in bdot's order (256 strided lane partials, the tree), in
// every thread; prod in LDS, 1024 threads.
__device__ inline double cgt_bdot(const double* prod, int na, double* red) {
  const int tid = threadIdx.x;
  if (tid < 256) {
    double p = 0.0;
    for (int i = tid; i < na; i += 256) p += prod[i];
    red[tid] = p;
  }
  __syncthreads();
  if (tid < 64) {
    const double s = cg_tree256_wave(red[tid], red[tid + 64], red[tid + 128], red[tid + 192]);
    if (tid == 0) red[256] = s;
  }
  __syncthreads();
  return red[256];
}

// Rows of the Gram product, G^T v, and coef = mean . v by the last block; one
// wave per row, FP64 accumulation of the FP32 Gram entries, lane-strided
// (the precision form of the SR-CG product: the Gram by FP32 MFMA once, na^2
// per product instead of rows * na).
__global__ void __launch_bounds__(256) k_gram_product(const float* G, int na, const double* v, const double* mean,
                                                      double* out, double* coef, const int* ctl) {
  if (ctl && ctl[CTL_DONE]) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (blockIdx.x == gridDim.x - 1) {
    __shared__ double red[256];
    const double c = block_bdot(mean, v, na, red);
    if (threadIdx.x == 0) *coef = c;
    return;
  }
  const int i = blockIdx.x * 4 + wave;
  if (i >= na) return;
  const float* col = G + (size_t)i * na;
  double acc = 0.0;
#pragma unroll 4
  for (int j = lane; j < na; j += 64) acc += (double)col[j] * v[j];
  acc = cg_tree64(acc);
  if (lane == 0) out[i] = acc;
}

// The part of an iteration behind its product: the superchunk fold into z
// (k_cg_fold2), then, by `stage`,
//   0  q = z, alpha, x += alpha d, r -= alpha q, beta, d = src + beta d, and
//      the head of the next iteration
//   1  (before a residual refresh) q = z, alpha, x += alpha d
//   2  (after it) r = g - z, beta, d, the next head
// (a Gram product is one superchunk).  nsup < 0: the fold went before, in a
// launch of its own, with z in q (stage 2: g - z in r).  The products of a dot
// are formed by all threads and summed in its order by 256 (in LDS, or in
// `prod` past CGT_NMAX).  Guards: a d.q or r.src that is not finite, a d.q or
// delta below 1e-20 in magnitude, an alpha or beta that is not finite end the
// solve with status -(iteration + 1); ctl[CTL_ITER] + j is the iteration.
__global__ void __launch_bounds__(CGT_NT) k_cg_tail(int stage, int j, int na, int nsup, const double* spart,
                                                    const double* mean, const double* diag, const double* g,
                                                    double* coef, double inv_w, double shift, double pfac,
                                                    int diag_scale, int max_it, double threshold, double* x,
                                                    double* r, double* d, double* q, double* prod, double* sc,
                                                    int period, int* ctl) {
  if (ctl[CTL_DONE]) return;
  extern __shared__ __align__(16) double cgt_lds[];
  double* const cgt_prod = na <= CGT_NMAX ? cgt_lds : prod;
  __shared__ double red[257];
  const int tid = threadIdx.x;
  const int iter = ctl[CTL_ITER] + j;
  const double* v = stage == 2 ? x : d;
  if (nsup >= 0) {
    const double cf = coef[0];
    for (int i = tid; i < na; i += CGT_NT) {
      double tot = nsup > 0 ? spart[i] : 0.0;
#pragma unroll 4
      for (int s = 1; s < nsup; ++s) tot += spart[(size_t)s * na + i];
      const double z = inv_w * tot - cf * mean[i] + shift * diag[i] * v[i];
      if (stage == 2) {
        r[i] = g[i] - z;
      } else {
        q[i] = z;
        cgt_prod[i] = d[i] * z;
      }
    }
  } else if (stage != 2) {
#pragma unroll 4
    for (int i = tid; i < na; i += CGT_NT) cgt_prod[i] = d[i] * q[i];
  }
  __syncthreads();
  if (stage != 2) {
    const double dq = cgt_bdot(cgt_prod, na, red);
    const double a = sc[0] / dq;
    if (!(dq - dq == 0.0) || fabs(dq) < 1.0e-20 || !(a - a == 0.0)) {
      if (tid == 0) cg_finish(ctl, -(long long)(iter + 1));
      return;
    }
    for (int i = tid; i < na; i += CGT_NT) {
      x[i] += a * d[i];
      if (stage == 0) r[i] -= a * q[i];
    }
    if (stage == 1) return;
    __syncthreads();
  }
  for (int i = tid; i < na; i += CGT_NT) {
    double s = r[i];
    if (diag_scale) q[i] = s = cg_precond(pfac, diag[i], s);
    cgt_prod[i] = r[i] * s;
  }
  __syncthreads();
  const double dn = cgt_bdot(cgt_prod, na, red);
  const double dl = sc[0];
  const double b = dn / dl;
  if (!(dn - dn == 0.0) || fabs(dl) < 1.0e-20 || !(b - b == 0.0)) {
    if (tid == 0) cg_finish(ctl, -(long long)(iter + 1));
    return;
  }
  for (int i = tid; i < na; i += CGT_NT) d[i] = (diag_scale ? q[i] : r[i]) + b * d[i];
  __syncthreads();
  if (tid == 0) {
    const double delta = diag_scale ? dn : dl * b;
    sc[0] = delta;
    cg_head(iter + 1, max_it, threshold, delta, ctl);
    if (j == period - 1) ctl[CTL_ITER] += period;
  }
}

}  // namespace mvmc_hip
