// Register-resident skew-symmetric Pfaffian + inverse of one plane per
// workgroup, for n <= RR_NMAX: the C PfaPack order of dsktf2
// (crates/pfapack/src/ltl.rs:61-191, :683-705), utu2pfa (utu2.rs:52-93)
// and utu2inv (utu2.rs:338-513 with the scalar trtri / trmm forms of
// backend.rs:233-300), every element receiving exactly the operation
// sequence of that order (bit-identical to the sequential loops; built with
// -ffp-contract=off).
//
// For the sizes whose triangle does not fit a CU's LDS several times
// (pfinv_lds.h serves the smaller ones): T x T threads, thread (a, b) =
// (tid % T, tid / T) owns the elements (i, j) = (a + T ri, b + T cj) of the
// plane's upper triangle and keeps them in registers.
//
// What bounds it is the dependent chain of n elimination steps, so the
// design cuts what a step waits for:
//   - one exchange through LDS and one barrier per step.  The pivot column
//     of a step is the y column of the step before, so its search, the
//     pivot's reciprocal and the x column come from the copy already in LDS,
//     the swapped column is staged straight into y, and every wave searches
//     the pivot by itself (16 waves per plane searching cost more than they
//     save: n = 224 0.6x; 4 waves, T = 16, it is);
//   - the block of the step's column picks one of R code bodies whose slots
//     and bounds are compile-time constants (no per-element tests inside).
// Measured: 2048 planes of n = 144 7470 -> 3320 us (before: the panel-delayed
// kernel), 1024 of n = 224 8580 -> 7200 us, complex 768 of n = 144 4080 ->
// 3190 us and of n = 160 4720 -> 4260 us (before: 1024 threads a plane, two
// barriers a step).
#pragma once
#include "common.h"

// on the kernel's lambdas: a call would put the register slots into memory
#define RR_INLINE __attribute__((always_inline))

namespace mvmc_hip {

constexpr int RR_NMAX = 224;  // largest n
constexpr int RR_NFULL = 64;  // largest n of utu2inv's small-matrix path (pfinv_lds.h)

// Orders the LDS traffic of the T x T workgroup: a barrier, or for the
// single wave of T = 8 (pfinv_lds.h), whose LDS operations complete in order,
// only a fence for the compiler.
template <int T>
__device__ __forceinline__ void rr_sync() {
  if constexpr (T == 8) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  } else {
    __syncthreads();
  }
}

// Keeps the compiler from merging the tails of sibling branches: merged code
// would index the register slots by a run-time choice, i.e. through memory.
#define RR_APART(tag) asm volatile("; branch %0" ::"n"(tag))

// Calls f.template operator()<k>() for the run-time k of [LO, HI).
template <int LO, int HI, class F>
__device__ __forceinline__ void rr_case(int k, F&& f) {
  if constexpr (LO + 1 == HI) {
    f.template operator()<LO>();
    RR_APART(LO);
  } else {
    constexpr int M = (LO + HI) / 2;
    if (k < M) rr_case<LO, M>(k, f);
    else rr_case<M, HI>(k, f);
  }
}

// for (X = LO; X < HI; ++X) with X a compile-time constant in the body:
// RR_FOR(X, LO, HI) { ... };  The register slots are indexed only by such
// constants from the start: left to the loop unroller, they end in memory.
template <int LO, int HI>
struct RrRange {
  template <class F>
  __device__ __forceinline__ void operator<<(F&& f) const {
    if constexpr (LO < HI) {
      f.template operator()<LO>();
      RrRange<LO + 1, HI>{} << f;
    }
  }
};
#define RR_FOR(X, LO, HI) RrRange<(LO), (HI)>{} << [&]<int X>() RR_INLINE

// Maximum over the wave's lanes (no NaN), in every lane.
__device__ __forceinline__ double rr_wave_max(double x) {
#define RR_DPP_MAX(ctrl)                                                                             \
  do {                                                                                               \
    const int lo_ = __double2loint(x), hi_ = __double2hiint(x);                                      \
    const double y_ = __hiloint2double(__builtin_amdgcn_update_dpp(hi_, hi_, ctrl, 0xf, 0xf, false), \
                                       __builtin_amdgcn_update_dpp(lo_, lo_, ctrl, 0xf, 0xf, false)); \
    x = y_ > x ? y_ : x;                                                                             \
  } while (0)
  RR_DPP_MAX(0x111);  // row_shr:1, 2, 4, 8: lane 15 of each row of 16 has the row's maximum
  RR_DPP_MAX(0x112);
  RR_DPP_MAX(0x114);
  RR_DPP_MAX(0x118);
  RR_DPP_MAX(0x142);  // row_bcast:15, row_bcast:31: lane 63 has the wave's
  RR_DPP_MAX(0x143);
#undef RR_DPP_MAX
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), 63),
                          __builtin_amdgcn_readlane(__double2loint(x), 63));
}

// LDS of one plane.  `vec`: the step vectors (two sets by step parity: a fast
// wave may write the next step's while a slow one still reads this step's),
// reused as the row blocks of the product and of the output.
constexpr int rr_vl(int T, int R) { return (T * R + 63) / 64 * 64; }  // padded vector length
// row stride of the T-row blocks: T lanes of a row beside the next row's
constexpr int rr_ldb(int T, int R) { return rr_vl(T, R) + T; }
// scalars of `vec`: 2 y columns, then per set x, u, r1, r2
constexpr int rr_vec_len(int T, int R) {
  const int step = 10 * rr_vl(T, R);
  const int blocks = 2 * T * rr_ldb(T, R);
  return step > blocks ? step : blocks;
}

template <class S>
struct RrLdsT {
  S* vec;
  S* sup;          // the superdiagonal A(i, i+1) after the LTL
  S *rneg, *rpos;  // complex solve: reciprocals of -vt[i] and vt[i]
  S* sa;           // [1] the Pfaffian
  int* finv;       // inverse of the output permutation
  double* sd;      // [16] max |a|^2 per wave
};
using RrLds = RrLdsT<double>;

template <class S, bool RECIP>
__host__ __device__ inline size_t rr_lds_bytes(int T, int R, int n) {
  const int nw = T * T / 64;
  return rnd16((size_t)rr_vec_len(T, R) * sizeof(S)) + rnd16((size_t)n * sizeof(S)) * (RECIP ? 3 : 1) + 16 +
         rnd16((size_t)n * 4) + rnd16((size_t)nw * 8);
}

template <class S, bool RECIP, int T, int R, class Carver>
__device__ inline RrLdsT<S> carve_rr(Carver& c, int n) {
  RrLdsT<S> L;
  L.vec = c.template take<S>(rr_vec_len(T, R));
  L.sup = c.template take<S>(n);
  L.rneg = RECIP ? c.template take<S>(n) : nullptr;
  L.rpos = RECIP ? c.template take<S>(n) : nullptr;
  L.sa = c.template take<S>(1);
  L.finv = c.template take<int>(n);
  L.sd = c.template take<double>(T * T / 64);
  return L;
}

// Scratch in global memory per workgroup, in scalars: M and C.
__host__ __device__ inline size_t rr_scratch_len(int n) { return (size_t)2 * n * n; }

// Slot of block (ri, cj) of the packed upper block triangle (cj >= ri).
template <int R>
__host__ __device__ constexpr int rr_slot(int ri, int cj) {
  return ri * R - ri * (ri - 1) / 2 + (cj - ri);
}

// C IDAMAX order of the pivot search: first index of the largest |x|; a NaN
// wins only at index 0 (the sequential scan starts from it).
__device__ inline double rr_key(double v, int i) {
  if (v != v) return i == 0 ? INFINITY : -1.0;
  return v;
}

// Arithmetic of the real planes (dsktf2 / utu2 with real operands): every
// operation is the one the sequential loops perform.
struct RrReal {
  using S = double;
  static constexpr bool kRecip = false;  // the solve divides by vt
  static __device__ __forceinline__ S zero() { return 0.0; }
  static __device__ __forceinline__ S one() { return 1.0; }
  static __device__ __forceinline__ S neg(S x) { return -x; }
  static __device__ __forceinline__ S add(S x, S y) { return x + y; }
  static __device__ __forceinline__ S sub(S x, S y) { return x - y; }
  static __device__ __forceinline__ S mul(S x, S y) { return x * y; }
  static __device__ __forceinline__ double mag2(S x) { return x * x; }
  static __device__ __forceinline__ double key(S x, int i) { return rr_key(fabs(x), i); }
  __device__ __forceinline__ S alpha(S pivot) const { return 1.0 / pivot; }
  // rank-2 update of one element: (c + x_i t1) - y_i t2
  static __device__ __forceinline__ S update(S c, S xi, S yi, S t1, S t2) { return (c + xi * t1) - yi * t2; }
  __device__ __forceinline__ S scale(S x, S alpha) const { return x * alpha; }
  static __device__ __forceinline__ S sign(bool neg) { return neg ? (0.0 - 1.0) : 1.0; }
  static __device__ __forceinline__ bool finite(S x) { return isfinite(x); }
  // solve: num / -vt (forward), num / vt (backward)
  static __device__ __forceinline__ S div_negvt(S num, S vt, S) { return num / -vt; }
  static __device__ __forceinline__ S div_vt(S num, S vt, S) { return num / vt; }
  static __device__ __forceinline__ S recip(S x) { return 1.0 / x; }
  static __device__ __forceinline__ S readlane(S x, int l) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), l),
                            __builtin_amdgcn_readlane(__double2loint(x), l));
  }
};

// One plane.  src(i, j) gives A(i, j) (any i, j < n).  On exit: info (0 ok,
// k > 0 zero pivot at 1-based row k, -1 non-finite Pfaffian), pf (the
// Pfaffian; on a zero pivot not formed), and for info == 0 the plane `out`
// (column-major, element (r, c) at r + c n) holds sign * A^{-1} (and out32,
// if set, the same rounded to FP32).  allzero (when check_zero) reports
// max |a|^2 < 1e-28 over the whole plane, in which case nothing else is
// done.  gs: rr_scratch_len scalars of global scratch.  Every thread of the
// T x T workgroup (blockDim.x == T * T) calls it; the results are uniform.
// T (R - 1) < n <= T R.
template <int T, int R, class Ar, class Src>
__device__ __forceinline__ void rr_pfinv(const Ar& ar, Src src, int n, typename Ar::S* out, float* out32, double sign,
                                         typename Ar::S* gs, RrLdsT<typename Ar::S>& L, typename Ar::S& pf, int& info,
                                         bool check_zero, bool& allzero) {
  using S = typename Ar::S;
  constexpr int NS = R * (R + 1) / 2;
  constexpr int NT = T * T, VL = rr_vl(T, R), LDB = rr_ldb(T, R), Q = VL / 64;
  constexpr int JC = (T * R + NT - 1) / NT;  // columns per thread where a thread owns whole columns
  // Complex planes of 10 blocks a side fill 220 of a thread's 512 registers
  // with slots; with a step's x and y of all rows beside them the kernel
  // spilled 513 (n = 152, 256 planes: 2064 us, where 1024 threads a plane had
  // taken 1480).  There the update goes by groups of RG block rows: 1385 us.
  constexpr bool TIGHT = sizeof(S) == 16 && R >= 10;
  constexpr int RG = 4;
  const int tid = threadIdx.x, lane = tid & 63;
  const int a0 = tid % T, b0 = tid / T;
  // copies of (a, b) the compiler cannot prove loop-invariant: the index
  // arithmetic of a step is formed in the step instead of being kept live
  // across the elimination (the registers hold the slots)
  int a = a0, b = b0;
#define RR_FRESH()                       \
  do {                                   \
    a = a0;                              \
    b = b0;                              \
    asm volatile("" : "+v"(a), "+v"(b)); \
  } while (0)
  S c[NS];
#define RC(ri, cj) c[rr_slot<R>(ri, cj)]
#ifdef MVMC_PHASE_CLOCKS
  long long rr_t0 = __builtin_readcyclecounter(), rr_ph[12] = {};
#define RR_PHASE(k)                                         \
  do {                                                      \
    const long long t_ = __builtin_readcyclecounter();      \
    rr_ph[k] += t_ - rr_t0;                                 \
    rr_t0 = t_;                                             \
  } while (0)
#else
#define RR_PHASE(k) \
  do {              \
  } while (0)
#endif
  // ---- gather (and the all-zero guard, pfaffian.rs:884-890: the plane is skew, so the upper half decides) ----
  double mx = 0.0;
RR_FOR(ri, 0, R) {
RR_FOR(cj, ri, R) {
      const int i = a + T * ri, j = b + T * cj;
      S x = Ar::zero();
      if (i < n && j < n && i <= j) {
        x = src(i, j);
        mx = fmax(mx, Ar::mag2(x));
      }
      RC(ri, cj) = x;
    };
  };
  if (check_zero) {
    mx = rr_wave_max(mx);
    if (lane == 0) L.sd[tid >> 6] = mx;
    __syncthreads();
    double m = 0.0;
    for (int k = 0; k < NT / 64; ++k) m = fmax(m, L.sd[k]);
    allzero = m < 1.0e-28;
    __syncthreads();
    if (allzero) return;
  } else {
    allzero = false;
  }
  S* const y0 = L.vec;
  auto setv = [&](int par, int k) { return L.vec + (2 + 4 * par + k) * VL; };

  RR_PHASE(0);
  // ---- dsktf2: k0 = n-1 .. 1 ----
  // first largest key of yv[0 .. m), each wave by itself
  auto pivot = [&](const S* yv, int m, int& kp, bool& zero) RR_INLINE {
    double key[Q], best = -2.0;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int i = lane + 64 * q;
      key[q] = i < m ? Ar::key(yv[i], i) : -2.0;
      best = key[q] > best ? key[q] : best;
    }
    best = rr_wave_max(best);
    kp = 0;
#pragma unroll
    for (int q = Q - 1; q >= 0; --q) {
      const unsigned long long hit = __ballot(key[q] == best);
      if (hit) kp = 64 * q + (int)__builtin_ctzll(hit);
    }
    zero = best == 0.0;
  };
  info = 0;
  // the last column, the first pivot column
  {
    const int k = n - 1;
    if (b == k % T)
      rr_case<0, R>(k / T, [&]<int K>() RR_INLINE {
RR_FOR(ri, 0, K + 1) { y0[a + T * ri] = RC(ri, K);
        };
      });
  }
  rr_sync<T>();
  int f[JC];  // the output permutation: position r holds index f(r); the swaps composed as they come
#pragma unroll
  for (int u = 0; u < JC; ++u) f[u] = tid + NT * u;
  bool neg = false;  // parity of the interchanges
  int kp = 0;
  bool zero = false;
  pivot(y0, n - 1, kp, zero);
  S xk = y0[kp];
  for (int k0 = n - 1; k0 >= 1; --k0) {
    const int kk0 = k0 - 1, par = k0 & 1;  // n is even: k0 = n - 1 reads y0, writes y1
    RR_FRESH();
    if (zero) {  // zero pivot column: the plane has no Pfaffian form to go on with
      info = kk0 + 1;
      break;
    }
    if (tid == 0) L.sup[kk0] = xk;
    if (kp != kk0) {
      neg = !neg;
#pragma unroll
      for (int u = 0; u < JC; ++u) f[u] = f[u] == kk0 ? kp : f[u] == kp ? kk0 : f[u];
    }
    if (kk0 == 0) break;
    const S* yp = L.vec + (par ? 0 : VL);
    S* yn = L.vec + (par ? VL : 0);
    S* xs = setv(par, 0);
    S* us = setv(par, 1);
    S* r1 = setv(par, 2);
    S* r2 = setv(par, 3);
    const int K0 = kk0 / T, kb = kk0 % T;
    // stage: x = column k0 with its rows kk0 and kp interchanged (column k0
    // is y of the step before), u = column kk0, y = column kk0 after the
    // interchange of rows/columns kk0 and kp in the upper triangle (with the
    // sign twiddles), r1 / r2 = rows kp / kk0 in the columns >= k0
#pragma unroll
    for (int q = 0; q < (VL + NT - 1) / NT; ++q) {
      const int i = tid + NT * q;
      if (i < kk0) xs[i] = yp[i == kp ? kk0 : i];
    }
    if (kp == kk0) {
      rr_case<0, R>(K0, [&]<int K>() RR_INLINE {
        if (b == kb) {
RR_FOR(ri, 0, K + 1) { yn[a + T * ri] = RC(ri, K);
          };
        }
      });
    } else {
      rr_case<0, R>(K0, [&]<int K>() RR_INLINE {
        if (b == kb) {
RR_FOR(ri, 0, K + 1) {
            const int i = a + T * ri;
            us[i] = RC(ri, K);
            if (i == kp) yn[i] = Ar::neg(RC(ri, K));
          };
        }
        if (a == kb) {
RR_FOR(cj, K, R) { r2[b + T * cj] = RC(K, cj);
          };
        }
      });
      const int kpb = kp % T;
      rr_case<0, R>(kp / T, [&]<int P>() RR_INLINE {
        if (b == kpb) {
RR_FOR(ri, 0, P + 1) {
            if (ri < P || a < kpb) yn[a + T * ri] = RC(ri, P);
          };
        }
        if (a == kpb) {
RR_FOR(cj, P, R) {
            const int j = b + T * cj;
            if (cj > P || b > kpb) {
              if (j < kk0) yn[j] = Ar::neg(RC(P, cj));
              else r1[j] = RC(P, cj);
            }
          };
        }
      });
    }
    RR_PHASE(1);  // stage
    rr_sync<T>();
    const S alpha = ar.alpha(xk);
    // the next step's pivot column is y, which this step's update leaves alone
    const int kpc = kp;
    pivot(yn, kk0, kp, zero);
    xk = yn[kp];
    RR_PHASE(2);
    if (kpc != kk0) {
      const int kpb = kpc % T;
      rr_case<0, R>(kpc / T, [&]<int P>() RR_INLINE {
        if (b == kpb) {
RR_FOR(ri, 0, P + 1) {
            if (ri < P || a < kpb) RC(ri, P) = us[a + T * ri];
          };
        }
        if (a == kpb) {
RR_FOR(cj, P, R) {
            const int j = b + T * cj;
            const S w = j < kk0 ? Ar::neg(us[j]) : r2[j];
            if (cj > P || b > kpb) RC(P, cj) = w;  // column kk0 follows below
          };
        }
      });
    }
    RR_PHASE(3);
    rr_case<0, R>(K0, [&]<int K>() RR_INLINE {
      if constexpr (!TIGHT) {
      S xi[K + 1], yi[K + 1];
RR_FOR(ri, 0, K + 1) {
        xi[ri] = xs[a + T * ri];
        yi[ri] = yn[a + T * ri];
      };
      if (kpc != kk0) {
        if (b == kb) {
RR_FOR(ri, 0, K + 1) {
            if (ri < K || a < kb) RC(ri, K) = yi[ri];
          };
        }
        if (a == kb) {
RR_FOR(cj, K, R) {
            if (cj > K || b > kb) RC(K, cj) = r1[b + T * cj];
          };
        }
      }
      // rank-2 update of the leading kk0 x kk0 block (elements on and below
      // the diagonal of a diagonal block are never read)
RR_FOR(cj, 0, K + 1) {
        const S yj = yn[b + T * cj], xj = xs[b + T * cj];
        const S t1 = Ar::mul(alpha, yj), t2 = Ar::mul(alpha, xj);
        if (cj < K || b < kb) {
RR_FOR(ri, 0, cj + 1) { RC(ri, cj) = Ar::update(RC(ri, cj), xi[ri], yi[ri], t1, t2);
          };
        }
      };
      // column k0 scaled (its rows are x)
      if (kb + 1 < T) {
        if (b == kb + 1) {
RR_FOR(ri, 0, K + 1) {
            if (ri < K || a < kb) RC(ri, K) = ar.scale(xi[ri], alpha);
          };
        }
        RR_APART(K + 100);
      } else if constexpr (K + 1 < R) {
        if (b == 0) {
RR_FOR(ri, 0, K + 1) {
            if (ri < K || a < kb) RC(ri, K + 1) = ar.scale(xi[ri], alpha);
          };
        }
      }
      } else {
        // the same by groups of RG block rows
        RR_FOR(h, 0, (K + RG) / RG) {
          constexpr int R0 = h * RG, R1 = R0 + RG < K + 1 ? R0 + RG : K + 1;
          S xi[R1 - R0], yi[R1 - R0];
          RR_FOR(ri, R0, R1) {
            xi[ri - R0] = xs[a + T * ri];
            yi[ri - R0] = yn[a + T * ri];
          };
          if (kpc != kk0) {
            if (b == kb) {
              RR_FOR(ri, R0, R1) {
                if (ri < K || a < kb) RC(ri, K) = yi[ri - R0];
              };
            }
            if (R1 == K + 1 && a == kb) {
              RR_FOR(cj, K, R) {
                if (cj > K || b > kb) RC(K, cj) = r1[b + T * cj];
              };
            }
          }
          RR_FOR(cj, R0, K + 1) {
            const S yj = yn[b + T * cj], xj = xs[b + T * cj];
            const S t1 = Ar::mul(alpha, yj), t2 = Ar::mul(alpha, xj);
            if (cj < K || b < kb) {
              RR_FOR(ri, R0, (cj + 1 < R1 ? cj + 1 : R1)) {
                RC(ri, cj) = Ar::update(RC(ri, cj), xi[ri - R0], yi[ri - R0], t1, t2);
              };
            }
          };
          if (kb + 1 < T) {
            if (b == kb + 1) {
              RR_FOR(ri, R0, R1) {
                if (ri < K || a < kb) RC(ri, K) = ar.scale(xi[ri - R0], alpha);
              };
            }
            RR_APART(K + 100 + 1000 * h);
          } else if constexpr (K + 1 < R) {
            if (b == 0) {
              RR_FOR(ri, R0, R1) {
                if (ri < K || a < kb) RC(ri, K + 1) = ar.scale(xi[ri - R0], alpha);
              };
            }
          }
        };
      }
    });
    RR_PHASE(4);
  }
  if (info != 0) {
    pf = Ar::zero();
    __syncthreads();
    return;
  }
  __syncthreads();
  RR_PHASE(4);
  // ---- utu2pfa: product of A(i, i+1), i even, sign by the count of moves ----
  if (tid == 0) {
    S p = Ar::one();
    int i = 0;
    for (; i + 16 <= n; i += 16) {
      S v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = L.sup[i + 2 * u];
#pragma unroll
      for (int u = 0; u < 8; ++u) p = Ar::mul(p, v[u]);
    }
    for (; i + 1 < n; i += 2) p = Ar::mul(p, L.sup[i]);
    L.sa[0] = Ar::mul(Ar::sign(neg), p);
  }
  if constexpr (Ar::kRecip)
    for (int i = tid; i + 1 < n; i += NT) {
      const S vt = Ar::neg(L.sup[i]);
      L.rneg[i] = Ar::recip(Ar::neg(vt));
      L.rpos[i] = Ar::recip(vt);
    }
  __syncthreads();
  pf = L.sa[0];
  if (!Ar::finite(pf)) {
    info = -1;
    __syncthreads();
    return;
  }
#pragma unroll
  for (int u = 0; u < JC; ++u)
    if (tid + NT * u < n) L.finv[f[u]] = tid + NT * u;

  RR_PHASE(5);
  // ---- utu2inv (its panel path, n > 64) ----
  // trtri('U','U') on B(i, j) = A(i, j+1), 0 <= i < j <= n-2: at step k the
  // column k of the inverse is final (Bn(i, k) = -acc(i, k), i < k) and
  // every acc(i, j), i < k < j, adds Bn(i, k) B(k, j) with row k of B still
  // as factored (no earlier step writes it): each element takes its k in
  // ascending order, as the row-chain loops do.
  for (int k = 1; k <= n - 2; ++k) {
    RR_FRESH();
    S* U = setv(k & 1, 0);   // column k of the inverse, rows < k
    S* Bk = setv(k & 1, 1);  // row k of B by plane column (> k + 1)
    const int kb = k % T;
    rr_case<0, R>(k / T, [&]<int K>() RR_INLINE {
      if (kb + 1 < T) {
        if (b == kb + 1) {
RR_FOR(ri, 0, K + 1) {
            const S x = Ar::neg(RC(ri, K));
            U[a + T * ri] = x;
            if (ri < K || a < kb) RC(ri, K) = x;
          };
        }
        RR_APART(K + 200);
      } else if constexpr (K + 1 < R) {
        if (b == 0) {
RR_FOR(ri, 0, K + 1) {
            const S x = Ar::neg(RC(ri, K + 1));
            U[a + T * ri] = x;
            if (ri < K || a < kb) RC(ri, K + 1) = x;
          };
        }
      }
      if (a == kb) {
RR_FOR(cj, K, R) { Bk[b + T * cj] = RC(K, cj);
        };
      }
    });
    rr_sync<T>();
    if (k <= n - 3)
      rr_case<0, R>(k / T, [&]<int K>() RR_INLINE {
        S ui[K + 1];
RR_FOR(ri, 0, K + 1) { ui[ri] = U[a + T * ri];
        };
RR_FOR(cj, K, R) {
          const S bj = Bk[b + T * cj];
          if (cj > K + 1 || b + T * cj >= k + 2) {
RR_FOR(ri, 0, K) { RC(ri, cj) = Ar::add(RC(ri, cj), Ar::mul(ui[ri], bj));
            };
            if (a < kb) RC(K, cj) = Ar::add(RC(K, cj), Ar::mul(ui[K], bj));
          }
        };
      });
  }
  RR_PHASE(6);
  // M (unit upper, M(i, j) = Bn(i, j) for i < j <= n-2, M(i, n-1) = 0 for
  // i < n-1), row-major in gs
  S* gm = gs;
  S* gc = gs + (size_t)n * n;
  RR_FRESH();
RR_FOR(ri, 0, R) {
RR_FOR(cj, ri, R) {
      const int i = a + T * ri, jj = b + T * cj;
      if (i + 1 < jj && jj < n) {
        gm[(size_t)i * n + (jj - 1)] = RC(ri, cj);
      }
    };
  };
  __syncthreads();
  auto mval = [&](int i, int j) RR_INLINE -> S {  // M(i, j), j < n
    if (j <= i) return j == i ? Ar::one() : Ar::zero();
    if (j == n - 1) return Ar::zero();
    return gm[(size_t)i * n + j];
  };
  RR_PHASE(7);
  // skew-tridiagonal solve T C = M (vt[i] = -A(i, i+1) = -sup[i]), a thread
  // per column, its two chains side by side:
  //   forward   C(1) = M(0) / -vt[0]; C(i+1) = (M(i) - C(i-1) vt[i-1]) / -vt[i], i even
  //   backward  C(n-2) = M(n-1) / vt[n-2]; C(i-1) = (M(i) + C(i+1) vt[i]) / vt[i-1], i odd descending
  // The forward chain fills the odd rows of C, the backward one the even
  // rows: the upper part to gc row-major, M read ahead.
#pragma unroll 1
  for (int u = 0; u < JC; ++u) {
    const int j = tid + NT * u;
    if (j < n) {
      // step s of the chains: forward row 2 s + 1 from M row 2 s,
      // backward row n - 2 - 2 s from M row n - 1 - 2 s; M of MB steps
      // loaded together, a batch ahead
      constexpr int MB = 4;
      const int steps = n / 2;
      S mf[MB], mb[MB], pfw = Ar::zero(), pbw = Ar::zero();
      auto fetch = [&](int s0, S (&vf)[MB], S (&vb)[MB]) RR_INLINE {
#pragma unroll
        for (int t = 0; t < MB; ++t) {
          vf[t] = s0 + t < steps ? mval(2 * (s0 + t), j) : Ar::zero();
          vb[t] = s0 + t < steps ? mval(n - 1 - 2 * (s0 + t), j) : Ar::zero();
        }
      };
      fetch(0, mf, mb);
#pragma unroll 1
      for (int s0 = 0; s0 < steps; s0 += MB) {
        S nf[MB], nb[MB];
        fetch(s0 + MB, nf, nb);
#pragma unroll
        for (int t = 0; t < MB; ++t) {
          const int s = s0 + t;
          if (s < steps) {
            const int i = 2 * s, k = n - 1 - 2 * s;
            const S vti = Ar::neg(L.sup[i]), vtm = Ar::neg(L.sup[k - 1]);
            S nu = mf[t], nv = mb[t];
            if (s > 0) {
              nu = Ar::sub(nu, Ar::mul(pfw, Ar::neg(L.sup[i - 1])));
              nv = Ar::add(nv, Ar::mul(pbw, Ar::neg(L.sup[k])));
            }
            pfw = Ar::div_negvt(nu, vti, Ar::kRecip ? L.rneg[i] : vti);
            pbw = Ar::div_vt(nv, vtm, Ar::kRecip ? L.rpos[k - 1] : vtm);
            if (i + 1 < j) gc[(size_t)(i + 1) * n + j] = pfw;
            if (k - 1 < j) gc[(size_t)(k - 1) * n + j] = pbw;
          }
        }
#pragma unroll
        for (int t = 0; t < MB; ++t) {
          mf[t] = nf[t];
          mb[t] = nb[t];
        }
      }
    }
  }
  __syncthreads();
  RR_FRESH();
RR_FOR(ri, 0, R) {
RR_FOR(cj, ri, R) {
      const int i = a + T * ri, j = b + T * cj;
      RC(ri, cj) = (i < j && j < n) ? gc[(size_t)i * n + j] : Ar::zero();
    };
  };
  RR_PHASE(8);
  // product C'(i, j) = C(i, j) + sum_{k < i} M(k, i) C(k, j), k ascending,
  // C as solved, of the upper part (the lower follows by skew
  // symmetry): k block by k block, T rows of M and C from gs through LDS.
  S* mb = L.vec;
  S* cb = L.vec + T * LDB;
#pragma unroll 1
  for (int kb = 0; kb < R; ++kb) {
    RR_FRESH();
    // rows kb T + b of M and C, columns a + T cj
    const int k = kb * T + b;
#pragma unroll 1
    for (int cj = kb; cj < R; ++cj) {
      const int j = a + T * cj;
      const bool in = k < j && j < n;
      mb[b * LDB + j] = in ? mval(k, j) : Ar::zero();
      cb[b * LDB + j] = in ? gc[(size_t)k * n + j] : Ar::zero();
    }
    __syncthreads();
    rr_case<0, R>(kb, [&]<int K>() RR_INLINE {
#pragma unroll 1
      for (int kk = 0; kk < T; ++kk) {
        S mi[R], cjv[R];
RR_FOR(r, K, R) {
          mi[r] = mb[kk * LDB + a + T * r];
          cjv[r] = cb[kk * LDB + b + T * r];
        };
RR_FOR(cj, K, R) {
RR_FOR(ri, K + 1, cj + 1) { RC(ri, cj) = Ar::add(RC(ri, cj), Ar::mul(mi[ri], cjv[cj]));
          };
          if (kk < a) RC(K, cj) = Ar::add(RC(K, cj), Ar::mul(mi[K], cjv[cj]));
        };
      }
    });
    __syncthreads();
  }
  RR_PHASE(9);
  // output: out(r, c) = sign * F(f(r), f(c)), F = the skew completion of C' (0
  // on the diagonal).  T columns of F at a time through LDS, each written as
  // one permuted column of out.
  {
    S* ob = L.vec;
#pragma unroll 1
    for (int blk = 0; blk < R; ++blk) {
      RR_FRESH();
      rr_case<0, R>(blk, [&]<int K>() RR_INLINE {
RR_FOR(ri, 0, K) { ob[b * LDB + a + T * ri] = RC(ri, K);
        };
        if (a < b) {
          ob[b * LDB + a + T * K] = RC(K, K);
          ob[a * LDB + b + T * K] = Ar::neg(RC(K, K));
        } else if (a == b) {
          ob[a * LDB + a + T * K] = Ar::zero();
        }
RR_FOR(cj, K + 1, R) { ob[a * LDB + b + T * cj] = Ar::neg(RC(K, cj));
        };
      });
      rr_sync<T>();
      const int v1 = min(T, n - T * blk);
#pragma unroll 1
      for (int v = 0; v < v1; ++v) {
        const size_t col = (size_t)L.finv[T * blk + v] * n;
#pragma unroll
        for (int u = 0; u < JC; ++u) {
          const int r = tid + NT * u;
          if (r < n) {
            S x = ob[v * LDB + f[u]];
            if (sign != 1.0) x = Ar::neg(x);
            out[col + r] = x;
            if constexpr (sizeof(S) == sizeof(double))
              if (out32) out32[col + r] = (float)x;
          }
        }
      }
      rr_sync<T>();
    }
  }
  __syncthreads();
  RR_PHASE(10);
#ifdef MVMC_PHASE_CLOCKS
  if (tid == 0 && blockIdx.x == 0)
    printf("rr n=%d cycles: gather %lld ltl stage %lld pivot %lld swap %lld update %lld pf %lld trtri %lld mwrite %lld "
           "solve %lld product %lld out %lld\n",
           n, rr_ph[0], rr_ph[1], rr_ph[2], rr_ph[3], rr_ph[4], rr_ph[5], rr_ph[6], rr_ph[7], rr_ph[8], rr_ph[9],
           rr_ph[10]);
#endif
#undef RR_PHASE
#undef RC
#undef RR_FRESH
}

}  // namespace mvmc_hip
