// Skew-symmetric Pfaffian + inverse of one plane per wave, the plane's upper
// triangle held in LDS, for n <= LP_NMAX: the C PfaPack order of dsktf2
// (crates/pfapack/src/ltl.rs:61-191, :683-705), utu2pfa (utu2.rs:52-93) and
// utu2inv (utu2.rs:338-513 with the scalar trtri / trmm forms of
// backend.rs:233-300), every element receiving exactly the operation
// sequence of that order (bit-identical to the sequential loops; built with
// -ffp-contract=off).
//
// What bounds it is the dependent chain of n elimination steps, each a
// pivot search, an interchange of two rows/columns anywhere in the plane and
// a rank-2 update.  One wave per plane needs no barrier (its LDS operations
// complete in order) and a CU runs several planes, which fills the chain's
// waits.  In LDS the interchange is one gather and one scatter of the two
// vectors, a lane per position and no branches, whichever pivot comes up.
// The triangle is stored in 8 x 8 blocks, element (a, b) of a block at
// a + 8 b = its lane, so the update reads and writes whole blocks at
// constant offsets, without bank conflicts; the block of the step's column
// picks one of R code bodies that hold only the blocks in use.  The product
// of the inverse is the one phase with enough work per element to want
// registers: there lane (a, b) holds the elements (a + 8 ri, b + 8 cj).
// Measured against a workgroup of 256 threads with barriers (n <= 64, the
// plane in registers) and a panel-delayed kernel (above): 4096 planes of
// n = 16 142 -> 39 us, 8192 of n = 64 3100 -> 820 us, 1777 of n = 66
// 1340 -> 380 us and of n = 98 2950 -> 1380 us; a step of n = 64 is 2500
// cycles (interchange and reciprocal 1150, update 1280, search 80), against
// 5000 with the plane in the wave's registers.
#pragma once
#include "pfinv_rr.h"

namespace mvmc_hip {

constexpr int LP_NMAX = 104;  // largest n (R = 13 blocks per side, three planes in a CU's LDS)
constexpr int LP_KB = 4;      // rows of C staged at a time by the product

// Scalar offset of block (ri, cj), ri <= cj, of the upper triangle.
__host__ __device__ constexpr int lp_blk(int ri, int cj) { return (cj * (cj + 1) / 2 + ri) * 64; }

template <class S>
struct LpPair {
  S a, b;
};

// LDS of one plane.
template <class S>
struct LpLds {
  S* m;            // the triangle; later the output columns
  S* vec;          // {x, y} and {t1, t2} of a step; later the rows of C
  S* sup;          // the superdiagonal A(i, i+1) after the LTL
  S *rneg, *rpos;  // complex solve: reciprocals of -vt[i] and vt[i]
  int* finv;       // inverse of the output permutation
};

constexpr int lp_m_len(int R) { return lp_blk(0, R) > 8 * rr_ldb(8, R) ? lp_blk(0, R) : 8 * rr_ldb(8, R); }
constexpr int lp_vec_len(int R) { return 32 * R > LP_KB * rr_ldb(8, R) ? 32 * R : LP_KB * rr_ldb(8, R); }

template <class S>
__host__ __device__ inline size_t lp_lds_bytes(int R, bool recip) {
  return rnd16((size_t)lp_m_len(R) * sizeof(S)) + rnd16((size_t)lp_vec_len(R) * sizeof(S)) +
         rnd16((size_t)8 * R * sizeof(S)) * (recip ? 3 : 1) + rnd16((size_t)8 * R * 4);
}

template <class S, bool RECIP, int R, class Carver>
__device__ inline LpLds<S> carve_lp(Carver& c) {
  LpLds<S> L;
  L.m = c.template take<S>(lp_m_len(R));
  L.vec = c.template take<S>(lp_vec_len(R));
  L.sup = c.template take<S>(8 * R);
  L.rneg = RECIP ? c.template take<S>(8 * R) : nullptr;
  L.rpos = RECIP ? c.template take<S>(8 * R) : nullptr;
  L.finv = c.template take<int>(8 * R);
  return L;
}

// Scratch in global memory per workgroup, in scalars: the solved C.
__host__ __device__ inline size_t lp_scratch_len(int n) { return (size_t)n * n; }

// Arguments and results as rr_pfinv; 8 (R - 1) < n <= 8 R; gs:
// lp_scratch_len scalars; one wave (blockDim.x == 64).
template <int R, bool FULL, class Ar, class Src>
__device__ __forceinline__ void lp_pfinv(const Ar& ar, Src src, int n, typename Ar::S* out, float* out32, double sign,
                                         typename Ar::S* gs, LpLds<typename Ar::S>& L, typename Ar::S& pf, int& info,
                                         bool check_zero, bool& allzero) {
  using S = typename Ar::S;
  using P = LpPair<S>;
  constexpr int LDB = rr_ldb(8, R), Q = (8 * R + 63) / 64;  // Q positions per lane: lane + 64 q
  const int lane = threadIdx.x;
  const int a0 = lane & 7, b0 = lane >> 3;
  int a = a0, b = b0;
#define RR_FRESH()                       \
  do {                                   \
    a = a0;                              \
    b = b0;                              \
    asm volatile("" : "+v"(a), "+v"(b)); \
  } while (0)
  S* const A = L.m;
  P* const xy = reinterpret_cast<P*>(L.vec);           // {x, y} of a row
  P* const tt = reinterpret_cast<P*>(L.vec) + 8 * R;   // {t1, t2} of a column
#ifdef MVMC_PHASE_CLOCKS
  long long rr_t0 = __builtin_readcyclecounter(), rr_ph[12] = {};
#define LP_PHASE(k)                                         \
  do {                                                      \
    const long long t_ = __builtin_readcyclecounter();      \
    rr_ph[k] += t_ - rr_t0;                                 \
    rr_t0 = t_;                                             \
  } while (0)
#else
#define LP_PHASE(k) \
  do {              \
  } while (0)
#endif

  // ---- gather: every block's loads in flight together ----
  double mx = 0.0;
  {
    S v[R * (R + 1) / 2];
    RR_FOR(cj, 0, R) {
      RR_FOR(ri, 0, cj + 1) {
        const int i = a + 8 * ri, j = b + 8 * cj;
        S x = Ar::zero();
        if (j < n && i < j) x = src(i, j);
        v[lp_blk(ri, cj) / 64] = x;
      };
    };
    RR_FOR(t, 0, R * (R + 1) / 2) {
      mx = fmax(mx, Ar::mag2(v[t]));
      A[64 * t + lane] = v[t];
    };
  }
  allzero = false;
  if (check_zero) {  // pfaffian.rs:884-890: the plane is skew, so the upper half decides
    allzero = rr_wave_max(mx) < 1.0e-28;
    if (allzero) return;
  }
  rr_sync<8>();
  LP_PHASE(0);

  // ---- dsktf2: k0 = n-1 .. 1 ----
  // x = column k0, the y of the step before; its first largest key, found at
  // the end of that step, is the pivot.  Element {i, p} of the triangle lies
  // at ci[q] + up(p) for i < p and at ri[q] + lo(p) for i > p.
  int ci[Q], ro[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int i = lane + 64 * q;
    ci[q] = 64 * (i >> 3) + (i & 7);
    ro[q] = lp_blk(0, i >> 3) + 8 * (i & 7);
  }
  auto up = [&](int p) RR_INLINE { return lp_blk(0, p >> 3) + 8 * (p & 7); };
  auto lo = [&](int p) RR_INLINE { return 64 * (p >> 3) + (p & 7); };
  auto pivot = [&](const S (&v)[Q], int m, int& kp, bool& zero) RR_INLINE {
    double key[Q], best = -2.0;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int i = lane + 64 * q;
      key[q] = i < m ? Ar::key(v[q], i) : -2.0;
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
  auto pick = [&](const S (&v)[Q], int p) RR_INLINE {  // position p's value in every lane
    S w = v[0];
    if constexpr (Q > 1) w = p >= 64 ? v[1] : v[0];
    return Ar::readlane(w, p & 63);
  };
  S x[Q], y[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int i = lane + 64 * q;
    x[q] = i < n - 1 ? A[ci[q] + up(n - 1)] : Ar::zero();
    y[q] = Ar::zero();
  }
  int kp = 0;
  bool zero = false;
  pivot(x, n - 1, kp, zero);
  info = 0;
  int f[Q];  // the output permutation: position r holds index f(r); the swaps composed as they come
#pragma unroll
  for (int q = 0; q < Q; ++q) f[q] = lane + 64 * q;
  bool neg = false;  // parity of the interchanges
  for (int k0 = n - 1; k0 >= 1; --k0) {
    const int kk0 = k0 - 1;
    RR_FRESH();
    if (zero) {  // zero pivot column: the plane has no Pfaffian form to go on with
      info = kk0 + 1;
      break;
    }
    const S xk = pick(x, kp);
    if (lane == 0) L.sup[kk0] = xk;
    if (kk0 == 0) break;
    const S alpha = ar.alpha(xk);
    const int ukk = up(kk0), lkk = lo(kk0), uk0 = up(k0);
    // interchange of rows/columns kk0 and kp in the upper triangle with the
    // sign twiddles: a lane moves its position's elements {i, kp}, {i, kk0}
    if (kp != kk0) {
      neg = !neg;
      const int ukp = up(kp), lkp = lo(kp);
      const S xq = pick(x, kk0);
      S r1[Q], r2[Q];
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int i = lane + 64 * q;
        f[q] = f[q] == kk0 ? kp : f[q] == kp ? kk0 : f[q];
        const bool in = i < n;
        r1[q] = A[in ? (i < kp ? ci[q] + ukp : ro[q] + lkp) : 0];
        r2[q] = A[in ? (i < kk0 ? ci[q] + ukk : ro[q] + lkk) : 0];
      }
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int i = lane + 64 * q;
        if (i == kp) x[q] = xq;
        const bool mid = i > kp && i < kk0;
        y[q] = i == kp ? Ar::neg(r2[q]) : mid ? Ar::neg(r1[q]) : r1[q];
        if (i < n && i != kp && i != kk0 && i != k0)
          A[i < kp ? ci[q] + ukp : ro[q] + lkp] = mid ? Ar::neg(r2[q]) : r2[q];
        if (i < n && i > k0) A[ro[q] + lkk] = r1[q];
      }
    } else {
#pragma unroll
      for (int q = 0; q < Q; ++q)
        if (lane + 64 * q < kk0) y[q] = A[ci[q] + ukk];
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int i = lane + 64 * q;
      if (i < kk0) {
        xy[i] = P{x[q], y[q]};
        tt[i] = P{Ar::mul(alpha, y[q]), Ar::mul(alpha, x[q])};
        A[ci[q] + uk0] = ar.scale(x[q], alpha);
      }
    }
    rr_sync<8>();
    LP_PHASE(1);
    // rank-2 update of the leading kk0 x kk0 block (elements on and below
    // the diagonal of a diagonal block are never read)
    rr_case<0, R>(kk0 >> 3, [&]<int K>() RR_INLINE {
      P r[K + 1];
      RR_FOR(ri, 0, K + 1) { r[ri] = xy[a + 8 * ri]; };
      RR_FOR(cj, 0, K + 1) {
        const P t = tt[b + 8 * cj];
        S c[cj + 1];
        RR_FOR(ri, 0, cj + 1) { c[ri] = A[lp_blk(ri, cj) + lane]; };
        if (cj < K || b < (kk0 & 7)) {
          RR_FOR(ri, 0, cj + 1) { A[lp_blk(ri, cj) + lane] = Ar::update(c[ri], r[ri].a, r[ri].b, t.a, t.b); };
        }
      };
    });
    LP_PHASE(2);
    // the next step's pivot column is y, which the update leaves alone
    pivot(y, kk0, kp, zero);
#pragma unroll
    for (int q = 0; q < Q; ++q) x[q] = y[q];
    rr_sync<8>();
    LP_PHASE(3);
  }
  if (info != 0) {
    pf = Ar::zero();
    return;
  }
  __syncthreads();
  // ---- utu2pfa: product of A(i, i+1), i even, sign by the count of moves ----
  {
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
    pf = Ar::mul(Ar::sign(neg), p);
  }
  if (!Ar::finite(pf)) {
    info = -1;
    return;
  }
  if constexpr (Ar::kRecip)
    for (int i = lane; i + 1 < n; i += 64) {
      const S vt = Ar::neg(L.sup[i]);
      L.rneg[i] = Ar::recip(Ar::neg(vt));
      L.rpos[i] = Ar::recip(vt);
    }
#pragma unroll
  for (int q = 0; q < Q; ++q)
    if (lane + 64 * q < n) L.finv[f[q]] = lane + 64 * q;
  __syncthreads();
  LP_PHASE(4);

  // ---- utu2inv (panel path for n > 64; the full form differs in the product) ----
  // trtri('U','U') on B(i, j) = A(i, j+1), 0 <= i < j <= n-2: at step k the
  // column k of the inverse is final (Bn(i, k) = -acc(i, k), i < k) and
  // every acc(i, j), i < k < j, adds Bn(i, k) B(k, j) with row k of B still
  // as factored (no earlier step writes it): each element takes its k in
  // ascending order, as the row-chain loops do.  acc stays in A.
  // Two steps a pass: column k+2 as step k leaves it is formed beside the
  // pass (rows < k of it receive step k's term), so every other element is
  // read and written once for both.
  for (int k = 1; k <= n - 3; k += 2) {
    RR_FRESH();
    const int kb = k & 7;                 // odd: k and k + 1 lie in one block row, k + 2 may not
    const S* u = A + up(k + 1) + a;       // columns k + 1 and k + 2 by rows
    const S* u2 = A + up(k + 2) + a;
    const S* w = A + kb + 8 * b;          // row k by columns; row k + 1 is one element further
    const S b2 = A[up(k + 2) + lo(k)];    // A(k, k + 2)
    if (kb != 7) {
      rr_case<0, R>(k >> 3, [&]<int K>() RR_INLINE {
        S ui[K + 1], vi[K + 1];
        RR_FOR(ri, 0, K + 1) {
          ui[ri] = Ar::neg(u[64 * ri]);
          const S raw = u2[64 * ri];
          const S upd = Ar::add(raw, Ar::mul(ui[ri], b2));
          vi[ri] = Ar::neg(ri < K || a < kb ? upd : raw);
        };
        RR_FOR(cj, K, R) {
          const S bj = w[lp_blk(K, cj)], dj = w[lp_blk(K, cj) + 1];
          S c[K + 1];
          RR_FOR(ri, 0, K + 1) { c[ri] = A[lp_blk(ri, cj) + lane]; };
          const int j = b + 8 * cj;
          if (cj > K + 1 || j >= k + 2) {
            const bool both = cj > K + 1 || j >= k + 3;
            RR_FOR(ri, 0, K) {
              const S t = Ar::add(c[ri], Ar::mul(ui[ri], bj));
              const S z = Ar::add(t, Ar::mul(vi[ri], dj));
              A[lp_blk(ri, cj) + lane] = both ? z : t;
            };
            if (a <= kb) {
              const S t = Ar::add(c[K], Ar::mul(ui[K], bj));
              const S y1 = a < kb ? t : c[K];
              const S z = Ar::add(y1, Ar::mul(vi[K], dj));
              A[lp_blk(K, cj) + lane] = both ? z : y1;
            }
          }
        };
      });
    } else {
      // rows k and k + 1 lie in block rows K and K + 1
      rr_case<0, R>(k >> 3, [&]<int K>() RR_INLINE {
        if constexpr (K + 1 < R) {
          S ui[K + 1], vi[K + 1];
          RR_FOR(ri, 0, K + 1) {
            ui[ri] = Ar::neg(u[64 * ri]);
            const S raw = u2[64 * ri];
            const S upd = Ar::add(raw, Ar::mul(ui[ri], b2));
            vi[ri] = Ar::neg(ri < K || a < kb ? upd : raw);
          };
          RR_FOR(cj, K + 1, R) {
            const S bj = w[lp_blk(K, cj)], dj = A[lp_blk(K + 1, cj) + 8 * b];
            S c[K + 1];
            RR_FOR(ri, 0, K + 1) { c[ri] = A[lp_blk(ri, cj) + lane]; };
            const int j = b + 8 * cj;
            if (cj > K + 1 || j >= k + 2) {
              const bool both = cj > K + 1 || j >= k + 3;
              RR_FOR(ri, 0, K + 1) {
                const S t = Ar::add(c[ri], Ar::mul(ui[ri], bj));
                const S y1 = ri < K || a < kb ? t : c[ri];
                const S z = Ar::add(y1, Ar::mul(vi[ri], dj));
                A[lp_blk(ri, cj) + lane] = both ? z : y1;
              };
            }
          };
        }
      });
    }
    rr_sync<8>();
  }
  LP_PHASE(5);
  // M unit upper: M(i, j) = Bn(i, j) = -acc for i < j <= n-2, M(i, n-1) = 0
  // for i < n-1
  auto mval = [&](int i, int j) RR_INLINE -> S {
    if (j <= i) return j == i ? Ar::one() : Ar::zero();
    if (j == n - 1) return Ar::zero();
    return Ar::neg(A[64 * (i >> 3) + (i & 7) + up(j + 1)]);
  };
  // skew-tridiagonal solve T C = M (vt[i] = -A(i, i+1) = -sup[i]), a lane
  // per column, its two chains side by side, C to gs row-major (panel form:
  // the upper part):
  //   forward   C(1) = M(0) / -vt[0]; C(i+1) = (M(i) - C(i-1) vt[i-1]) / -vt[i], i even
  //   backward  C(n-2) = M(n-1) / vt[n-2]; C(i-1) = (M(i) + C(i+1) vt[i]) / vt[i-1], i odd descending
  {
    S pfw[Q], pbw[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) pfw[q] = pbw[q] = Ar::zero();
#pragma unroll 2
    for (int s = 0; 2 * s < n; ++s) {
      const int i = 2 * s, k = n - 1 - 2 * s;
      const S vti = Ar::neg(L.sup[i]), vtm = Ar::neg(L.sup[k - 1]);
      const S vtp = s > 0 ? Ar::neg(L.sup[i - 1]) : Ar::zero(), vtk = s > 0 ? Ar::neg(L.sup[k]) : Ar::zero();
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int j = lane + 64 * q;
        if (j < n) {
          S nu = mval(i, j), nv = mval(k, j);
          if (s > 0) {
            nu = Ar::sub(nu, Ar::mul(pfw[q], vtp));
            nv = Ar::add(nv, Ar::mul(pbw[q], vtk));
          }
          pfw[q] = Ar::div_negvt(nu, vti, Ar::kRecip ? L.rneg[i] : vti);
          pbw[q] = Ar::div_vt(nv, vtm, Ar::kRecip ? L.rpos[k - 1] : vtm);
          if (FULL || i + 1 < j) gs[(size_t)(i + 1) * n + j] = pfw[q];
          if (FULL || k - 1 < j) gs[(size_t)(k - 1) * n + j] = pbw[q];
        }
      }
    }
  }
  __syncthreads();
  LP_PHASE(6);
  // product C'(i, j) = C(i, j) + sum_{k < i} M(k, i) C(k, j), k ascending, C
  // as solved: k by k, the rows of C LP_KB at a time through LDS (the next
  // ones loaded meanwhile), M from LDS.  Panel form: the upper part (the
  // lower follows by skew symmetry).  Full form: every element (the
  // small-matrix path multiplies the column-permuted C; a column's result
  // depends on that column alone, so the permutation moves to the output);
  // in two column halves where the whole would crowd the registers.
  // Then the output: out(r, c) = sign * F(f(r), f(c)), F = C' (full form) or
  // the skew completion of C' (panel form, 0 on the diagonal): columns of F
  // through LDS, each written as one permuted column of out.
  auto put = [&](const S* ob, int v, int row) RR_INLINE {
    const int col = L.finv[v] * n;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int r = lane + 64 * q;
      if (r < n) {
        S w = ob[row * LDB + f[q]];
        if (sign != 1.0) w = Ar::neg(w);
        out[col + r] = w;
        if constexpr (sizeof(S) == sizeof(double))
          if (out32) out32[col + r] = (float)w;
      }
    }
  };
  constexpr int G = FULL && R > 4 ? 2 : 1, HC = (R + G - 1) / G;  // column groups of HC blocks
  RR_FOR(g, 0, G) {
    constexpr int C0 = g * HC, C1 = C0 + HC < R ? C0 + HC : R;
    S c[FULL ? R * HC : R * (R + 1) / 2];
#define RC(ri, cj) c[FULL ? (ri) * HC + (cj) - C0 : rr_slot<R>(ri, cj)]
    RR_FRESH();
    RR_FOR(ri, 0, R) {
      RR_FOR(cj, FULL ? C0 : ri, C1) {
        const int i = a + 8 * ri, j = b + 8 * cj;
        RC(ri, cj) = (FULL || i < j) && i < n && j < n ? gs[i * n + j] : Ar::zero();
      };
    };
    LP_PHASE(7);
    {
      S* const cb = L.vec;
      S pre[LP_KB * Q];
      auto fetch = [&](int k0) RR_INLINE {
        RR_FOR(u, 0, LP_KB * Q) {
          const int k = k0 + u / Q, j = lane + 64 * (u % Q);
          pre[u] = k < n && j < n && (FULL || k < j) ? gs[k * n + j] : Ar::zero();
        };
      };
      fetch(0);
#pragma unroll 1
      for (int k0 = 0; k0 < n - 1; k0 += LP_KB) {
        RR_FRESH();
        RR_FOR(u, 0, LP_KB * Q) {
          const int j = lane + 64 * (u % Q);
          if (j < LDB) cb[(u / Q) * LDB + j] = pre[u];
        };
        rr_sync<8>();
        fetch(k0 + LP_KB);
        rr_case<0, R>(k0 >> 3, [&]<int K>() RR_INLINE {
          // M(k, i) = -A(k, i + 1): column i + 1 = a + 8 r + 1 lies in block
          // column r, or r + 1 for a = 7
          constexpr int CL = FULL ? C0 : (K > C0 ? K : C0);
          const int k1 = min(LP_KB, n - 1 - k0);
          const int carry = a == 7 ? 64 : 0, within = (k0 & 7) + 8 * ((a + 1) & 7);
#pragma unroll 2
          for (int kk = 0; kk < k1; ++kk) {
            const int k = k0 + kk;
            S mi[R], cv[R];
            RR_FOR(r, K, R) {
              const bool in = r + 1 < R || a + 8 * r < n - 1;
              const S v = A[in ? lp_blk(K, r) + carry * (r + 1) + within + kk : 0];
              mi[r] = in ? Ar::neg(v) : Ar::zero();
            };
            RR_FOR(r, CL, C1) { cv[r] = cb[kk * LDB + b + 8 * r]; };
            RR_FOR(cj, CL, C1) {
              RR_FOR(ri, K + 1, (FULL ? R : cj + 1)) { RC(ri, cj) = Ar::add(RC(ri, cj), Ar::mul(mi[ri], cv[cj])); };
            };
            if (k < a + 8 * K) {
              RR_FOR(cj, CL, C1) { RC(K, cj) = Ar::add(RC(K, cj), Ar::mul(mi[K], cv[cj])); };
            }
          }
        });
        rr_sync<8>();
      }
    }
    LP_PHASE(8);
    RR_FRESH();
    if constexpr (FULL) {
      // four columns at a time (M is still wanted by the next group)
      S* const ob = L.vec;
#pragma unroll 1
      for (int h = 2 * C0; h < 2 * C1; ++h) {
        rr_case<C0, C1>(h >> 1, [&]<int K>() RR_INLINE {
          if ((b >> 2) == (h & 1)) {
            RR_FOR(ri, 0, R) { ob[(b & 3) * LDB + a + 8 * ri] = RC(ri, K); };
          }
        });
        rr_sync<8>();
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (4 * h + v < n) put(ob, 4 * h + v, v);
        rr_sync<8>();
      }
    } else {
      S* const ob = L.m;
#pragma unroll 1
      for (int blk = 0; blk < R; ++blk) {
        rr_case<0, R>(blk, [&]<int K>() RR_INLINE {
          RR_FOR(ri, 0, K) { ob[b * LDB + a + 8 * ri] = RC(ri, K); };
          if (a < b) {
            ob[b * LDB + a + 8 * K] = RC(K, K);
            ob[a * LDB + b + 8 * K] = Ar::neg(RC(K, K));
          } else if (a == b) {
            ob[a * LDB + a + 8 * K] = Ar::zero();
          }
          RR_FOR(cj, K + 1, R) { ob[a * LDB + b + 8 * cj] = Ar::neg(RC(K, cj)); };
        });
        rr_sync<8>();
#pragma unroll 4
        for (int v = 0; v < 8; ++v)
          if (8 * blk + v < n) put(ob, 8 * blk + v, v);
        rr_sync<8>();
      }
    }
#undef RC
  };
  __syncthreads();
  LP_PHASE(9);
#ifdef MVMC_PHASE_CLOCKS
  if (lane == 0 && blockIdx.x == 0)
    printf("lp n=%d cycles: gather %lld ltl interchange %lld update %lld pivot %lld pf %lld trtri %lld solve %lld "
           "load %lld product %lld out %lld\n",
           n, rr_ph[0], rr_ph[1], rr_ph[2], rr_ph[3], rr_ph[4], rr_ph[5], rr_ph[6], rr_ph[7], rr_ph[8], rr_ph[9]);
#endif
#undef LP_PHASE
#undef RR_FRESH
}

}  // namespace mvmc_hip
