// Pfaffian + inverse of real planes (pfinv_lds.h, pfinv_rr.h) as kernels:
// persistent grids over planes of a batched call or of an ensemble's
// walkers.  Compiled once per RR_PART (a range of sizes) so that the parts
// build side by side.
#include "rr_planes.h"

#include "pfinv_lds.h"
#include "pfinv_rr.h"

namespace mvmc_hip {
namespace {

// Plane `item` of an ensemble job: the (site, spin) rows of its walker's
// configuration into rs.  Returns 0 if the plane is to be factorised, 1 if
// its walker needs nothing, 2 if the configuration is invalid.
__device__ __forceinline__ int rr_rows(const RrJob& job, int w, int* rs) {
  const EnsView& v = job.v;
  const int tid = threadIdx.x, nt = blockDim.x;
  const int* ei = job.mode == RR_MEASURE ? v.s_idx + ((size_t)w * v.nsample + job.s) * v.n
                                         : v.ele_idx + (size_t)w * v.n;
  int bad = 0, nonzero = 0, nonneg = 0;
  for (int i = tid; i < v.n; i += nt) {
    const int r = ei[i];
    rs[i] = r + (i / v.ne) * v.ns;
    bad |= r < 0 || r >= v.ns;
    nonzero |= r != 0;
    nonneg |= r >= 0;
  }
  if (job.mode == RR_MEASURE) {  // the all-zero / all-negative placeholder of a sample
    const int some = __syncthreads_or(nonzero), pos = __syncthreads_or(nonneg);
    if (!some || !pos) return 1;
  }
  return __syncthreads_or(bad) ? 2 : 0;
}

// Items are taken in grid strides: planes of a batched call, (walker, QP
// plane) pairs of an ensemble job, so that a few walkers with many planes
// fill the chip as many planes do.  An ensemble plane leaves its Pfaffian in
// pf_new and its outcome in pinfo; k_rr_finish decides per walker.
// plane(A, ld, rs, sign...) factorises one plane: A(i, j) = in[i + j n], or
// gathered from the Slater table -S[rs_j][rs_i] (pfaffian.rs:1107-1188);
// inverse, or minus the inverse (mVMC's InvM).
template <int NT, class Plane>
__device__ __forceinline__ void rr_items(const RrJob& job, int* rs, Plane plane) {
  const int n = job.n, tid = threadIdx.x;
  const bool ens = job.mode != RR_BATCHED;
  const int nqp = ens ? job.v.nqp : 1;
  const int items = !ens ? job.count : (job.mode == RR_REBUILD ? *job.v.nflag : job.v.W) * nqp;
  if (!ens) {
    for (int i = tid; i < n; i += NT) rs[i] = i;
    __syncthreads();
  }
  for (int item = blockIdx.x; item < items; item += gridDim.x) {
    const double* A;
    double* out;
    float* out32 = nullptr;
    int ld, q = 0, w = 0;
    if (!ens) {
      A = (const double*)job.in + (size_t)item * n * n;
      out = (double*)job.out + (size_t)item * n * n;
      ld = n;
    } else {
      const EnsView& v = job.v;
      w = item / nqp;
      q = item - w * nqp;
      if (job.mode == RR_REBUILD) w = v.rlist[w];
      if (job.mode == RR_BEGIN && !v.wstate[(size_t)w * 8]) continue;
      __syncthreads();  // rs of the plane before
      const int skip = rr_rows(job, w, rs);
      if (skip) {
        if (tid == 0) {
          v.pinfo[(size_t)w * nqp + q] = skip == 1 ? RR_SKIPPED : RR_BAD_SITE;
          if (skip == 2) atomicCAS(v.status, 0, (int)ST_BAD_INPUT);
        }
        continue;
      }
      ld = v.n2;
      A = v.slater + (size_t)q * ld * ld;
      const size_t off = ((size_t)w * nqp + q) * n * n;
      out = v.inv + off;
      if (v.inv32 && job.mode != RR_MEASURE) out32 = v.inv32 + off;
    }
    double pfv = 0.0;
    int info = 0;
    bool az = false;
    plane([&](int i, int j) { const double x = A[(size_t)rs[j] * ld + rs[i]]; return ens ? -x : x; }, out, out32,
          ens ? -1.0 : 1.0, pfv, info, job.mode == RR_REBUILD || job.mode == RR_MEASURE, az);
    if (!ens) {
      if (tid == 0) {
        job.status[item] = info;
        ((double*)job.pf)[item] = info > 0 ? 0.0 : pfv;
      }
      if (info != 0)
        for (int e = tid; e < n * n; e += NT) out[e] = 0.0;
    } else if (tid == 0) {
      job.v.pinfo[(size_t)w * nqp + q] = az ? RR_ALL_ZERO : info;
      job.v.pf_new[(size_t)w * nqp + q] = pfv;
    }
  }
}

// n <= LP_NMAX: one wave per plane, the plane in LDS (pfinv_lds.h).  The LDS
// admits seven planes per CU at n = 64 and fewer above, so the larger ones
// may use the registers of a whole SIMD.
template <int R, bool FULL>
__global__ void __launch_bounds__(64, R <= 8 ? 2 : 1) k_lp_planes(RrJob job) {
  extern __shared__ __align__(16) char lds[];
  Carver c{lds};
  int* rs = c.take<int>(job.n);
  LpLds<double> L = carve_lp<double, false, R>(c);
  double* gs = (double*)job.gs + (size_t)blockIdx.x * lp_scratch_len(job.n);
  rr_items<64>(job, rs, [&](auto src, double* out, float* out32, double sign, double& pf, int& info, bool chk,
                            bool& az) RR_INLINE {
    lp_pfinv<R, FULL>(RrReal{}, src, job.n, out, out32, sign, gs, L, pf, info, chk, az);
  });
}

// n > LP_NMAX: four waves per plane, the plane in registers (pfinv_rr.h);
// two planes per CU while the registers admit it.
template <int R>
__global__ void __launch_bounds__(256, R <= 10 ? 2 : 1) k_rr_planes(RrJob job) {
  extern __shared__ __align__(16) char lds[];
  Carver c{lds};
  int* rs = c.take<int>(job.n);
  RrLds L = carve_rr<double, false, 16, R>(c, job.n);
  double* gs = (double*)job.gs + (size_t)blockIdx.x * rr_scratch_len(job.n);
  rr_items<256>(job, rs, [&](auto src, double* out, float* out32, double sign, double& pf, int& info, bool chk,
                             bool& az) RR_INLINE {
    rr_pfinv<16, R>(RrReal{}, src, job.n, out, out32, sign, gs, L, pf, info, chk, az);
  });
}

}  // namespace

#if RR_PART == 0
const void* rr_kernel_small(int r) {
  switch (r) {
    case 1: return (const void*)k_lp_planes<1, true>;
    case 2: return (const void*)k_lp_planes<2, true>;
    case 3: return (const void*)k_lp_planes<3, true>;
    case 4: return (const void*)k_lp_planes<4, true>;
    case 5: return (const void*)k_lp_planes<5, true>;
    case 6: return (const void*)k_lp_planes<6, true>;
    case 7: return (const void*)k_lp_planes<7, true>;
    case 8: return (const void*)k_lp_planes<8, true>;
  }
  return nullptr;
}
#elif RR_PART == 1
const void* rr_kernel_mid(int r) {
  switch (r) {
    case 9: return (const void*)k_lp_planes<9, false>;
    case 10: return (const void*)k_lp_planes<10, false>;
    case 11: return (const void*)k_lp_planes<11, false>;
    case 12: return (const void*)k_lp_planes<12, false>;
    case 13: return (const void*)k_lp_planes<13, false>;
  }
  return nullptr;
}
#elif RR_PART == 2
const void* rr_kernel_large(int r) {
  switch (r) {
    case 7: return (const void*)k_rr_planes<7>;
    case 8: return (const void*)k_rr_planes<8>;
    case 9: return (const void*)k_rr_planes<9>;
    case 10: return (const void*)k_rr_planes<10>;
  }
  return nullptr;
}
#else
const void* rr_kernel_huge(int r) {
  switch (r) {
    case 11: return (const void*)k_rr_planes<11>;
    case 12: return (const void*)k_rr_planes<12>;
    case 13: return (const void*)k_rr_planes<13>;
    case 14: return (const void*)k_rr_planes<14>;
  }
  return nullptr;
}
#endif

}  // namespace mvmc_hip
