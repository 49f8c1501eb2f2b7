// Batched Pfaffian + inverse of complex skew-symmetric planes: the kernels of
// pfinv_lds.h (n <= 64) and pfinv_rr.h (n <= 160) with the complex
// arithmetic of the reference's scalar pfapack build, element by element as
// wg_pfinv_c128 (pfinv_c128_dev.h) performs it:
//   LTL^T  (crates/pfapack/src/ltl.rs:61-191) pivot by the first largest
//          |re| + |im|; order 0 = zsktf2: alpha = Julia 1/pivot
//          (julia_complex.rs:36-77), column k0 scaled by complex products
//          (backend.rs:351-355); order 1 = zsktf2_c_compat: alpha =
//          (re, -im) / (re^2 + im^2) (ltl.rs:256-263), scaling with fused
//          multiply-adds (ltl.rs:303-315); rank-2 update c + (x t1 - y t2)
//          (ltl.rs:707-818)
//   inverse (utu2.rs:399-515): trtri 'U','U', the skew-tridiagonal solve
//          multiplying by Julia reciprocals of -vt and vt
//          (utu2.rs:110-282, julia_complex.rs:79-122), the product and the
//          permutations as the real kernel.
// Complex arithmetic is num_complex's; the library is built with
// -ffp-contract=off.  Compiled once per RR_PART (a range of sizes).
#include "cplx.h"
#include "pfinv_lds.h"
#include "pfinv_rr.h"
#include "rr_planes.h"

namespace mvmc_hip {
namespace {

struct RrCplx {
  int order;  // 0 zsktf2, 1 zsktf2_c_compat
  using S = cz;
  static constexpr bool kRecip = true;  // the solve multiplies by Julia reciprocals
  static __device__ __forceinline__ S zero() { return cz{0.0, 0.0}; }
  static __device__ __forceinline__ S one() { return cz{1.0, 0.0}; }
  static __device__ __forceinline__ S neg(S x) { return cz_neg(x); }
  static __device__ __forceinline__ S add(S x, S y) { return cz_add(x, y); }
  static __device__ __forceinline__ S sub(S x, S y) { return cz_sub(x, y); }
  static __device__ __forceinline__ S mul(S x, S y) { return cz_mul(x, y); }
  static __device__ __forceinline__ double mag2(S x) { return x.re * x.re + x.im * x.im; }
  // |re| + |im|: a NaN wins only at index 0, as the sequential scan
  static __device__ __forceinline__ double key(S x, int i) { return rr_key(fabs(x.re) + fabs(x.im), i); }
  __device__ __forceinline__ S alpha(S pv) const {
    if (order == 0) return julia_div(cz{1.0, 0.0}, pv);
    const double den = pv.re * pv.re + pv.im * pv.im;
    return cz{pv.re / den, -pv.im / den};
  }
  static __device__ __forceinline__ S update(S c, S xi, S yi, S t1, S t2) {
    return cz_add(c, cz_sub(cz_mul(xi, t1), cz_mul(yi, t2)));
  }
  __device__ __forceinline__ S scale(S v, S alpha) const {
    if (order == 0) return cz_mul(v, alpha);
    return cz{fma(alpha.re, v.re, -(alpha.im * v.im)), fma(alpha.re, v.im, alpha.im * v.re)};
  }
  static __device__ __forceinline__ S sign(bool neg) { return neg ? cz{0.0 - 1.0, 0.0 - 0.0} : cz{1.0, 0.0}; }
  static __device__ __forceinline__ bool finite(S x) { return isfinite(x.re) && isfinite(x.im); }
  static __device__ __forceinline__ S div_negvt(S num, S, S rneg) { return cz_mul(num, rneg); }
  static __device__ __forceinline__ S div_vt(S num, S, S rpos) { return cz_mul(num, rpos); }
  static __device__ __forceinline__ S recip(S x) { return julia_recip(x); }
  static __device__ __forceinline__ S readlane(S x, int l) {
    return cz{RrReal::readlane(x.re, l), RrReal::readlane(x.im, l)};
  }
};

// Planes blockIdx.x, + gridDim.x, ... of [count][n][n] complex column-major
// planes.  Results and statuses as k_pfinv_c128 (a failed plane's inverse
// zero-filled, pf 0 on a zero pivot, the computed pf when non-finite);
// in == out works in place (a plane is read whole before it is written).
template <int NT, class Plane>
__device__ __forceinline__ void rr_planes_c128(const RrJob& job, Plane plane) {
  const int n = job.n, tid = threadIdx.x;
  for (int p = blockIdx.x; p < job.count; p += gridDim.x) {
    const cz* A = (const cz*)job.in + (size_t)p * n * n;
    cz* O = (cz*)job.out + (size_t)p * n * n;
    cz pfv{0.0, 0.0};
    int info = 0;
    bool az = false;
    plane([&](int i, int j) { return A[i + (size_t)j * n]; }, O, pfv, info, az);
    if (tid == 0) {
      job.status[p] = info;
      ((cz*)job.pf)[p] = info > 0 ? cz{0.0, 0.0} : pfv;
    }
    if (info != 0)
      for (int e = tid; e < n * n; e += NT) O[e] = cz{0.0, 0.0};
    __syncthreads();
  }
}

template <int R>
__global__ void __launch_bounds__(64, R <= 4 ? 2 : 1) k_lp_planes_c128(RrJob job) {
  extern __shared__ __align__(16) char lds[];
  Carver c{lds};
  LpLds<cz> L = carve_lp<cz, true, R>(c);
  cz* gs = (cz*)job.gs + (size_t)blockIdx.x * lp_scratch_len(job.n);
  rr_planes_c128<64>(job, [&](auto src, cz* out, cz& pf, int& info, bool& az) RR_INLINE {
    lp_pfinv<R, true>(RrCplx{job.order}, src, job.n, out, nullptr, 1.0, gs, L, pf, info, false, az);
  });
}

template <int R>
__global__ void __launch_bounds__(256, R <= 6 ? 2 : 1) k_rr_planes_c128(RrJob job) {
  extern __shared__ __align__(16) char lds[];
  Carver c{lds};
  RrLdsT<cz> L = carve_rr<cz, true, 16, R>(c, job.n);
  cz* gs = (cz*)job.gs + (size_t)blockIdx.x * rr_scratch_len(job.n);
  rr_planes_c128<256>(job, [&](auto src, cz* out, cz& pf, int& info, bool& az) RR_INLINE {
    rr_pfinv<16, R>(RrCplx{job.order}, src, job.n, out, nullptr, 1.0, gs, L, pf, info, false, az);
  });
}

}  // namespace

#if RR_PART == 0
const void* rr_kernel_c128_small(int r) {
  switch (r) {
    case 1: return (const void*)k_lp_planes_c128<1>;
    case 2: return (const void*)k_lp_planes_c128<2>;
    case 3: return (const void*)k_lp_planes_c128<3>;
    case 4: return (const void*)k_lp_planes_c128<4>;
    case 5: return (const void*)k_lp_planes_c128<5>;
    case 6: return (const void*)k_lp_planes_c128<6>;
    case 7: return (const void*)k_lp_planes_c128<7>;
    case 8: return (const void*)k_lp_planes_c128<8>;
  }
  return nullptr;
}
#else
const void* rr_kernel_c128_large(int r) {
  switch (r) {
    case 5: return (const void*)k_rr_planes_c128<5>;
    case 6: return (const void*)k_rr_planes_c128<6>;
    case 7: return (const void*)k_rr_planes_c128<7>;
    case 8: return (const void*)k_rr_planes_c128<8>;
    case 9: return (const void*)k_rr_planes_c128<9>;
    case 10: return (const void*)k_rr_planes_c128<10>;
  }
  return nullptr;
}
#endif

}  // namespace mvmc_hip
