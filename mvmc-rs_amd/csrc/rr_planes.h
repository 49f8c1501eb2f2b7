// Launch interface of the Pfaffian + inverse kernels of one plane per
// workgroup (rr_planes.hip real, rr_planes_c128.hip complex): planes are the unit of
// work, whether they come from a batched call or from an ensemble's walkers.
#pragma once
#include <hip/hip_runtime.h>

#include "ensemble.h"

namespace mvmc_hip {

enum RrMode : int {
  RR_BATCHED = 0,  // planes in -> out
  RR_REBUILD = 1,  // the QP planes of the walkers k_block handed over (nflag[0], rlist)
  RR_BEGIN = 2,    // of the walkers that resume from their burn configuration (wstate[0])
  RR_MEASURE = 3,  // of every walker's saved sample s
};

struct RrJob {
  int mode;
  int n, count;  // batched: planes
  const void* in;
  void* out;
  void* pf;
  int* status;
  void* gs;   // scratch, RrPlan::scratch bytes per workgroup
  int order;  // complex LTL order
  int s;      // RR_MEASURE
  EnsView v;  // RR_REBUILD, RR_BEGIN, RR_MEASURE
};

// Kernel for planes of order n (kernel == nullptr: n not covered), its LDS,
// the scratch of a workgroup and the workgroups that are resident on the
// current device.
struct RrPlan {
  const void* kernel = nullptr;
  int threads = 0;
  size_t lds = 0, scratch = 0;
  int resident = 0;
};

// The instances, by blocks per side; compiled in parts (one object each).
const void* rr_kernel_small(int r);       // n <= 64: r = ceil(n / 8)
const void* rr_kernel_mid(int r);         // n <= 104: r = ceil(n / 8)
const void* rr_kernel_large(int r);       // n <= 160: r = ceil(n / 16)
const void* rr_kernel_huge(int r);        // n <= 224: r = ceil(n / 16)
const void* rr_kernel_c128_small(int r);  // complex, n <= 64: r = ceil(n / 8)
const void* rr_kernel_c128_large(int r);  // complex, n <= 160: r = ceil(n / 16)

}  // namespace mvmc_hip
