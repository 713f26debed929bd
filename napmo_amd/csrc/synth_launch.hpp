// The synthesis launchers (defined in synth_kernel.hpp, instantiated per lmax in
// synth_inst_*.hip) and the inverse radial transform they share with the pair lists.
#pragma once

#include <hip/hip_runtime.h>

#include "common.hpp"
#include "kernels.hpp"

namespace napmo {

static __device__ inline double rtf_inv(int kind, double p0, double p1, int n, double r) {
  if (kind == 0) return -(acos((r - p0) / (r + p0)) / p1) + n;
  if (kind == 1) return pow(r / p0, 1.0 / p1) - 1;
  return r;
}

template <int LMAX>
void launch_synth_t(dim3 g, dim3 b, hipStream_t s, const AtomTables &at, const double *x,
                    const double *y, const double *z, long N, const double *T, const double *aL,
                    const double *aR, int acc, int ext_mode, double *v);
template <int LMAX>
void launch_synth2_t(int np, hipStream_t s, const AtomTables &at, const double *geo, long N,
                     const int *list, const int *wave_bucket, long nwaves, const double *T,
                     const double *aL, const double *aR, double *contrib);

}  // namespace napmo
