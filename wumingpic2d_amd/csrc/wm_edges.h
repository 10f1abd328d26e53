// wm_edges.h -- the particle boundaries' arithmetic on one particle, shared by
// the boundary kernels (wm_bc.hip) and the resident step's push
// (wm_particle.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace wm_edges {

// largest double below s (s finite)
__device__ inline double pred_d(double s) {
  if (s == 0.0) return -__longlong_as_double(1LL);
  long long b = __double_as_longlong(s);
  b += (s > 0.0) ? -1 : 1;
  return __longlong_as_double(b);
}

// a + b rounded toward -inf (boundary_periodic.f90:74, 124), exact via TwoSum.
__device__ inline double add_rd(double a, double b) {
  const double s = __dadd_rn(a, b);
  const double bb = __dsub_rn(s, a);
  const double err = __dadd_rn(__dsub_rn(a, __dsub_rn(s, bb)), __dsub_rn(b, bb));
  return err < 0.0 ? pred_d(s) : s;
}

}  // namespace wm_edges
