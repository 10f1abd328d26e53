// wm_solve.h -- what the two field solvers share: the streaming one
// (wm_field.hip) and the one on chip (wm_solve.hip).
#pragma once
#include "wm_internal.h"

struct SolveConst {      // field constants, field.f90:53-57
  double f1, f2, f3, f4, f5, gfac, delt;
  double fpt;            // 4 pi delt
};

static inline SolveConst make_fc(const wm_grid &g) {
  const double pi = 3.141592653589793115997963468544185461590576171875;  // field.f90:13
  SolveConst f;
  f.f1 = g.c * g.delt / g.delx;
  f.f2 = g.gfac * f.f1 * f.f1;
  f.f3 = 4.0 * pi * g.delx / g.c;
  const double t = g.delx / (g.c * g.delt * g.gfac);
  f.f4 = 4.0 + t * t;
  f.f5 = t * t;
  f.gfac = g.gfac;
  f.delt = g.delt;
  f.fpt = 4. * pi * g.delt;
  return f;
}

// The on-chip solve's result: iterations and ite_max reached, per component.
struct SolveOut {
  int ite[3], err[3];
};
// What a step's last kernel leaves in pinned host memory.
struct SolveReport {
  SolveOut out;
  int abort_;            // the on-chip solve gave up
  int derr;              // device error bits
  unsigned long long ts[8];   // wm_ctx::ts
  unsigned long long begin;   // the clock as the update began
  unsigned seq;          // written last: which report this is
  // the clock as the update's last workgroup ends, of this report and the last
  // (by seq's lowest bit): there once the stream's next kernel has begun
  unsigned long long end[2];
};
// One thread leaves the report (abort_ null: the solve streamed).
__device__ inline void leave_report(SolveReport *host, const SolveOut &out, int given,
                                    const int *derr, const unsigned long long *ts,
                                    unsigned long long begin, unsigned seq) {
  host->out = out;
  host->abort_ = given;
  host->derr = *derr;
#pragma unroll
  for (int k = 0; k < 8; ++k) host->ts[k] = ts[k];
  host->begin = begin;
  __threadfence_system();
  __hip_atomic_store(&host->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
// One thread of the update's last workgroup leaves the clock.
__device__ inline void leave_end(SolveReport *host, unsigned seq) {
  __hip_atomic_store(&host->end[seq & 1], (unsigned long long)wall_clock64(), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_SYSTEM);
}
// The field update's kernels skip when the on-chip solve before them gave up
// or failed (null: after a streaming solve).
struct SolveGate {
  const int *abort_ = nullptr;
  const SolveOut *out = nullptr;
  __device__ bool closed() const {
    return abort_ && (*abort_ || out->err[0] || out->err[1] || out->err[2]);
  }
};

__device__ inline int wrapm(int a, int n) { return a < 0 ? a + n : (a >= n ? a - n : a); }
