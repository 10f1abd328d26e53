// wm_mover.h -- the current of a cell's crossing particles as sums of outer
// products, a row of Jx, Jy or Jz in each of the cell's 16 lanes (both forms'
// pushes).
#pragma once
#include <hip/hip_runtime.h>

namespace wm_mover {

constexpr int YN = 17;           // values of a mover's y side

// A lane's part in the sums of its cell's movers: one row of Jx, Jy or Jz, all
// five columns.  With X = s0x + dx / 2, Y = s0y + dy / 2 and wy the
// running sum of -q dy/dt dy, the three are sums over the movers of outer
// products with X or dx (field.f90:274-298):
//   Jy = X wy,  Jz = q vz (X Y + dx dy / 12),
//   Jx = the running sum along x of -q dx/dt dx Y, taken at the end.
// A lane's factors are V = y[p] y[s] (of X) and W = y[w] y[t] (of dx), y the
// mover's y side in LDS: Y 0..4, wy 5..8, dy 9..13, then q vz, q vz / 12,
// -q dx/dt; p or w -1: zero.
struct Role {
  int p, s, w, t, out;           // out: first of the cell's sums, -1: none
};
__device__ inline Role role_of(int lane16) {
  Role r{-1, 0, -1, 0, -1};
  if (lane16 < 5) {
    r.w = lane16;
    r.t = 16;
    r.out = lane16;              // Jx: + 5 a
  } else if (lane16 < 9) {
    r.p = lane16;
    r.out = 20 + lane16 - 5;     // Jy: + 4 a
  } else if (lane16 < 14) {
    r.p = lane16 - 9;
    r.s = 14;
    r.w = lane16;
    r.t = 15;
    r.out = 40 + lane16 - 9;     // Jz: + 5 a
  }
  return r;
}

// A lane's mover sums of one cell into its 65 values.
__device__ inline void put_sums(double *cb, const Role &r, const double (&v)[5]) {
  if (r.out < 0) return;
  if (r.out < 20) {
    double t = 0.0;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      t += v[a];
      cb[r.out + 5 * a] = t;
    }
  } else {
    const int st = r.out < 40 ? 4 : 5;
#pragma unroll
    for (int a = 0; a < 5; ++a) cb[r.out + st * a] = v[a];
  }
}

}  // namespace wm_mover
