// wm_particle.hip -- Buneman-Boris push and Esirkepov deposit (FP64 form).
//
// The resident step's kernel, push and deposit in one, is k_push_step below.
// The host-array entry points push and deposit apart, in k_particle.  Its work
// decomposition: one workgroup per (row j, chunk of CHUNK cells); the
// workgroup's 256 lanes form 32 groups of 8 lanes, group g owns cell
// i0+g and its 8 lanes stride through that cell's particles of every species
// (the reference's cell -> species -> particle loop, particle.f90:85-94 and
// field.f90:212-221).  Particles of one cell are contiguous (sorted); a
// group's windows of 16 particles start at the 16-particle boundary at or
// below the cell's first particle (lanes outside the cell idle), and lane
// sub takes the window's particles sub and 8 + sub, so the group's two
// loads of an array cover one aligned 128-byte line.
//
// Push fields come from a per-workgroup LDS tile of the cell-centred fields.
// Deposit: each lane accumulates the stay-in-cell stencils of its particles
// in registers (all in the same cell), the 8 lanes of a group combine by
// butterfly shuffles; cell-crossing particles are listed in LDS as they are
// found and their full 5x5 stencils summed after the cell's loop.  The
// workgroup assembles its 5 x (CHUNK+4) current tile in LDS in a fixed
// order.  Tiles go to a partial buffer that a gather
// kernel sums in a fixed order, so the deposit is deterministic (no
// floating-point atomics).
#include "wm_internal.h"
#include "wm_edges.h"
#include "wm_mover.h"
#include "wm_order.h"

namespace {

using wm_mover::put_sums;
using wm_mover::Role;
using wm_mover::role_of;
using wm_mover::YN;

constexpr int CHUNK = WM_CHUNK_HOST64;   // cells per workgroup
constexpr int GROUP = 8;              // lanes per cell
constexpr int TW = CHUNK + 2;         // push tile width (halo 1)
constexpr int DW = CHUNK + 4;         // deposit tile width (halo 2)
constexpr int TILE = 5 * DW * 3;      // doubles per deposit tile
constexpr int NACC = 65;              // Jx 4x5 + Jy 5x4 + Jz 5x5
constexpr int MCAP = 24;              // a cell's movers listed in LDS at a time

struct PP {                           // particle-kernel parameters
  int nx, ny, nxgs, nys, nsp, cap, nchunk;
  double d_delx, delt, c, qc_scale;   // qc_scale = delx / delt
  double ic2;                         // 1 / c^2
  double q[WM_MAXSP], r[WM_MAXSP];
  // the shock's injection edge, applied to the pushed particle before its
  // current (proj/shock/app.f90:112-114): inj, nxs, the left mirror point
  // 2 (nxs+1) delx, xend and u0 (boundary_shock.f90:266-294)
  int inj, xs;
  double delx, wl, xend, u0;
  // the resident step's particle boundaries, applied as the particle is
  // stored: xmode 1 the periodic wrap, 2 the walls' mirrors, 0 neither
  int xmode, xe;
  double spanx, spany, wr;
};

// What the resident step's push leaves for the row order (wm_order.h).
struct Order {
  const unsigned *perm;          // the rows' order now: species-plane index per slot
  uint16_t *code;                // per slot
  int4 *kind;                    // per cell: to the left, staying, to the right, others
  int *farcnt, *far;             // particles more than one cell away: per new cell; rows with any
};

// Where the kernel reads its particles: the slots themselves, or through
// Order::perm with 32-bit byte offsets into the species' plane (planes below
// 4 GB) or 64-bit ones.
enum { SRC_SLOT = 0, SRC_PERM32 = 1, SRC_PERM64 = 2 };

__device__ inline void injection_edge(double &x, double &ux, double &uy, double &uz,
                                      const PP &P) {
  if ((int)(x / P.delx) < P.xs + 1) {
    x = P.wl - x;
    ux = -ux;
  } else if (x > P.xend) {
    x = 2.0 * P.xend - x;
    ux = 2.0 * P.u0 - ux;
  } else {
    return;
  }
  uy = -uy;
  uz = -uz;
}

__device__ inline void shape(double dh, double &sm, double &s0, double &sp) {
  // 2nd-order (TSC) weights: particle.f90:98-100
  sm = 0.5 * (0.5 - dh) * (0.5 - dh);
  s0 = 0.75 - dh * dh;
  sp = 0.5 * (0.5 + dh) * (0.5 + dh);
}

// Cell-centred field tile: T[(k*3 + b)*TW + col], b = row j-1..j+1,
// col = i - (i0 - 1).
template <int TW>
__device__ inline void load_tmp_tile(double *T, const double *tmp, int TX,
                                     size_t tps, int jl, int c0, int ncol) {
  // tmp planes hold cells (nxs-1 .. nxe+1) x (nys-1 .. nye+1); local column
  // index of cell i is i - (nxs-1); c0 = local column of i0 - 1.
  for (int t = threadIdx.x; t < 6 * 3 * TW; t += blockDim.x) {
    const int col = t % TW;
    const int b = (t / TW) % 3;
    const int k = t / (3 * TW);
    double v = 0.0;
    if (col < ncol) v = tmp[(size_t)k * tps + (size_t)(c0 + col) + (size_t)TX * (size_t)(jl + b)];
    T[t] = v;
  }
}

struct PushOut { double x, y, ux, uy, uz, ig; };   // ig = 1 / gamma of the new u

__device__ inline PushOut boris(const double *T, int gcol, double x, double y,
                                double ux, double uy, double uz, int i, int j,
                                const PP &P, double fac1, double txxx, double fac2) {
  // particle.f90:96-161
  double sx0, sx1, sx2, sy0, sy1, sy2;
  shape(x * P.d_delx - 0.5 - i, sx0, sx1, sx2);
  shape(y * P.d_delx - 0.5 - j, sy0, sy1, sy2);
  double f[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    const double *Tk = T + k * 3 * TW + gcol;   // gcol = column of i-1
    f[k] = (Tk[0] * sx0 + Tk[1] * sx1 + Tk[2] * sx2) * sy0 +
           (Tk[TW] * sx0 + Tk[TW + 1] * sx1 + Tk[TW + 2] * sx2) * sy1 +
           (Tk[2 * TW] * sx0 + Tk[2 * TW + 1] * sx1 + Tk[2 * TW + 2] * sx2) * sy2;
  }
  const double bpx = f[0], bpy = f[1], bpz = f[2];
  const double epx = f[3], epy = f[4], epz = f[5];
  double uvm1 = ux + fac1 * epx;
  double uvm2 = uy + fac1 * epy;
  double uvm3 = uz + fac1 * epz;
  const double gam = sqrt(P.c * P.c + uvm1 * uvm1 + uvm2 * uvm2 + uvm3 * uvm3);
  const double igam = 1.0 / gam;
  const double fac1r = fac1 * igam;
  const double fac2r = fac2 / (gam + txxx * (bpx * bpx + bpy * bpy + bpz * bpz) * igam);
  const double uvm4 = uvm1 + fac1r * (uvm2 * bpz - uvm3 * bpy);
  const double uvm5 = uvm2 + fac1r * (uvm3 * bpx - uvm1 * bpz);
  const double uvm6 = uvm3 + fac1r * (uvm1 * bpy - uvm2 * bpx);
  uvm1 = uvm1 + fac2r * (uvm5 * bpz - uvm6 * bpy);
  uvm2 = uvm2 + fac2r * (uvm6 * bpx - uvm4 * bpz);
  uvm3 = uvm3 + fac2r * (uvm4 * bpy - uvm5 * bpx);
  PushOut o;
  o.ux = uvm1 + fac1 * epx;
  o.uy = uvm2 + fac1 * epy;
  o.uz = uvm3 + fac1 * epz;
  const double ig = 1.0 / sqrt(1.0 + (o.ux * o.ux + o.uy * o.uy + o.uz * o.uz) / (P.c * P.c));
  o.x = x + o.ux * P.delt * ig;
  o.y = y + o.uy * P.delt * ig;
  o.ig = ig;
  return o;
}

// Shape data of one particle's move for the Esirkepov deposit
// (field.f90:224-268): s0 at the old position around cell (i, j), ds = s1
// shifted by the cell increment minus s0.  Returns false when the particle
// jumped more than one cell.
struct Move {
  double s0x[5], s0y[5], dsx[5], dsy[5];
};

__device__ inline void place_s1(double a, double b, double c, int inc, double *ds) {
  // s1 placed at offset inc (the smo_1..3 selection of field.f90:244-251)
  ds[0] = inc < 0 ? a : 0.0;
  ds[1] = inc < 0 ? b : (inc == 0 ? a : 0.0);
  ds[2] = inc < 0 ? c : (inc == 0 ? b : a);
  ds[3] = inc > 0 ? b : (inc == 0 ? c : 0.0);
  ds[4] = inc > 0 ? c : 0.0;
}

__device__ inline bool make_move(Move &m, double x0, double y0, double x1, double y1, int i,
                                 int j, const PP &P) {
  m.s0x[0] = m.s0x[4] = m.s0y[0] = m.s0y[4] = 0.0;
  shape(x0 * P.d_delx - 0.5 - i, m.s0x[1], m.s0x[2], m.s0x[3]);
  shape(y0 * P.d_delx - 0.5 - j, m.s0y[1], m.s0y[2], m.s0y[3]);
  const int i2 = (int)(x1 * P.d_delx), j2 = (int)(y1 * P.d_delx);
  double a, b, c;
  shape(x1 * P.d_delx - 0.5 - i2, a, b, c);
  place_s1(a, b, c, i2 - i, m.dsx);
  shape(y1 * P.d_delx - 0.5 - j2, a, b, c);
  place_s1(a, b, c, j2 - j, m.dsy);
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    m.dsx[k] -= m.s0x[k];
    m.dsy[k] -= m.s0y[k];
  }
  return (i2 - i >= -1 && i2 - i <= 1) && (j2 - j >= -1 && j2 - j <= 1);
}

// Full 5x5 stencil of one current component (field.f90:274-298) into acc:
//  C = 0: Jx, acc[a*5+b], tile column a+1 (a = 0..3), pjx(ip+1,jp) =
//         pjx(ip,jp) - q dx/dt ds_x(ip) (s0_y(jp) + ds_y(jp)/2)
//  C = 1: Jy, acc[a*4+b], tile row b+1 (b = 0..3), the same along y
//  C = 2: Jz, acc[a*5+b], q gvz (s0x s0y + dsx s0y/2 + s0x dsy/2 + dsx dsy/3)
template <int C>
__device__ inline void stencil(double *acc, const Move &m, double qc, double qv) {
  if (C == 0) {
    double w = 0.0;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      w -= qc * m.dsx[a];
#pragma unroll
      for (int b = 0; b < 5; ++b) acc[a * 5 + b] += w * (m.s0y[b] + 0.5 * m.dsy[b]);
    }
  } else if (C == 1) {
    double w = 0.0;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      w -= qc * m.dsy[b];
#pragma unroll
      for (int a = 0; a < 5; ++a) acc[a * 4 + b] += (m.s0x[a] + 0.5 * m.dsx[a]) * w;
    }
  } else {
    const double third = 1.0 / 3.0;
#pragma unroll
    for (int a = 0; a < 5; ++a) {
      const double za = qv * (m.s0x[a] + 0.5 * m.dsx[a]);
      const double zb = qv * (0.5 * m.s0x[a] + third * m.dsx[a]);
#pragma unroll
      for (int b = 0; b < 5; ++b) acc[a * 5 + b] += za * m.s0y[b] + zb * m.dsy[b];
    }
  }
}

// A particle that stays in its cell has s0 and ds supported on offsets 1..3
// only, so of the 65 stencil values just the 27 below can be non-zero
// (every other value is an exact zero in the reference's arithmetic):
//   Jx tile columns 2..4 x rows 1..3, Jy columns 1..3 x rows 2..4,
//   Jz columns 1..3 x rows 1..3.
// core[0..8] Jx (a-1)*3+(b-1) with a = W index 1..3; core[9..17] Jy
// (a-1)*3+(b-1) with b = W index 1..3; core[18..26] Jz (a-1)*3+(b-1).
__device__ inline void stencil_core(double *core, double x0, double y0, double x1,
                                    double y1, double gvz, int i, int j, double q,
                                    const PP &P) {
  double sx[3], sy[3], dx[3], dy[3];
  shape(x0 * P.d_delx - 0.5 - i, sx[0], sx[1], sx[2]);
  shape(y0 * P.d_delx - 0.5 - j, sy[0], sy[1], sy[2]);
  shape(x1 * P.d_delx - 0.5 - i, dx[0], dx[1], dx[2]);
  shape(y1 * P.d_delx - 0.5 - j, dy[0], dy[1], dy[2]);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    dx[k] -= sx[k];
    dy[k] -= sy[k];
  }
  const double qc = q * P.qc_scale;
  const double qv = q * gvz;
  double X[3], Y[3], wx[3], wy[3];
  double w1 = 0.0, w2 = 0.0;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    X[k] = sx[k] + 0.5 * dx[k];
    Y[k] = sy[k] + 0.5 * dy[k];
    w1 -= qc * dx[k];
    w2 -= qc * dy[k];
    wx[k] = w1;
    wy[k] = w2;
  }
  const double third = 1.0 / 3.0;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const double za = qv * X[a];
    const double zb = qv * (0.5 * sx[a] + third * dx[a]);
#pragma unroll
    for (int b = 0; b < 3; ++b) {
      core[a * 3 + b] += wx[a] * Y[b];
      core[9 + a * 3 + b] += X[a] * wy[b];
      core[18 + a * 3 + b] += za * sy[b] + zb * dy[b];
    }
  }
}

// Index of a core value in the 65-value cell layout of acc_at().
__device__ inline int core_slot(int c) {
  const int comp = c / 9, a = (c % 9) / 3 + 1, b = c % 3 + 1;
  if (comp == 0) return a * 5 + b;             // Jx: W index a -> acc (a, b)
  if (comp == 1) return 20 + a * 4 + b;        // Jy: acc (a, W index b)
  return 40 + a * 5 + b;
}

// Value of accumulator set `cb` (one cell) at tile offset (a, b) for comp.
__device__ inline double acc_at(const double *cb, int comp, int a, int b) {
  if (comp == 0) return a >= 1 ? cb[(a - 1) * 5 + b] : 0.0;
  if (comp == 1) return b >= 1 ? cb[20 + a * 4 + (b - 1)] : 0.0;
  return cb[40 + a * 5 + b];
}

__device__ inline double group_sum(double v) {
  v += __shfl_xor(v, 1, GROUP);
  v += __shfl_xor(v, 2, GROUP);
  v += __shfl_xor(v, 4, GROUP);
  return v;
}

// Contribution of one component of a cell's crossing particles, combined
// over the group and added by lane 0 to cellbuf: the cell's LDS list L (x0,
// y0, x1, y1, q v_z), lane sub taking entries sub, sub + GROUP, ...
template <int C>
__device__ inline void crossing_pass(double *cb, int sub, const double *L, int nl, int i, int j,
                                     double q, const PP &P) {
  constexpr int N = C == 2 ? 25 : 20;
  double acc[N];
#pragma unroll
  for (int k = 0; k < N; ++k) acc[k] = 0.0;
  const double qc = q * P.qc_scale;
  for (int e = sub; e < nl; e += GROUP) {
    Move m;
    make_move(m, L[e], L[MCAP + e], L[2 * MCAP + e], L[3 * MCAP + e], i, j, P);
    stencil<C>(acc, m, qc, L[4 * MCAP + e]);
  }
  const int off = C == 0 ? 0 : (C == 1 ? 20 : 40);
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const double v = group_sum(acc[k]);
    if (sub == 0) cb[off + k] += v;
  }
}

// Element k of a row segment that starts at seg (the same in every lane):
// a 32-bit byte offset from a scalar base, so that no per-lane 64-bit
// address is kept per array.  A segment holds fewer than 2^29 doubles.
__device__ inline double seg_ld(const double *seg, int k) {
  return *(const double *)((const char *)seg + (unsigned)k * 8u);
}
__device__ inline void seg_st(double *seg, int k, double v) {
  *(double *)((char *)seg + (unsigned)k * 8u) = v;
}

// The push alone or the deposit alone, of rows in place (the host-array entry
// points); the resident step's kernel is k_push_step below.
template <bool PUSH, bool DEPOSIT>
__global__ __launch_bounds__(256, 3) void k_particle(
    PP P, const int *__restrict__ cumcnt,
    const double *__restrict__ tmp, int TX, size_t tps,
    const double *__restrict__ xa, const double *__restrict__ ya,
    const double *__restrict__ uxa, const double *__restrict__ uya,
    const double *__restrict__ uza,
    double *__restrict__ xb, double *__restrict__ yb,
    double *__restrict__ uxb, double *__restrict__ uyb,
    double *__restrict__ uzb,
    double *__restrict__ part, int *__restrict__ derr) {
  __shared__ double T[PUSH ? 6 * 3 * TW : 1];
  __shared__ double cellbuf[DEPOSIT ? CHUNK * NACC : 1];
  // per cell: up to MCAP of its movers, as [x0 | y0 | x1 | y1 | q v_z][entry],
  // so that their full stencils need not read the banks again (their lines
  // are gone from L2 by then)
  __shared__ double mvl[DEPOSIT ? CHUNK * 5 * MCAP : 1];
  const int chunk = blockIdx.x;
  const int jl = blockIdx.y;                 // row j = nys + jl
  const int j = P.nys + jl;
  const int i0 = P.nxgs + chunk * CHUNK;
  const int ncell = min(CHUNK, P.nx - chunk * CHUNK);
  if (PUSH) load_tmp_tile<TW>(T, tmp, TX, tps, jl, chunk * CHUNK, min(TW, ncell + 2));
  if (DEPOSIT)
    for (int e = threadIdx.x; e < CHUNK * NACC; e += blockDim.x) cellbuf[e] = 0.0;
  __syncthreads();
  const int g = threadIdx.x / GROUP;
  const int sub = threadIdx.x % GROUP;
  const int i = i0 + g;
  double *cb = cellbuf + g * NACC;
  double *L = mvl + (DEPOSIT ? g * 5 * MCAP : 0);
  const int wg = (threadIdx.x & 63) / GROUP;   // the group's place in its wavefront
  double core[DEPOSIT ? 27 : 1];
  if (DEPOSIT) {
#pragma unroll
    for (int k = 0; k < 27; ++k) core[k] = 0.0;
  }
  int bad = 0;
  if (g < ncell) {
    for (int s = 0; s < P.nsp; ++s) {
      const size_t seg = (size_t)s * P.ny + jl;
      const int *cc = cumcnt + seg * (size_t)(P.nx + 1);
      const int kb = max(0, cc[i - P.nxgs]), ke = min(P.cap, cc[i - P.nxgs + 1]);
      const size_t base = seg * (size_t)P.cap;
      const double q = P.q[s], r = P.r[s];
      const double fac1 = q / r * 0.5 * P.delt;
      const double txxx = fac1 * fac1;
      const double fac2 = q * P.delt / r;
      // windows of 2 GROUP consecutive particles start at the 2 GROUP
      // boundary at or below the cell's first particle, so that each array's
      // load is one aligned 128-byte line for the group; lane sub takes the
      // window's particles sub and GROUP + sub, in that order
      const int ka = kb - kb % (2 * GROUP);
      // bases: the same for the whole workgroup, 32-bit indices below
      const double *Xa = xa + base, *Ya = ya + base;
      const double *Uxa = uxa + base, *Uya = uya + base, *Uza = uza + base;
      double *Xb = xb + base, *Yb = yb + base;
      double *Uxb = uxb + base, *Uyb = uyb + base, *Uzb = uzb + base;
      int mcnt = 0;                            // the list's entries (lane 0's is kept)
      // particle k: pushed and stored, its stay-in-cell stencil added; a
      // crossing one returns true with its deposit inputs
      auto one = [&](int k, double x0, double y0, double cux, double cuy, double cuz, double &x1,
                     double &y1, double &qv) {
        if (k < kb || k >= ke) return false;   // before or after the cell
        double ux, uy, uz;
        // keep the 54 tile values in LDS instead of hoisting them into
        // registers for the whole cell loop (occupancy)
        __asm__ volatile("" ::: "memory");
        int i2, j2;
        if (PUSH) {
          PushOut o = boris(T, g, x0, y0, cux, cuy, cuz, i, j, P, fac1, txxx, fac2);
          x1 = o.x; y1 = o.y;
          i2 = (int)(x1 * P.d_delx);
          j2 = (int)(y1 * P.d_delx);
          seg_st(Xb, k, o.x); seg_st(Yb, k, o.y);
          seg_st(Uxb, k, o.ux); seg_st(Uyb, k, o.uy); seg_st(Uzb, k, o.uz);
        } else {
          x1 = seg_ld(Xb, k); y1 = seg_ld(Yb, k);
          ux = seg_ld(Uxb, k); uy = seg_ld(Uyb, k); uz = seg_ld(Uzb, k);
          i2 = (int)(x1 * P.d_delx);
          j2 = (int)(y1 * P.d_delx);
        }
        if (DEPOSIT) {
          // v_z = u_z / gamma, field.f90:270
          const double gvz = uz / sqrt(1.0 + (ux * ux + uy * uy + uz * uz) / (P.c * P.c));
          if (i2 == i && j2 == j) {
            stencil_core(core, x0, y0, x1, y1, gvz, i, j, q, P);
          } else {
            if (!(i2 - i >= -1 && i2 - i <= 1 && j2 - j >= -1 && j2 - j <= 1)) bad |= DERR_JUMP;
            qv = q * gvz;
            return true;
          }
        }
        return false;
      };
      // a crossing particle goes to the cell's LDS list in (window, lane)
      // order, ranked by a ballot over the group
      auto record = [&](bool cross, double x0, double y0, double x1, double y1, double qv) {
        const unsigned gb = (unsigned)(__ballot(cross) >> (GROUP * wg)) & 0xFFu;
        if (cross) {
          const int e = mcnt + __popc(gb & ((1u << sub) - 1u));
          L[e] = x0;
          L[MCAP + e] = y0;
          L[2 * MCAP + e] = x1;
          L[3 * MCAP + e] = y1;
          L[4 * MCAP + e] = qv;
        }
        mcnt += __popc(gb);
      };
      bool more = kb < ke;
      int k = (more ? ka : ke) + sub;
      // a pass over the cell's windows until the cell ends or some cell's
      // list could overflow in the next window (then the lists are deposited
      // and the pass goes on): the same for the wavefront
      while (__ballot(more) != 0ULL) {
        for (; k - sub < ke && __ballot(mcnt > MCAP - 2 * GROUP) == 0ULL; k += 2 * GROUP) {
          // both halves' loads issued together, each index clamped into the
          // cell's particles (a lane outside them reads a neighbour and idles)
          const int kA = min(max(k, kb), ke - 1), kB = min(max(k + GROUP, kb), ke - 1);
          const double xA = seg_ld(Xa, kA), yA = seg_ld(Ya, kA);
          const double xB = seg_ld(Xa, kB), yB = seg_ld(Ya, kB);
          double uxA = 0, uyA = 0, uzA = 0, uxB = 0, uyB = 0, uzB = 0;
          if (PUSH) {
            uxA = seg_ld(Uxa, kA); uyA = seg_ld(Uya, kA); uzA = seg_ld(Uza, kA);
            uxB = seg_ld(Uxa, kB); uyB = seg_ld(Uya, kB); uzB = seg_ld(Uza, kB);
          }
          // one particle at a time: interleaving the two would need twice the
          // registers of one push and deposit
          double x1, y1, qv = 0.0;
          bool cr = one(k, xA, yA, uxA, uyA, uzA, x1, y1, qv);
          if (DEPOSIT) record(cr, xA, yA, x1, y1, qv);
          __builtin_amdgcn_sched_barrier(0);
          cr = one(k + GROUP, xB, yB, uxB, uyB, uzB, x1, y1, qv);
          if (DEPOSIT) record(cr, xB, yB, x1, y1, qv);
        }
        more = k - sub < ke;
        if (DEPOSIT) {
          // add the stay-in-cell stencils of this species over the 8 lanes
#pragma unroll
          for (int c = 0; c < 27; ++c) {
            const double v = group_sum(core[c]);
            core[c] = 0.0;
            if (sub == 0) cb[core_slot(c)] += v;
          }
          __builtin_amdgcn_wave_barrier();     // the group reads what its lanes listed
          const int nl = __shfl(mcnt, 0, GROUP);
          if (__ballot(nl > 0)) {
            // cell-crossing particles: full 5x5 stencils, one component at a time
            crossing_pass<0>(cb, sub, L, nl, i, j, q, P);
            crossing_pass<1>(cb, sub, L, nl, i, j, q, P);
            crossing_pass<2>(cb, sub, L, nl, i, j, q, P);
          }
          __builtin_amdgcn_wave_barrier();     // the list is read before it is filled again
          mcnt = 0;
        }
      }
    }
  }
  if (bad) atomicOr(derr, bad);
  if (DEPOSIT) {
    __syncthreads();
    // assemble the workgroup tile [b][t][comp] in a fixed order
    double *out = part + ((size_t)jl * P.nchunk + chunk) * TILE;
    for (int e = threadIdx.x; e < TILE; e += blockDim.x) {
      const int comp = e % 3;
      const int t = (e / 3) % DW;
      const int b = e / (3 * DW);
      double sum = 0.0;
      const int glo = max(0, t - 4), ghi = min(ncell - 1, t);
      for (int gg = glo; gg <= ghi; ++gg) sum += acc_at(cellbuf + gg * NACC, comp, t - gg, b);
      out[e] = sum;
    }
  }
}

// ------------------------------------------------ the resident step's push
// Push, particle_x, Esirkepov deposit and the row order's inputs in one pass
// over the particles: read through the pending order (Order::perm), written
// sorted, 40 bytes each way, plus 4 bytes of index and 2 of code.
//
// A group of 8 or 16 lanes per cell (wm_k_push_step), in steps of as many
// consecutive particles.  Loads run two steps ahead of their use and indexes
// four; a step's results wait in registers and are stored in front of the next
// step's loads, since loads and stores complete in order and whatever is waited
// for should have been issued two steps ago.  A workgroup is 8 cells, one
// wavefront or two: with eight wavefronts and 32 cells, more than half of the
// wavefronts' time went into waiting for the densest cells of the workgroup at
// its end.
//
// Per cell, over all species: 21 stay-in-cell stencil values per lane (of the
// 27 values of the 3 x 3 cores, Jx's last column and Jy's last row carry the
// sum of all three shape changes, which is zero), and a list of the crossing
// particles in LDS, summed when some cell's list could overflow in the next
// two steps and at the end.  A hot plasma has a third of its particles cross a
// cell's edge in a step, so the movers are half of the work: see mover_sums.
//
// The TSC gather of particle.f90:107-129 inside a cell is a biquadratic in
// the in-cell offsets: nine coefficients per field and cell (LDS), 8 FMAs a
// field.
//
// Two wavefronts a SIMD (197 registers with 16 lanes a cell, 224 with 8): bound by FP64 operations (half of the
// issue slots) and the memory path together; alone, loads and stores take 0.92
// ms and the arithmetic 0.91 at 1024 x 512 cells with 32 per cell, both 1.1.
// Measured against 8 lanes a cell, 32 cells and lists summed component by
// component: 2048 x 2048, 64 per cell: 18.9 -> 15.6 ms; 256 x 64, 64 per cell,
// pinched: 224 -> 128 us; 1024 x 512, 32 per cell: 1.68 -> 1.37 ms; 499 x 309, 21
// per cell: 424 -> 325 us.
constexpr int PCH = WM_CHUNK_STEP64;  // cells of a workgroup
constexpr int PTW = PCH + 2, PDW = PCH + 4, PTILE = 5 * PDW * 3;
constexpr int CFN = 10;               // doubles per field and cell (9 coefficients, padded)
constexpr int NCORE = 21;

// w-(o) = 1/2 - o + o^2/2, w0(o) = 1/2 + o - o^2, w+(o) = o^2/2:
// sum_ab T(a, b) w_a(ox) w_b(oy) = sum_ij C_ij ox^i oy^j, C row i at 3 i.
__device__ inline void cell_coeffs(double *cf, const double *Tk) {
  constexpr int TW = PTW;
  double R[3][3];
#pragma unroll
  for (int b = 0; b < 3; ++b) {
    const double m = Tk[b * TW], z = Tk[b * TW + 1], p = Tk[b * TW + 2];
    R[b][0] = 0.5 * (m + z);
    R[b][1] = z - m;
    R[b][2] = 0.5 * ((m - z) + (p - z));
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    cf[3 * i] = 0.5 * (R[0][i] + R[1][i]);
    cf[3 * i + 1] = R[1][i] - R[0][i];
    cf[3 * i + 2] = 0.5 * ((R[0][i] - R[1][i]) + (R[2][i] - R[1][i]));
  }
}

// A square that has overflowed (a momentum above 1e154) as one of the largest
// numbers, by one 32-bit operation (a NaN becomes a number too: the momentum it
// comes from is none).
__device__ inline double below_inf(double a) {
  return __hiloint2double((int)min((unsigned)__double2hiint(a), 0x7FEFFFFFu), __double2loint(a));
}
// 1 / sqrt(a), a > 0 normal: the hardware's estimate (to about 2^-23) and two
// Newton steps in FMAs, within an ulp.  At infinity the estimate is zero, as the
// quotient is, and the steps leave it there.
__device__ inline double rsqrt64(double a) {
  double y = __builtin_amdgcn_rsq(a);
  a = below_inf(a);
  double h = 0.5 * y;
  double e = fma(-a * y, h, 0.5);      // 1/2 - a y^2 / 2
  y = fma(y, e, y);
  h = 0.5 * y;
  const double g = a * y;              // sqrt(a) to twice the estimate's bits
  e = fma(-g, h, 0.5);
  return fma(y, e, y);
}

__device__ inline PushOut boris_coeffs(const double2 *cf, double ox, double oy, double x, double y,
                                       double ux, double uy, double uz, const PP &P, double fac1,
                                       double txxx, double fac2) {
  double f[6];
#pragma unroll
  for (int kk = 0; kk < 6; ++kk) {
    const int k = (kk + 3) % 6;
    const double2 a = cf[5 * k], b = cf[5 * k + 1], c = cf[5 * k + 2], d = cf[5 * k + 3],
                  e = cf[5 * k + 4];
    const double r0 = fma(oy, fma(oy, b.x, a.y), a.x);
    const double r1 = fma(oy, fma(oy, c.y, c.x), b.y);
    const double r2 = fma(oy, fma(oy, e.x, d.y), d.x);
    f[k] = fma(ox, fma(ox, r2, r1), r0);
    __asm__ volatile("" ::: "memory");   // one field's coefficients in registers at a time
  }
  const double bpx = f[0], bpy = f[1], bpz = f[2];
  const double epx = f[3], epy = f[4], epz = f[5];
  // particle.f90:131-161
  double uvm1 = ux + fac1 * epx;
  double uvm2 = uy + fac1 * epy;
  double uvm3 = uz + fac1 * epz;
  // fac2 / (gam + txxx b^2 / gam) by igam alone, which is zero where gam has
  // overflowed
  const double igam = rsqrt64(P.c * P.c + uvm1 * uvm1 + uvm2 * uvm2 + uvm3 * uvm3);
  const double fac1r = fac1 * igam;
  const double fac2r =
      fac2 * igam / fma(txxx * (bpx * bpx + bpy * bpy + bpz * bpz) * igam, igam, 1.0);
  const double uvm4 = uvm1 + fac1r * (uvm2 * bpz - uvm3 * bpy);
  const double uvm5 = uvm2 + fac1r * (uvm3 * bpx - uvm1 * bpz);
  const double uvm6 = uvm3 + fac1r * (uvm1 * bpy - uvm2 * bpx);
  uvm1 = uvm1 + fac2r * (uvm5 * bpz - uvm6 * bpy);
  uvm2 = uvm2 + fac2r * (uvm6 * bpx - uvm4 * bpz);
  uvm3 = uvm3 + fac2r * (uvm4 * bpy - uvm5 * bpx);
  PushOut o;
  o.ux = uvm1 + fac1 * epx;
  o.uy = uvm2 + fac1 * epy;
  o.uz = uvm3 + fac1 * epz;
  const double ig = rsqrt64(1.0 + (o.ux * o.ux + o.uy * o.uy + o.uz * o.uz) * P.ic2);
  o.x = x + o.ux * P.delt * ig;
  o.y = y + o.uy * P.delt * ig;
  o.ig = ig;
  return o;
}

// Weights at the cell's -1, 0, +1 neighbours for the old offset o0 and their
// change to o1 in the same cell, taken directly: d+ = (o1 - o0)(o1 + o0) / 2,
// d- = (o1 - o0)(o1 + o0 - 2) / 2, d0 = -(d- + d+).
__device__ inline void shape_delta(double o0, double o1, double *s, double *d) {
  const double t = 1.0 - o0;
  s[0] = (0.5 * t) * t;
  s[2] = (0.5 * o0) * o0;
  s[1] = (1.0 - s[0]) - s[2];
  const double hd = 0.5 * (o1 - o0), sg = o1 + o0;
  d[2] = hd * sg;
  d[0] = hd * (sg - 2.0);
  d[1] = -(d[0] + d[2]);
}

// A particle that stays in its cell: Jx (a < 2, b < 3) at 0..5, Jy (a < 3,
// b < 2) at 6..11, Jz (3 x 3) at 12..20.  Jx and Jy weigh -q dx/dt times the
// running sum of the shape changes: -qc d-, then qc d+ (their sum is zero).
// Jz's s0x s0y + dx s0y / 2 + s0x dy / 2 + dx dy / 3 is X Y + dx dy / 12 with
// X = s0x + dx / 2, Y = s0y + dy / 2.
__device__ inline void core_add(double *core, double ox0, double oy0, double ox1, double oy1,
                                double qc, double qv) {
  double sx[3], sy[3], dx[3], dy[3], X[3], Y[3];
  shape_delta(ox0, ox1, sx, dx);
  shape_delta(oy0, oy1, sy, dy);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    X[k] = fma(0.5, dx[k], sx[k]);
    Y[k] = fma(0.5, dy[k], sy[k]);
  }
  const double wx0 = -(qc * dx[0]), wx1 = qc * dx[2];
  const double wy0 = -(qc * dy[0]), wy1 = qc * dy[2];
#pragma unroll
  for (int b = 0; b < 3; ++b) {
    core[b] = fma(wx0, Y[b], core[b]);
    core[3 + b] = fma(wx1, Y[b], core[3 + b]);
  }
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    core[6 + 2 * a] = fma(X[a], wy0, core[6 + 2 * a]);
    core[7 + 2 * a] = fma(X[a], wy1, core[7 + 2 * a]);
  }
  const double qv12 = qv * (1.0 / 12.0);
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const double za = qv * X[a], zb = qv12 * dx[a];
#pragma unroll
    for (int b = 0; b < 3; ++b) {
      double &c = core[12 + a * 3 + b];
      c = fma(za, Y[b], c);
      c = fma(zb, dy[b], c);
    }
  }
}

// Slot of core value e in the 65-value cell layout of acc_at().
__device__ inline int core_at(int e) {
  if (e < 6) return (1 + e / 3) * 5 + 1 + e % 3;                 // Jx: tile column 2 + a
  if (e < 12) return 20 + (1 + (e - 6) / 2) * 4 + 1 + (e - 6) % 2;   // Jy: tile row 2 + b
  return 40 + (1 + (e - 12) / 3) * 5 + 1 + (e - 12) % 3;
}

template <int CTRL>
__device__ inline double dpp_f64(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xF, 0xF, true);
  return __longlong_as_double((long long)(unsigned)lo | ((long long)hi << 32));
}

// Sums of 24 values over the 8 or 16 lanes of a group, by halving: in each
// exchange a lane keeps one half of the values and adds its partner's share of
// them (partners: lane xor 8, the mirrored lane of its eight, lane xor 2, and
// lane xor 1; of 16 lanes the last adds the three that are left).  Lane sub
// ends with the sums of values slot .. slot + 2, which it returns, in v[0..2];
// of 16 lanes the odd ones have what the even ones have.  About 6
// instructions a value against 12 or 15 for a butterfly of each.
template <int M, int CTRL>
__device__ inline void halve(double *v, bool up) {
#pragma unroll
  for (int e = 0; e < M / 2; ++e) {
    const double a = v[e], b = v[M / 2 + e];
    const double keep = up ? b : a, give = up ? a : b;
    v[e] = keep + dpp_f64<CTRL>(give);
  }
}
template <int PG>
__device__ inline int group_sums(double *v, int sub) {
  if (PG == 8) {
    halve<24, 0x141>(v, sub & 4);        // row_half_mirror: lane 7 - sub of its eight
    halve<12, 0x4E>(v, sub & 2);         // quad_perm [2,3,0,1]
    halve<6, 0xB1>(v, sub & 1);          // quad_perm [1,0,3,2]
    return ((sub >> 2) & 1) * 12 + ((sub >> 1) & 1) * 6 + (sub & 1) * 3;
  }
  halve<24, 0x128>(v, sub & 8);          // row_ror:8: lane xor 8
  halve<12, 0x141>(v, sub & 4);
  halve<6, 0x4E>(v, sub & 2);
#pragma unroll
  for (int e = 0; e < 3; ++e) v[e] += dpp_f64<0xB1>(v[e]);
  return ((sub >> 3) & 1) * 12 + ((sub >> 2) & 1) * 6 + ((sub >> 1) & 1) * 3;
}

// acc[a] += gx[a] V + dx[a] W with gx and dx those of lane N of the row of 16.
// One instruction a product: the row broadcast is the multiply-add's own
// operand modifier (the wait covers it after a write of gx or dx).
template <int N>
__device__ inline void add_outer(double (&acc)[5], const double (&gx)[5], const double (&dx)[5],
                                 double V, double W) {
#define WM_ROW "row_newbcast:%17 row_mask:0xf bank_mask:0xf\n\t"
  __asm__("s_nop 4\n\t"
          "v_fmac_f64_dpp %0, %5, %15 " WM_ROW "v_fmac_f64_dpp %1, %6, %15 " WM_ROW
          "v_fmac_f64_dpp %2, %7, %15 " WM_ROW "v_fmac_f64_dpp %3, %8, %15 " WM_ROW
          "v_fmac_f64_dpp %4, %9, %15 " WM_ROW "v_fmac_f64_dpp %0, %10, %16 " WM_ROW
          "v_fmac_f64_dpp %1, %11, %16 " WM_ROW "v_fmac_f64_dpp %2, %12, %16 " WM_ROW
          "v_fmac_f64_dpp %3, %13, %16 " WM_ROW "v_fmac_f64_dpp %4, %14, %16 " WM_ROW
          : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3]), "+v"(acc[4])
          : "v"(gx[0]), "v"(gx[1]), "v"(gx[2]), "v"(gx[3]), "v"(gx[4]), "v"(dx[0]), "v"(dx[1]),
            "v"(dx[2]), "v"(dx[3]), "v"(dx[4]), "v"(V), "v"(W), "n"(N));
#undef WM_ROW
}

// The listed movers' current, added to the lanes' sums (with 8 lanes a cell A
// and B are those of the row's two cells; with 16 A).  PG movers of a cell at a
// time: lane sub prepares its cell's mover e0 + sub and keeps its x side, the y
// sides go to LDS (Y: the cell's; Ya, Yb: the row's first and second cell's),
// and the row's 16 lanes take the movers of its cells one after the other.
// No reduction: a lane's sums are its own.  All 64 lanes call it.
// (One component after another over the list, a lane a mover, took three
// passes over the shapes and 80 values through the lanes' reduction: 471
// million vector instructions a step at 1024 x 512 against 339.)
template <int PG>
__device__ inline void outer_sums(double (&A)[5], double (&B)[5], const double (&gx)[5],
                                  const double (&dx)[5], const double *Ya, const double *Yb,
                                  const Role &r, bool jy, unsigned long long has) {
  auto factors = [&](const double *y, double &V, double &W) {
    const double p = y[r.p < 0 ? 0 : r.p], s = y[r.s], w = y[r.w < 0 ? 0 : r.w], t = y[r.t];
    V = r.p < 0 ? 0.0 : (jy ? p : p * s);
    W = r.w < 0 ? 0.0 : w * t;
  };
#define WM_PAIR(N0)                                                                 \
  if (has & (0x0001000100010001ULL << (N0))) {                                      \
    double V0, W0, V1, W1;                                                          \
    const double *y = (PG == 8 && (N0) >= 8 ? Yb : Ya) + ((N0) & (PG - 1)) * YN;    \
    factors(y, V0, W0);                                                             \
    factors(y + YN, V1, W1);                                                        \
    add_outer<(N0)>(PG == 8 && (N0) >= 8 ? B : A, gx, dx, V0, W0);                  \
    add_outer<(N0) + 1>(PG == 8 && (N0) >= 8 ? B : A, gx, dx, V1, W1);              \
  }
  WM_PAIR(0) WM_PAIR(2) WM_PAIR(4) WM_PAIR(6)
  WM_PAIR(8) WM_PAIR(10) WM_PAIR(12) WM_PAIR(14)
#undef WM_PAIR
}
template <int PG, int MLC>
__device__ inline void mover_sums(double (&A)[5], double (&B)[5], int sub, const double *L,
                                  const uint8_t *Ls, double *Y, const double *Ya,
                                  const double *Yb, const Role &r, int nl, int i, int j,
                                  const PP &P, const double *qcs) {
  const bool jy = r.out >= 20 && r.out < 40;
  for (int e0 = 0; __ballot(e0 < nl) != 0ULL; e0 += PG) {
    const int e = e0 + sub;
    const unsigned long long has = __ballot(e < nl);
    double gx[5], dx[5], gy[5], dy[5], qv = 0.0, qc = 0.0;
    if (e < nl) {
      Move m;
      make_move(m, L[e], L[MLC + e], L[2 * MLC + e], L[3 * MLC + e], i, j, P);
      qv = L[4 * MLC + e];
      qc = qcs[Ls[e]];
#pragma unroll
      for (int k = 0; k < 5; ++k) {
        dx[k] = m.dsx[k];
        dy[k] = m.dsy[k];
        gx[k] = fma(0.5, dx[k], m.s0x[k]);
        gy[k] = fma(0.5, dy[k], m.s0y[k]);
      }
    } else {
#pragma unroll
      for (int k = 0; k < 5; ++k) gx[k] = dx[k] = gy[k] = dy[k] = 0.0;
    }
    double *y = Y + sub * YN, w = 0.0;
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      y[k] = gy[k];
      y[9 + k] = dy[k];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      w -= qc * dy[k];
      y[5 + k] = w;
    }
    y[14] = qv;
    y[15] = qv * (1.0 / 12.0);
    y[16] = -qc;
    __builtin_amdgcn_wave_barrier();
    outer_sums<PG>(A, B, gx, dx, Ya, Yb, r, jy, has);
    __builtin_amdgcn_wave_barrier();
  }
}

struct Part {
  double x, y, ux, uy, uz;
};

// A loaded particle in registers of its own, so that the next load can have
// the old ones: left to itself the compiler loads elsewhere and copies at the
// end of the step, which waits for everything in flight.
__device__ inline Part take(const Part &n) {
  Part c;
  __asm__ volatile("v_mov_b64 %0, %5\n\tv_mov_b64 %1, %6\n\tv_mov_b64 %2, %7\n\t"
                   "v_mov_b64 %3, %8\n\tv_mov_b64 %4, %9"
                   : "=&v"(c.x), "=&v"(c.y), "=&v"(c.ux), "=&v"(c.uy), "=&v"(c.uz)
                   : "v"(n.x), "v"(n.y), "v"(n.ux), "v"(n.uy), "v"(n.uz));
  return c;
}

template <int SRC, bool WALLS, int PG>
__global__ __launch_bounds__(PCH * PG, 2) void k_push_step(PP P, const int *__restrict__ cumcnt,
                                                      const double *__restrict__ tmp, int TX,
                                                      size_t tps, Rec64 A, Rec64 B, Order O,
                                                      double *__restrict__ part,
                                                      int *__restrict__ derr,
                                                      unsigned long long *ts) {
  wm_stamp(ts, 1);
  constexpr int PTH = PCH * PG;
  constexpr int MLC = PG == 8 ? 23 : 47;       // a cell's listed movers
  __shared__ __attribute__((aligned(16))) double CF[PCH * 6 * CFN];
  // the movers' lists [x0 | y0 | x1 | y1 | q v_z][entry] per cell and their y
  // sides; before them, the chunk's cell-centred fields, behind them the
  // cells' sums
  __shared__ double mvl[PCH * (5 * MLC + YN * PG)];
  __shared__ uint8_t mvs[PCH * MLC];       // the entries' species
  __shared__ int mk[PCH * 4];              // moves out of a cell: left, right, others
  __shared__ double qcs[WM_MAXSP];         // q delx / dt of the species
  static_assert(6 * 3 * PTW <= PCH * 5 * MLC && NACC <= 5 * MLC + YN * PG,
                "the fields and the sums fit the lists' space");
  double *T = mvl, *cellbuf = mvl;
  // consecutive chunks on one XCD, which then has both parts of the lines that
  // two of them share (workgroups go to the 8 XCDs in turn)
  const unsigned nb = gridDim.x, per = nb / 8, cut = nb - per * 8;
  const unsigned xcd = blockIdx.x % 8, at = xcd * per + min(xcd, cut) + blockIdx.x / 8;
  const int chunk = at % P.nchunk;
  const int jl = at / P.nchunk;              // row j = nys + jl
  const int j = P.nys + jl;
  const int i0 = P.nxgs + chunk * PCH;
  const int ncell = min(PCH, P.nx - chunk * PCH);
  const int g = threadIdx.x / PG;
  const int sub = threadIdx.x % PG;
  const int il = chunk * PCH + g, i = i0 + g;
  // a species' slots of this group's cell (none beyond the row's cells)
  int kb, ke, kbn = 0, ken = 0;                // this species, the next
  auto slots = [&](int s, int &b, int &e) {
    b = e = 0;
    if (g < ncell && s < P.nsp) {
      const int *cc = cumcnt + ((size_t)s * P.ny + jl) * (size_t)(P.nx + 1) + il;
      b = max(0, cc[0]);
      e = max(b, min(P.cap, cc[1]));
    }
  };
  // the particle of slot q: where it is, and itself
  auto src = [&](int s, int q, int b, int e) {
    q = max(0, min(max(q, b), e - 1));
    const unsigned p =
        SRC == SRC_SLOT ? (unsigned)q : O.perm[((size_t)s * P.ny + jl) * (size_t)P.cap + q];
    return b == e ? 0u : p;                    // an empty cell's is not read
  };
  auto load = [&](int s, unsigned p) {
    const size_t sb = SRC == SRC_SLOT ? ((size_t)s * P.ny + jl) * (size_t)P.cap
                                      : (size_t)s * P.ny * (size_t)P.cap;
    const double *Xa = A.x + sb, *Ya = A.y + sb, *Uxa = A.ux + sb, *Uya = A.uy + sb, *Uza = A.uz + sb;
    if (SRC == SRC_PERM64)
      return Part{Xa[(size_t)p], Ya[(size_t)p], Uxa[(size_t)p], Uya[(size_t)p], Uza[(size_t)p]};
    return Part{seg_ld(Xa, (int)p), seg_ld(Ya, (int)p), seg_ld(Uxa, (int)p), seg_ld(Uya, (int)p),
                seg_ld(Uza, (int)p)};
  };
  // The chains of loads that start a species (slots, places, particles) run
  // beside the fields' here, and the second species' beside the first's.
  if (threadIdx.x < WM_MAXSP) qcs[threadIdx.x] = P.q[threadIdx.x] * P.qc_scale;
  slots(0, kb, ke);
  slots(1, kbn, ken);
  load_tmp_tile<PTW>(T, tmp, TX, tps, jl, chunk * PCH, min(PTW, ncell + 2));
  int k = kb + sub;
  const unsigned p0 = src(0, k, kb, ke), p1 = src(0, k + PG, kb, ke);
  // where the particles of the two steps after those in n0 and n1 come from
  unsigned f0 = src(0, k + 2 * PG, kb, ke), f1 = src(0, k + 3 * PG, kb, ke);
  const int kn = kbn + sub;
  unsigned q0 = 0, q1 = 0, q2 = 0, q3 = 0;
  if (P.nsp > 1) {
    q0 = src(1, kn, kbn, ken);
    q1 = src(1, kn + PG, kbn, ken);
    q2 = src(1, kn + 2 * PG, kbn, ken);
    q3 = src(1, kn + 3 * PG, kbn, ken);
  }
  __syncthreads();
  Part n0 = load(0, p0), n1 = load(0, p1);     // the next two steps' particles
  if (threadIdx.x < PCH * 6) {
    const int c = threadIdx.x % PCH, k = threadIdx.x / PCH;
    cell_coeffs(CF + (c * 6 + k) * CFN, T + k * 3 * PTW + c);
  }
  __syncthreads();
  double *cb = cellbuf + g * NACC;
  double *L = mvl + g * 5 * MLC;
  double *Ys = mvl + PCH * 5 * MLC;
  uint8_t *Ls = mvs + g * MLC;
  const double2 *cf = (const double2 *)(CF + g * 6 * CFN);
  const int wg = (threadIdx.x & 63) / PG;   // the group's place in its wavefront
  const Role role = role_of(threadIdx.x & 15);
  int bad = 0;
  double core[24], mv[5], mw[5];               // the cell's own sums, its movers' (8 lanes: the
                                               // row's two cells' movers')
#pragma unroll
  for (int e = 0; e < 24; ++e) core[e] = 0.0;
#pragma unroll
  for (int e = 0; e < 5; ++e) mv[e] = mw[e] = 0.0;
  {
    // The step's results wait in registers and are stored at the top of the
    // next, in front of its loads: loads and stores complete in order, and
    // whatever is waited for was issued a whole step earlier.
    Part out{};
    unsigned ocd = 0;
    int ok = -1;                               // their slot, -1: none
    int mcnt = 0;                              // the list's entries
    if (sub < 4) mk[g * 4 + sub] = 0;
    for (int s = 0;;) {
      const size_t seg = (size_t)s * P.ny + jl, base = seg * (size_t)P.cap;
      const double q = P.q[s], r = P.r[s];
      const double fac1 = q / r * 0.5 * P.delt;
      const double txxx = fac1 * fac1;
      const double fac2 = q * P.delt / r;
      const double qc = q * P.qc_scale;
      auto put = [&] {
        if (ok < 0) return;
        O.code[base + ok] = (uint16_t)ocd;
        seg_st(B.x + base, ok, out.x);
        seg_st(B.y + base, ok, out.y);
        seg_st(B.ux + base, ok, out.ux);
        seg_st(B.uy + base, ok, out.uy);
        seg_st(B.uz + base, ok, out.uz);
        ok = -1;
      };
      auto step = [&](Part &n, unsigned &f) {
        const Part c = take(n);
        put();
        n = load(s, f);
        f = src(s, k + 4 * PG, kb, ke);
        bool cross = false;
        double qv = 0.0, x1 = 0.0, y1 = 0.0;
        if (k >= kb && k < ke) {
          const double ox = c.x * P.d_delx - i, oy = c.y * P.d_delx - j;
          PushOut o = boris_coeffs(cf, ox, oy, c.x, c.y, c.ux, c.uy, c.uz, P, fac1, txxx, fac2);
          if (WALLS && P.inj) injection_edge(o.x, o.ux, o.uy, o.uz, P);
          x1 = o.x;
          y1 = o.y;
          const int i2 = (int)(x1 * P.d_delx), j2 = (int)(y1 * P.d_delx);
          cross = i2 != i || j2 != j;
          // field.f90:270's v_z = u_z / gamma with the push's 1 / gamma of the
          // same u, except where the shock's injection edge may have
          // reflected it
          const double gvz = !(WALLS && P.inj) ? o.uz * o.ig
                                    : o.uz / sqrt(1.0 + (o.ux * o.ux + o.uy * o.uy + o.uz * o.uz) /
                                                            (P.c * P.c));
          qv = q * gvz;
          if (!cross) core_add(core, ox, oy, x1 * P.d_delx - i, y1 * P.d_delx - j, qc, qv);
          unsigned cd = (unsigned)il << 2;
          if (cross || (WALLS && P.xmode == 2)) {
            // particle_x and particle_y of the stored state (the deposit takes
            // the unwrapped one), as boundary_periodic.f90 and the wall
            // families' particle_x write them
            if (!(i2 - i >= -1 && i2 - i <= 1)) bad |= DERR_JUMP;
            int inew = i2;
            if (!WALLS) {
              if (i2 < P.nxgs) o.x = wm_edges::add_rd(o.x, P.spanx);
              else if (i2 >= P.nxgs + P.nx) o.x = wm_edges::add_rd(o.x, -P.spanx);
              inew = (int)o.x;
            } else if (P.xmode == 2) {
              const bool lo = i2 < P.xs + 1, hi = i2 >= P.xe - 1;
              if (lo || hi) {
                o.x = (lo ? P.wl : P.wr) - o.x;
                o.ux = -o.ux;
                o.uy = -o.uy;
                o.uz = -o.uz;
                inew = (int)o.x;
              }
            }
            const int d = j2 - j;
            if (j2 < P.nys) o.y = wm_edges::add_rd(o.y, P.spany);
            else if (j2 >= P.nys + P.ny) o.y = wm_edges::add_rd(o.y, -P.spany);
            int cn = inew - P.nxgs;
            if (cn < 0 || cn >= P.nx) {
              bad |= DERR_RANGE;
              cn = min(max(cn, 0), P.nx - 1);
            }
            if (d < -1 || d > 1) bad |= DERR_JUMP;
            int dc = cn - il;
            if (!WALLS) dc = dc == P.nx - 1 ? -1 : (dc == 1 - P.nx ? 1 : dc);
            const bool out = d == 1 || d == -1, far = !out && (dc < -1 || dc > 1);
            cd = (unsigned)cn << 2 | (out ? (d == 1 ? WM_CODE_UP : WM_CODE_DOWN)
                                          : (far ? WM_CODE_FAR : WM_CODE_STAY));
            if (far) {                         // (a wall's mirror from a cell beyond it)
              atomicAdd(O.farcnt + seg * P.nx + cn, 1);
              O.far[seg] = 1;
            }
            if (out || dc != 0) atomicAdd(&mk[g * 4 + (out || far ? 2 : (dc < 0 ? 0 : 1))], 1);
          }
          out = Part{o.x, o.y, o.ux, o.uy, o.uz};
          ocd = cd;
          ok = k;
        }
        // a crossing particle goes to the cell's list in (step, lane) order,
        // ranked by a ballot over the group
        const unsigned gb = (unsigned)(__ballot(cross) >> (PG * wg)) & ((1u << PG) - 1u);
        if (cross) {
          const int e = mcnt + __popc(gb & ((1u << sub) - 1u));
          L[e] = c.x;
          L[MLC + e] = c.y;
          L[2 * MLC + e] = x1;
          L[3 * MLC + e] = y1;
          L[4 * MLC + e] = qv;
          Ls[e] = (uint8_t)s;
        }
        mcnt += __popc(gb);
        k += PG;
      };
      for (; k - sub < ke && __ballot(mcnt > MLC - 2 * PG) == 0ULL;) {
        step(n0, f0);
        if (__ballot(k - sub < ke) == 0ULL) break;   // (the next species' loads start anew)
        step(n1, f1);
      }
      put();
      if (__ballot(k - sub < ke) == 0ULL) {    // every cell's particles of this species are done
        __builtin_amdgcn_wave_barrier();
        if (sub == 0 && g < ncell) {
          const int l = mk[g * 4], rr = mk[g * 4 + 1], o = mk[g * 4 + 2];
          O.kind[seg * P.nx + il] = make_int4(l, ke - kb - l - rr - o, rr, o);
        }
        __builtin_amdgcn_wave_barrier();
        if (++s < P.nsp) {
          if (sub < 4) mk[g * 4 + sub] = 0;
          kb = kbn;
          ke = ken;
          k = kb + sub;
          if (s > 1) {
            q0 = src(s, k, kb, ke);
            q1 = src(s, k + PG, kb, ke);
            q2 = src(s, k + 2 * PG, kb, ke);
            q3 = src(s, k + 3 * PG, kb, ke);
          }
          n0 = load(s, q0);
          n1 = load(s, q1);
          f0 = q2;
          f1 = q3;
          slots(s + 1, kbn, ken);
          continue;
        }
      }
      __builtin_amdgcn_wave_barrier();         // the group reads what its lanes listed
      const int ga = PG == 8 ? g & ~1 : g, gb = PG == 8 ? g | 1 : g;
      mover_sums<PG, MLC>(mv, mw, sub, L, Ls, Ys + g * (YN * PG), Ys + ga * (YN * PG),
                          Ys + gb * (YN * PG), role, mcnt, i, j, P, qcs);
      mcnt = 0;
      if (s == P.nsp) break;
    }
  }
  if (bad) atomicOr(derr, bad);
  __syncthreads();                             // the lists' space is free
  if (PG == 8) {
    put_sums(cellbuf + (g & ~1) * NACC, role, mv);
    put_sums(cellbuf + (g | 1) * NACC, role, mw);
  } else {
    put_sums(cb, role, mv);
  }
  __builtin_amdgcn_wave_barrier();
  const int s0 = group_sums<PG>(core, sub);
  if (PG == 8 || (sub & 1) == 0) {
#pragma unroll
    for (int e = 0; e < 3; ++e)
      if (s0 + e < NCORE) cb[core_at(s0 + e)] += core[e];
  }
  __syncthreads();
  // assemble the workgroup tile [b][t][comp] in a fixed order
  double *out = part + ((size_t)jl * P.nchunk + chunk) * PTILE;
  for (int e = threadIdx.x; e < PTILE; e += PTH) {
    const int comp = e % 3;
    const int t = (e / 3) % PDW;
    const int b = e / (3 * PDW);
    double sum = 0.0;
    const int glo = max(0, t - 4), ghi = min(ncell - 1, t);
    for (int gg = glo; gg <= ghi; ++gg) sum += acc_at(cellbuf + gg * NACC, comp, t - gg, b);
    out[e] = sum;
  }
}

// Cell-centred fields, particle.f90:68-81, on cells nxs-1..nxe+1, nys-1..nye+1.
// Also clears the rows' far marks for the push that follows.
__global__ void k_cell_fields(FieldGeom fg, const double *__restrict__ uf,
                              double *__restrict__ tmp, int TX, int TY, size_t tps,
                              int *__restrict__ far, int nseg, unsigned long long *ts) {
  wm_stamp(ts, 0);
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < nseg) far[t] = 0;
  if (t >= TX * TY) return;
  const int a = t % TX, b = t / TX;
  // cell (i, j) = (nxs-1+a, nys-1+b) -> ghost-inclusive local (a+1, b+1)
  const size_t c0 = (size_t)(a + 1) + (size_t)fg.gx * (size_t)(b + 1);
  const size_t gx = fg.gx;
  const double *B1 = uf, *B2 = uf + fg.ps, *B3 = uf + 2 * fg.ps;
  const double *E1 = uf + 3 * fg.ps, *E2 = uf + 4 * fg.ps, *E3 = uf + 5 * fg.ps;
  tmp[t] = 0.5 * (B1[c0] + B1[c0 + gx]);
  tmp[tps + t] = 0.5 * (B2[c0] + B2[c0 + 1]);
  tmp[2 * tps + t] = 0.25 * (B3[c0] + B3[c0 + 1] + B3[c0 + gx] + B3[c0 + gx + 1]);
  tmp[3 * tps + t] = 0.5 * (E1[c0] + E1[c0 + 1]);
  tmp[4 * tps + t] = 0.5 * (E2[c0] + E2[c0 + gx]);
  tmp[5 * tps + t] = E3[c0];
}

PP make_pp(const wm_ctx *ctx) {
  PP P;
  const wm_grid &g = ctx->g;
  P.nx = g.nx; P.ny = g.ny; P.nxgs = g.nxgs; P.nys = g.nys; P.nsp = g.nsp;
  P.cap = ctx->cap;
  P.nchunk = wm_cdiv(g.nx, CHUNK);
  P.d_delx = 1.0 / g.delx;
  P.delt = g.delt;
  P.c = g.c;
  P.ic2 = 1.0 / (g.c * g.c);
  P.qc_scale = g.delx * (1.0 / g.delt);
  for (int s = 0; s < WM_MAXSP; ++s) {
    P.q[s] = s < g.nsp ? g.q[s] : 0.0;
    P.r[s] = s < g.nsp ? g.r[s] : 1.0;
  }
  P.inj = 0;
  P.xs = ctx->xe > 0 ? ctx->xs : g.nxgs;
  P.delx = g.delx;
  P.wl = 2.0 * (P.xs + 1) * g.delx;
  P.xend = 0.0;
  P.u0 = 0.0;
  P.xmode = 0;
  P.xe = ctx->xe > 0 ? ctx->xe : g.nxge;
  P.spanx = (double)(g.nxge - g.nxgs + 1) * g.delx;
  P.spany = (double)(g.nyge - g.nygs + 1) * g.delx;
  P.wr = 2.0 * (P.xe - 1) * g.delx;
  return P;
}

template <bool PUSH, bool DEP>
int launch_particle(wm_ctx *ctx, int a, int b) {
  const PP P = make_pp(ctx);
  const int TX = ctx->g.nx + 2;
  const size_t tps = (size_t)TX * (size_t)(ctx->g.ny + 2);
  const PBank &A = ctx->bank[a];
  const PBank &B = ctx->bank[b];
  hipLaunchKernelGGL((k_particle<PUSH, DEP>), dim3(P.nchunk, P.ny), dim3(256), 0, ctx->stream, P,
                     ctx->cumcnt, ctx->tmp, TX, tps, A.x, A.y, A.ux, A.uy, A.uz,
                     B.x, B.y, B.ux, B.uy, B.uz, ctx->dep_part, ctx->derr);
  WM_HIP(hipGetLastError());
  return WM_OK;
}

}  // namespace

size_t wm_deposit_part_elems(int nx, int ny) {
  return (size_t)ny * std::max((size_t)wm_cdiv(nx, CHUNK) * TILE, (size_t)wm_cdiv(nx, PCH) * PTILE);
}

int wm_k_cell_fields(wm_ctx *ctx) {
  const int TX = ctx->g.nx + 2, TY = ctx->g.ny + 2;
  const size_t tps = (size_t)TX * TY;
  const int nseg = ctx->g.nsp * ctx->g.ny;
  hipLaunchKernelGGL(k_cell_fields, dim3(wm_cdiv(std::max((long long)TX * TY, (long long)nseg), 256)),
                     dim3(256), 0, ctx->stream, ctx->fg, ctx->uf, ctx->tmp, TX, TY, tps, ctx->far,
                     nseg, ctx->ts);
  WM_HIP(hipGetLastError());
  return WM_OK;
}

int wm_k_push(wm_ctx *ctx, int src, int dst) { return launch_particle<true, false>(ctx, src, dst); }
int wm_k_deposit(wm_ctx *ctx, int oldb, int newb) { return launch_particle<false, true>(ctx, oldb, newb); }
// The resident step's push, from bank 0 (read in its order, if one is
// pending) into bank 1, which becomes bank 0: the shock's injection edge
// before the current, the periodic wrap or the reconnection's walls
// (app.f90:104-105, proj/reconnection/app.f90:104; the shock has neither,
// proj/shock/app.f90:113) as it is stored.
int wm_k_push_step(wm_ctx *ctx) {
  PP P = make_pp(ctx);
  if (ctx->bcf == WM_BC_SHOCK) {
    P.inj = 1;
    P.u0 = ctx->u0;
    P.xend = wm_injection_xend(ctx, ctx->u0);
  }
  P.xmode = ctx->bcf == WM_BC_PERIODIC ? 1 : ctx->bcf == WM_BC_RECONNECTION ? 2 : 0;
  const int TX = ctx->g.nx + 2;
  const size_t tps = (size_t)TX * (size_t)(ctx->g.ny + 2);
  const Order O{ctx->perm, ctx->code, ctx->kind, ctx->farcnt, ctx->far};
  // a species' plane below 4 GB is addressed by 32-bit byte offsets
  const int src = !ctx->perm_valid                          ? SRC_SLOT
                  : (size_t)P.ny * P.cap <= ctx->plane32    ? SRC_PERM32
                                                            : SRC_PERM64;
  // Lanes of a cell: steps of 16 waste lanes on few particles, steps of 8 take
  // the longer over many, and over the dense cells of a small grid whose
  // wavefronts are all resident.  16 against 8, time ratio after 10 and 200
  // steps of a two-stream plasma, 1024 x 1024 cells: 1.47 and 1.42 at 8
  // particles per cell and species, 1.24 and 1.19 at 24, 1.08 and 1.12 at 32,
  // 0.95 and 1.05 at 40, 0.88 and 1.00 at 48; 512 x 512: 1.10 and 1.08 at 32,
  // 0.98 and 1.04 at 40, 0.86 and 0.91 at 64; 256 x 256: 1.13 and 1.01 at 24, 1.02
  // and 0.91 at 32; 256 x 192: 1.11 and 0.98, 1.06 and 0.94; 256 x 128: 1.17 and
  // 0.91, 1.05 and 0.83; 256 x 64: 1.31 and 0.89, 1.24 and 0.73; 128 x 64: 0.87 and
  // 0.63, 0.83 and 0.59.  So the line lies where a run's pinched part, the longer
  // one, begins to lose more than its first steps gain.  At 8 per cell eight lanes
  // are the faster from 16384 cells on (1.5 and 1.06).
  const long long cells = (long long)P.nx * P.ny;
  const bool eight = cells > 32768 && ctx->npart <= 36 * cells * P.nsp;
#define WM_PUSH(S, W) (eight ? k_push_step<S, W, 8> : k_push_step<S, W, 16>)
  auto kernel = P.xmode == 1 ? (src == SRC_SLOT     ? WM_PUSH(SRC_SLOT, false)
                                : src == SRC_PERM32 ? WM_PUSH(SRC_PERM32, false)
                                                    : WM_PUSH(SRC_PERM64, false))
                             : (src == SRC_SLOT     ? WM_PUSH(SRC_SLOT, true)
                                : src == SRC_PERM32 ? WM_PUSH(SRC_PERM32, true)
                                                    : WM_PUSH(SRC_PERM64, true));
#undef WM_PUSH
  P.nchunk = wm_cdiv(P.nx, PCH);
  hipLaunchKernelGGL(kernel, dim3(P.nchunk * P.ny), dim3(PCH * (eight ? 8 : 16)), 0, ctx->stream, P, ctx->cumcnt,
                     ctx->tmp, TX, tps, ctx->bank[0], ctx->bank[1], O, ctx->dep_part, ctx->derr,
                     ctx->ts);
  WM_HIP(hipGetLastError());
  std::swap(ctx->bank[0], ctx->bank[1]);
  return WM_OK;
}
