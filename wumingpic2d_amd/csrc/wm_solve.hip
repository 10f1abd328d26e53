// wm_solve.hip -- the implicit field advance (field.f90:125-184) for grids
// that fit on the chip: right-hand side, conjugate gradients and field update
// in three launches.
//
// The streaming solver (wm_field.hip) launches four kernels an iteration; at
// the few iterations a step takes (7 at the reference's 1e-6) small grids
// spend the solve in launch gaps and host checks, and larger ones read and
// write every vector from memory each time.  Here each workgroup keeps a tile
// of 128 x 4 R cells of one component on the chip for the whole solve: r,
// phi and q = A p in registers (a lane a column, R rows), p in LDS.  An
// iteration is one exchange between the component's workgroups: every
// workgroup publishes its partial sums and its edge cells of q, and waits for
// all others' sums and its four neighbours' edges.  The halo cells' r and p
// are advanced by every workgroup itself with the same arithmetic as their
// owner's, so one exchange serves both the sums and the halo.
//
// One exchange an iteration needs beta before the new residual's norm has been
// summed: beta = |r'|^2 / |r|^2 with |r'|^2 = |r|^2 - 2 alpha r.q +
// alpha^2 q.q from sums of the last sweep.  The residual's own norm (the stop
// test, alpha) is summed from the residual itself.
//
// Exchanges.  A published double is two 8-byte words, each a half of it beside
// a 32-bit tag that counts exchanges, so data and flag arrive together and
// neither fences nor barriers are needed.  Two buffers alternate: a workgroup
// publishes exchange e + 2 only after it has all sums of e + 1, which every
// other published after it had read exchange e.
//
// Every workgroup has to run at the same time as the others.  The launch has
// at most as many as the device has CUs, contexts of this process share that
// number (Slots), and whatever else occupies the CUs ends without waiting
// for this kernel.  Should they still not meet within a tenth of a second
// (another process on the same GPU, say), the kernel gives up and the host runs
// the streaming solver, from whatever df holds by then: the old change, or the
// new one where a component or a workgroup had come to its end.  The solves
// after it stream, a thousand the first time and twice as many each further
// time, so that what the waits cost stays below what the streaming does.
//
// Bound by the exchanges: about 4 us an iteration at 256 x 64 (the kernel 36 us
// for 7), of which the sweeps are 1.6; at 1024 x 1024 by the sweeps of 16 rows a
// lane, two components and then the third (161 us; the right-hand side before it
// takes 40).
#include <chrono>
#include <condition_variable>
#include <mutex>

#include "wm_internal.h"
#include "wm_debug.h"
#include "wm_solve.h"

namespace {

constexpr int NTH = 512;          // threads of a workgroup: 8 wavefronts
constexpr int TXC = 128;          // columns of a tile that has others beside it
constexpr long long PATIENCE_MS = 100;
constexpr int REST_FIRST = 1000, REST_MOST = 1 << 30;   // solves to stream after giving up

typedef unsigned long long u64;

__device__ inline void put_word(u64 *p, u64 v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline u64 get_word(const u64 *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void publish(u64 *p, double v, unsigned tag) {
  const u64 b = (u64)__double_as_longlong(v);
  put_word(p, (u64)tag << 32 | (b & 0xFFFFFFFFu));
  put_word(p + 1, (u64)tag << 32 | b >> 32);
}
struct Wait {
  int *abort_;
  long long until;
};
// N published doubles from p once all carry the tag; false when given up.
template <int N>
__device__ inline bool await(const u64 *p, unsigned tag, double *v, const Wait &W) {
  for (unsigned n = 1;; ++n) {
    u64 w[2 * N];
    bool ok = true;
#pragma unroll
    for (int k = 0; k < 2 * N; ++k) w[k] = get_word(p + k);
#pragma unroll
    for (int k = 0; k < 2 * N; ++k) ok = ok && (unsigned)(w[k] >> 32) == tag;
    if (ok) {
#pragma unroll
      for (int k = 0; k < N; ++k)
        v[k] = __longlong_as_double((long long)((w[2 * k] & 0xFFFFFFFFu) | w[2 * k + 1] << 32));
      return true;
    }
    if ((n & 63u) == 0u &&
        (__hip_atomic_load(W.abort_, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0 ||
         (long long)wall_clock64() > W.until))
      return false;
  }
}

template <int CTRL, int ROWS = 0xF>
__device__ inline double dpp_f64(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xF, ROWS == 0xF);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xF, ROWS == 0xF);
  return __longlong_as_double((long long)(unsigned)lo | ((long long)hi << 32));
}
// Fixed-order wavefront sum, in lane 63: rows of 16 lanes, then row 0 into
// row 1 and row 2 into row 3, then row 1 into row 3.
__device__ inline double wave_sum63(double v) {
  v += dpp_f64<0xB1>(v);          // quad_perm [1,0,3,2]
  v += dpp_f64<0x4E>(v);          // quad_perm [2,3,0,1]
  v += dpp_f64<0x141>(v);         // row_half_mirror
  v += dpp_f64<0x140>(v);         // row_mirror
  v += dpp_f64<0x142, 0xA>(v);    // row_bcast 15
  v += dpp_f64<0x143, 0xC>(v);    // row_bcast 31
  return v;
}
// Sums of NV values over the workgroup, in every thread (sh: two of these
// alternate, so that one barrier is enough).
template <int NV>
__device__ inline void wg_sum(double (&v)[NV], double (*sh)[NTH / 64]) {
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const double w = wave_sum63(v[k]);
    if ((threadIdx.x & 63) == 63) sh[k][threadIdx.x >> 6] = w;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    double t = sh[k][0];
#pragma unroll
    for (int q = 1; q < NTH / 64; ++q) t += sh[k][q];
    v[k] = t;
  }
}

struct SArgs {
  FieldGeom fg;
  SolveConst f;
  XSide X;
  int nbx, nby;                   // tiles of a component
  double err;
  int ite_max;
  const double *uf, *uj;
  double *df;
  double *b, *r;                  // f5 gkl and the initial residual, nx x ny planes
  u64 *sums, *edges;              // [group][2][W][8 words], [group][2][W][512][2 words]
  unsigned tag0;
  long long patience;             // of a wait, in ticks of the clock
  int *abort_;
  int abort0;                     // what it begins with
  SolveOut *out;
  unsigned long long *ts;
  bool stamp;                     // the solve begins here
};

// f5 gkl of component l at interior cell (ii, jj): field.f90:125-146.
__device__ inline double rhs(const SArgs &A, int l, int ii, int jj) {
  const size_t gx = A.fg.gx, ps = A.fg.ps;
  const size_t c = (size_t)(ii + 2) + gx * (size_t)(jj + 2);
  const double *B = A.uf + (size_t)l * ps;
  const double *E1 = A.uf + 3 * ps, *E2 = A.uf + 4 * ps, *E3 = A.uf + 5 * ps;
  const double *J1 = A.uj, *J2 = A.uj + ps, *J3 = A.uj + 2 * ps;
  const SolveConst &f = A.f;
  const double lap = B[c - gx] + B[c - 1] - 4. * B[c] + B[c + 1] + B[c + gx];
  double g;
  if (l == 0)
    g = f.f2 * (lap + f.f3 * (-J3[c - gx] + J3[c])) - f.f1 * (-E3[c - gx] + E3[c]);
  else if (l == 1)
    g = f.f2 * (lap - f.f3 * (-J3[c - 1] + J3[c])) + f.f1 * (-E3[c - 1] + E3[c]);
  else
    g = f.f2 * (lap + f.f3 * (-J2[c - 1] + J2[c] + J1[c - gx] - J1[c])) -
        f.f1 * (-E2[c - 1] + E2[c] + E1[c - gx] - E1[c]);
  return f.f5 * g;
}

// phi at column a (0-based of the active ones), row b of component l with the
// periodic halo or the wall ghosts (boundary_shock.f90:603-623).
__device__ inline double phi_at(const SArgs &A, int l, int a, int b, int wx) {
  b = wrapm(b, A.fg.ny);
  double s = 1.0;
  if (!A.X.wall) {
    a = wrapm(a, wx);
  } else if (a < 0) {
    if (l == 0) s = -1.0;
    a = l == 0 ? 0 : 1;
  } else if (a >= wx) {
    return 0.0;
  }
  return s * A.df[(size_t)l * A.fg.ps + (size_t)(A.X.xa + a + 2) + (size_t)A.fg.gx * (size_t)(b + 2)];
}

// b = f5 gkl and r = b - A phi (field.f90:350-385) of every active cell; also
// clears the mark of a solve that gave up.
__global__ __launch_bounds__(256) void k_tile_start(SArgs A) {
  const int t = blockIdx.x * 256 + threadIdx.x, l = blockIdx.y;
  const int nx = A.fg.nx, n = nx * A.fg.ny;
  if (A.stamp) wm_stamp(A.ts, 3);
  if (t == 0 && l == 0) *A.abort_ = A.abort0;
  if (t >= n) return;
  const int ii = t % nx, jj = t / nx;
  if (ii < A.X.xa || ii > A.X.xb) return;
  const int a = ii - A.X.xa, wx = A.X.xb - A.X.xa + 1;
  const double b = rhs(A, l, ii, jj);
  const double r = b + phi_at(A, l, a, jj - 1, wx) + phi_at(A, l, a - 1, jj, wx) -
                   A.f.f4 * phi_at(A, l, a, jj, wx) + phi_at(A, l, a + 1, jj, wx) +
                   phi_at(A, l, a, jj + 1, wx);
  A.b[(size_t)l * n + t] = b;
  A.r[(size_t)l * n + t] = r;
}

// A tile of 64 NWX columns and (8 / NWX) R rows, NWX wavefronts side by side.
// SOLO: the grid is one tile, no exchanges.
template <int R, int NWX, bool SOLO>
__global__ __launch_bounds__(NTH) void k_cg_tiles(SArgs A) {
  constexpr int TX = 64 * NWX, TY = 8 / NWX * R, PIT = TX + 2;
  static_assert(SOLO || (TX == TXC && TY <= 128), "a thread per halo cell");
  extern __shared__ double P[];   // (TY + 2) x PIT
  __shared__ double sh[2][4][NTH / 64];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int W = SOLO ? 1 : A.nbx * A.nby, me = SOLO ? 0 : blockIdx.x, bx = SOLO ? 0 : me % A.nbx,
            by = SOLO ? 0 : me / A.nbx;
  const int wx = A.X.xb - A.X.xa + 1, ny = A.fg.ny;
  const int x0 = bx * TX, y0 = by * TY;
  const int tw = min(TX, wx - x0), th = min(TY, ny - y0);
  const int col = wv % NWX * 64 + lane, r0 = wv / NWX * R;   // this lane's column, first row
  const bool incol = col < tw;
  double *Pc = P + (r0 + 1) * PIT + col + 1;
  u64 *sums = A.sums + (size_t)blockIdx.y * 2 * W * 8;
  u64 *edges = A.edges + (size_t)blockIdx.y * 2 * W * 1024;
  // a halo cell (south and north rows, west and east columns) that comes from
  // this tile itself: the period, or a wall
  const bool wallW = A.X.wall && bx == 0, wallE = A.X.wall && bx == A.nbx - 1;
  auto halo_at = [&](int side, int at) {
    return side == 0   ? P + at + 1
           : side == 1 ? P + (th + 1) * PIT + at + 1
           : side == 2 ? P + (at + 1) * PIT
                       : P + (at + 1) * PIT + tw + 1;
  };
  auto own_halo = [&](int side, int at, int l) {
    double *h = halo_at(side, at);
    if (side == 2 && wallW)
      *h = l == 0 ? -h[1] : h[2];
    else if (side == 3 && wallE)
      *h = 0.0;
    else
      *h = side == 0   ? P[th * PIT + at + 1]
           : side == 1 ? P[PIT + at + 1]
           : side == 2 ? P[(at + 1) * PIT + tw]
                       : P[(at + 1) * PIT + 1];
  };
  // this thread's halo cell where tiles lie side by side
  const int side = tid >> 7, at = tid & 127;
  const bool hin = !SOLO && (side < 2 ? at < tw : at < th);
  double *Ph = halo_at(side, hin ? at : 0);
  // does it come from another tile's edge (its opposite side)?
  const bool remote = hin && !(side == 2 && wallW) && !(side == 3 && wallE) &&
                      (side < 2 ? A.nby > 1 : A.nbx > 1);
  const int nb = side == 0   ? wrapm(by - 1, A.nby) * A.nbx + bx
                 : side == 1 ? wrapm(by + 1, A.nby) * A.nbx + bx
                 : side == 2 ? by * A.nbx + wrapm(bx - 1, A.nbx)
                             : by * A.nbx + wrapm(bx + 1, A.nbx);
  const u64 *hsrc = edges + ((size_t)nb * 512 + (side ^ 1) * 128 + at) * 2;
  u64 *mine = edges + (size_t)me * 1024;
  const size_t ebuf = (size_t)W * 1024, sbuf = (size_t)W * 8;
  const Wait wait{A.abort_, (long long)wall_clock64() + A.patience};
  unsigned ex = 0;                // exchanges so far
  const double f4 = A.f.f4;

  // publishes the tile's edge cells of v
  auto put_edges = [&](const double (&v)[R]) {
    if (SOLO) return;
    u64 *m = mine + (ex & 1) * ebuf;
    const unsigned tag = A.tag0 + ex;
    if (A.nby > 1 && incol) {
#pragma unroll
      for (int i = 0; i < R; ++i) {
        if (r0 + i == 0) publish(m + col * 2, v[i], tag);
        if (r0 + i == th - 1) publish(m + (128 + col) * 2, v[i], tag);
      }
    }
    if (A.nbx > 1 && (col == 0 || col == tw - 1)) {
#pragma unroll
      for (int i = 0; i < R; ++i)
        if (r0 + i < th) {
          if (col == 0) publish(m + (256 + r0 + i) * 2, v[i], tag);
          if (col == tw - 1) publish(m + (384 + r0 + i) * 2, v[i], tag);
        }
    }
  };
  // the component's totals of the workgroups' v, and this thread's halo value;
  // false (in every thread) when given up
  auto exchange = [&](double (&v)[4], bool edges_too, double &halo) {
    wg_sum<4>(v, sh[0]);
    if (!SOLO && W > 1) {
      const unsigned tag = A.tag0 + ex;
      u64 *s = sums + (ex & 1) * sbuf;
      if (tid == 0) {
#pragma unroll
        for (int k = 0; k < 4; ++k) publish(s + me * 8 + 2 * k, v[k], tag);
      }
      bool bad = false;
      if (remote && edges_too) bad = !await<1>(hsrc + (ex & 1) * ebuf, tag, &halo, wait);
      double t[4] = {0.0, 0.0, 0.0, 0.0};
      if (tid < W) bad |= !await<4>(s + tid * 8, tag, t, wait);
      if (__syncthreads_or(bad)) {
        if (tid == 0) __hip_atomic_store(A.abort_, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return false;
      }
      wg_sum<4>(t, sh[1]);
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = t[k];
    }
    ++ex;
    return true;
  };

  for (int l = blockIdx.y; l < 3; l += gridDim.y) {
    double r[R], ph[R], q[R], v[4] = {0.0, 0.0, 0.0, 0.0};
    double hr = 0.0, hp = 0.0, hq = 0.0;               // the halo cell's r, p, q
    // b.b and r.r; p = r
    const double *rl = A.r + (size_t)l * A.fg.nx * ny, *bl = A.b + (size_t)l * A.fg.nx * ny;
    const int o = A.X.xa + x0 + col + A.fg.nx * (y0 + r0);
#pragma unroll
    for (int i = 0; i < R; ++i) {
      r[i] = ph[i] = q[i] = 0.0;
      if (incol && r0 + i < th) {
        r[i] = rl[o + A.fg.nx * i];
        q[i] = bl[o + A.fg.nx * i];
        ph[i] = A.df[(size_t)l * A.fg.ps + (size_t)(A.X.xa + x0 + col + 2) +
                     (size_t)A.fg.gx * (size_t)(y0 + r0 + i + 2)];
      }
    }
    if (remote) {
      const int a = wrapm(side < 2 ? x0 + at : (side == 2 ? x0 - 1 : x0 + tw), wx);
      const int b = wrapm(side >= 2 ? y0 + at : (side == 0 ? y0 - 1 : y0 + th), ny);
      hr = rl[A.X.xa + a + A.fg.nx * b];
    }
#pragma unroll
    for (int i = 0; i < R; ++i) {
      v[0] = fma(q[i], q[i], v[0]);
      v[1] = fma(r[i], r[i], v[1]);
      if (incol && r0 + i < th) Pc[i * PIT] = r[i];
    }
    if (!exchange(v, false, hq)) return;
    hp = hr;
    double sum_g = v[0], eps = sqrt(v[0]) * A.err, sumr = v[1];
    int ite = 0, err = 0;
    if (sqrt(sumr) > eps && sum_g > eps) {
      for (;;) {
        // p is in LDS: its halo, then q = A p and the sums of r.r, p.q, r.q, q.q
        if (remote) *Ph = hp;
        __syncthreads();
        if (SOLO) {
          for (int h = tid; h < 2 * (tw + th); h += NTH) {
            const int hx = h - 2 * tw;
            if (hx < 0) own_halo(h >= tw, h >= tw ? h - tw : h, l);
            else own_halo(hx >= th ? 3 : 2, hx >= th ? hx - th : hx, l);
          }
        } else if (hin && !remote) {
          own_halo(side, at, l);
        }
        __syncthreads();
        v[0] = v[1] = v[2] = v[3] = 0.0;
        if (incol) {
          double s = Pc[-PIT], c = Pc[0];
#pragma unroll
          for (int i = 0; i < R; ++i) {
            const double n = Pc[(i + 1) * PIT];
            if (r0 + i < th) {
              // field.f90:400-402
              double ap = -s - Pc[i * PIT - 1];
              ap = fma(f4, c, ap) - Pc[i * PIT + 1] - n;
              q[i] = ap;
              v[0] = fma(r[i], r[i], v[0]);
              v[1] = fma(c, ap, v[1]);
              v[2] = fma(r[i], ap, v[2]);
              v[3] = fma(ap, ap, v[3]);
            }
            s = c;
            c = n;
          }
        }
        put_edges(q);
        if (!exchange(v, true, hq)) return;
        // field.f90:387-450
        sumr = v[0];
        ++ite;
        const double av = sumr / v[1];
        sum_g = sqrt(sumr);
        if (ite >= A.ite_max) err = 1;
        const bool stop = !(sum_g > eps) || err;
        const double bv = fmax(fma(av, fma(av, v[3], -2.0 * v[2]), sumr), 0.0) / sumr;
#pragma unroll
        for (int i = 0; i < R; ++i)
          if (incol && r0 + i < th) {
            const double p = Pc[i * PIT];
            ph[i] = fma(av, p, ph[i]);
            r[i] = fma(-av, q[i], r[i]);
            Pc[i * PIT] = fma(bv, p, r[i]);
          }
        hr = fma(-av, hq, hr);
        hp = fma(bv, hp, hr);
        if (stop) break;
      }
#pragma unroll
      for (int i = 0; i < R; ++i)
        if (incol && r0 + i < th)
          A.df[(size_t)l * A.fg.ps + (size_t)(A.X.xa + x0 + col + 2) +
               (size_t)A.fg.gx * (size_t)(y0 + r0 + i + 2)] = ph[i];
    }
    if (me == 0 && tid == 0) {
      A.out->ite[l] = ite;
      A.out->err[l] = err;
      atomicMax(A.ts + 4, (unsigned long long)wall_clock64());
    }
    __syncthreads();                                   // P is filled again
  }
}

// The field update for the periodic box, one cell of the ghost-inclusive
// planes per thread (field.f90:150-184): delta B of the cell's periodic image
// is the solution, delta E follows from it (:154-171); the sums go to the
// other set of planes, so no cell waits for its neighbours' old values.  Bound
// by memory: 18 planes moved in one launch, where filling the ghosts, delta E,
// the ghosts again and the sum moved 30 in six.  Skipped when the solve gave up
// or failed (abort_ null: it streamed, and has been checked).  Also hands the
// solve's and the step's status to the host.
__global__ __launch_bounds__(256) void k_field_update(FieldGeom fg, SolveConst f,
                                                      const double *__restrict__ uf,
                                                      const double *__restrict__ uj,
                                                      const double *__restrict__ df,
                                                      double *__restrict__ un, const int *abort_,
                                                      const SolveOut *out, const int *derr,
                                                      const unsigned long long *ts, unsigned seq,
                                                      SolveReport *host) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  const int given = abort_ ? *abort_ : 0;
  const SolveOut o = abort_ ? *out : SolveOut{};
  if (t == 0) leave_report(host, o, given, derr, ts, wall_clock64(), seq);
  if (given || o.err[0] || o.err[1] || o.err[2] || t >= fg.gx * fg.gy) return;
  const int li = t % fg.gx, lj = t / fg.gx;
  const int ci = wrapm(li - 2, fg.nx);
  int cj = lj - 2;
  if (cj < 0 || cj >= fg.ny) {
    cj %= fg.ny;
    if (cj < 0) cj += fg.ny;
  }
  const size_t gx = fg.gx, ps = fg.ps, c = (size_t)(ci + 2) + gx * (size_t)(cj + 2);
  const size_t ce = (size_t)(wrapm(ci + 1, fg.nx) + 2) + gx * (size_t)(cj + 2);
  const size_t cn = (size_t)(ci + 2) + gx * (size_t)(wrapm(cj + 1, fg.ny) + 2);
  const double *dB1 = df, *dB2 = df + ps, *dB3 = df + 2 * ps;
  const double *B1 = uf, *B2 = uf + ps, *B3 = uf + 2 * ps;
  const double b1 = dB1[c], b2 = dB2[c], b3 = dB3[c];
  const double e1 = f.f1 * (f.gfac * (-b3 + dB3[cn]) + (-B3[c] + B3[c + gx])) - f.fpt * uj[c];
  const double e2 = -f.f1 * (f.gfac * (-b3 + dB3[ce]) + (-B3[c] + B3[c + 1])) - f.fpt * uj[ps + c];
  const double e3 = f.f1 * (f.gfac * (-b2 + dB2[ce] + b1 - dB1[cn]) +
                            (-B2[c] + B2[c + 1] + B1[c] - B1[c + gx])) -
                    f.fpt * uj[2 * ps + c];
  un[t] = uf[t] + b1;
  un[ps + t] = uf[ps + t] + b2;
  un[2 * ps + t] = uf[2 * ps + t] + b3;
  un[3 * ps + t] = uf[3 * ps + t] + e1;
  un[4 * ps + t] = uf[4 * ps + t] + e2;
  un[5 * ps + t] = uf[5 * ps + t] + e3;
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) leave_end(host, seq);
}

// The same between conducting walls (active columns L .. E of the
// ghost-inclusive planes, boundary_shock.f90:326-405,
// boundary_reconnection.f90:280-359): rows wrap, then Bx, Ey, Ez are odd about
// the left wall and By, Bz, Ex even; right of the shock's box is zero, the
// reconnection's right wall is the mirror image and rewrites column E of Bx,
// Ey and Ez.  delta E at a cell that takes another's is worked out there.  What
// no rule writes (two columns out, and E + 1 of the reconnection's odd
// components) is added as it stands, and df is left as the separate kernels
// leave it: the walls may move.  Columns outside L - 2 .. E + 2 are copied.
// One launch for seven, 32 us of a step at 256 x 128.
struct WallField {
  const double *df;
  size_t ps;
  int L, E;
  bool shock;
  // delta B of component k at column li (L - 1 .. E + 1) of the interior row
  // that begins at ro
  __device__ double dB(int k, int li, size_t ro) const {
    const double *R = df + (size_t)k * ps + ro;
    if (li == L - 1) return k == 0 ? -R[L] : R[L + 1];
    if (li == E && k == 0 && !shock) return -R[E - 1];
    if (li == E + 1) return shock ? 0.0 : (k == 0 ? R[li] : R[E - 1]);
    return R[li];
  }
};
__global__ __launch_bounds__(256) void k_walls_update(FieldGeom fg, SolveConst f, XSide X,
                                                      const double *__restrict__ uf,
                                                      const double *__restrict__ uj, double *df,
                                                      double *__restrict__ un, const int *abort_,
                                                      const SolveOut *out, const int *derr,
                                                      const unsigned long long *ts, unsigned seq,
                                                      SolveReport *host) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  const int given = abort_ ? *abort_ : 0;
  const SolveOut o = abort_ ? *out : SolveOut{};
  if (t == 0) leave_report(host, o, given, derr, ts, wall_clock64(), seq);
  if (given || o.err[0] || o.err[1] || o.err[2] || t >= fg.gx * fg.gy) return;
  const int li = t % fg.gx, lj = t / fg.gx;
  const size_t gx = fg.gx, ps = fg.ps;
  const WallField W{df, ps, X.xa + 2, X.xb + 2, X.wall == WM_BC_SHOCK};
  double d[6];
  if (li < W.L - 1 || li > W.E + 1) {
    const bool add = li == W.L - 2 || li == W.E + 2;
#pragma unroll
    for (int k = 0; k < 6; ++k) d[k] = add ? df[k * ps + t] : 0.0;
  } else {
    int j = (lj - 2) % fg.ny;
    if (j < 0) j += fg.ny;
    const size_t ro = gx * (size_t)(j + 2), rn = gx * (size_t)(wrapm(j + 1, fg.ny) + 2);
    const double *B1 = uf, *B2 = uf + ps, *B3 = uf + 2 * ps;
    auto dE = [&](int k, int col) {            // field.f90:154-171
      const size_t c = (size_t)col + ro;
      if (k == 3)
        return f.f1 * (f.gfac * (-W.dB(2, col, ro) + W.dB(2, col, rn)) + (-B3[c] + B3[c + gx])) -
               f.fpt * uj[c];
      if (k == 4)
        return -f.f1 * (f.gfac * (-W.dB(2, col, ro) + W.dB(2, col + 1, ro)) + (-B3[c] + B3[c + 1])) -
               f.fpt * uj[ps + c];
      return f.f1 * (f.gfac * (-W.dB(1, col, ro) + W.dB(1, col + 1, ro) + W.dB(0, col, ro) -
                               W.dB(0, col, rn)) +
                     (-B2[c] + B2[c + 1] + B1[c] - B1[c + gx])) -
             f.fpt * uj[2 * ps + c];
    };
    const bool left = li == W.L - 1, right = li == W.E + 1, stale = right && !W.shock;
#pragma unroll
    for (int k = 0; k < 3; ++k) d[k] = stale && k == 0 ? df[t] : W.dB(k, li, ro);
    if (right && W.shock) {
      d[3] = d[4] = d[5] = 0.0;
    } else {
      d[3] = dE(3, left ? W.L + 1 : (right ? W.E - 1 : li));
      const bool odd = left || (li == W.E && !W.shock);
      const int col = left ? W.L : (odd ? W.E - 1 : li);
#pragma unroll
      for (int k = 4; k < 6; ++k) {
        if (stale) {
          d[k] = df[k * ps + t];
        } else {
          const double v = dE(k, col);
          d[k] = odd ? -v : v;
        }
      }
    }
#pragma unroll
    for (int k = 0; k < 6; ++k)                // (delta B inside the box is there)
      if (k >= 3 || left || right || li == W.E || lj < 2 || lj >= fg.ny + 2)
        if (!(stale && (k == 0 || k > 3))) df[k * ps + t] = d[k];
  }
#pragma unroll
  for (int k = 0; k < 6; ++k) un[k * ps + t] = uf[k * ps + t] + d[k];
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) leave_end(host, seq);
}

// The device's CUs shared by the contexts of this process: a solve in flight
// holds as many as it has workgroups.
struct Slots {
  std::mutex m;
  std::condition_variable cv;
  int used = 0;
};
constexpr int MAX_DEV = 64;
Slots slots[MAX_DEV];

struct Plan {
  int R = 0, nwx = 2, nbx = 1, nby = 1, groups = 3;   // R 0: does not fit
  bool solo = false;
  int workgroups() const { return nbx * nby * groups; }
};

// The tile, and how many of the three components run side by side: the least
// estimate of an iteration's time in microseconds, from the time of both kernels
// at 7 iterations, launches and all, measured for every plan: a row of cells 0.4 (alone on its CU
// 0.2), an exchange 3 and 0.08 a workgroup that takes part, a component that
// waits for another's end a whole iteration more.  Both kernels, us, at 4, 8 and
// 16 rows a lane: 256 x 64: 44, 52, 69; 512 x 128: 49, 55, 76; 499 x 309: 84,
// 69, 85; 1024 x 256: 158 (two turns), 79, 92.  One workgroup a component
// against several: 250 x 24: 35 and 42; 128 x 64: 35 and 40; 500 x 16: 39 and
// 42.  Streaming: 116 to 145 up to 512 x 128, 184 at 499 x 309 (69 here), 350 at
// 1024 x 512 (116), 625 at 1024 x 1024 (235).
Plan make_plan(int wx, int ny, int ncu) {
  Plan best;
  double least = 1e300;
  auto consider = [&](const Plan &p, double us) {
    if (us < least) {
      least = us;
      best = p;
    }
  };
  for (int R = 4; R <= 16; R *= 2) {
    Plan p;
    p.R = R;
    for (p.nwx = 2; p.nwx <= 8; p.nwx *= 2)
      if (wx <= 64 * p.nwx && ny <= 8 / p.nwx * R) {
        p.solo = true;
        consider(p, 0.5 + 0.2 * R);
      }
    p.solo = false;
    p.nwx = 2;
    p.nbx = wm_cdiv(wx, TXC);
    p.nby = wm_cdiv(ny, 4 * R);
    const long long W = (long long)p.nbx * p.nby;
    if (W > ncu || W > NTH) continue;
    p.groups = 3 * W <= ncu ? 3 : (2 * W <= ncu ? 2 : 1);
    consider(p, (4 - p.groups) * (3.0 + 0.4 * R + 0.08 * (double)W));
  }
  return best;
}

template <int R, int NWX, bool SOLO>
void launch_tiles(const Plan &p, const SArgs &A, hipStream_t st) {
  constexpr size_t lds = sizeof(double) * (8 / NWX * R + 2) * (64 * NWX + 2);
  static_assert(lds + 1024 <= 163840, "a tile fits a CU's LDS");
  if (lds > 65536)
    (void)hipFuncSetAttribute((const void *)k_cg_tiles<R, NWX, SOLO>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  hipLaunchKernelGGL((k_cg_tiles<R, NWX, SOLO>), dim3(p.nbx * p.nby, p.groups), dim3(NTH), lds, st, A);
}
template <int R>
void launch_tiles(const Plan &p, const SArgs &A, hipStream_t st) {
  if (!p.solo) launch_tiles<R, 2, false>(p, A, st);
  else if (p.nwx == 2) launch_tiles<R, 2, true>(p, A, st);
  else if (p.nwx == 4) launch_tiles<R, 4, true>(p, A, st);
  else launch_tiles<R, 8, true>(p, A, st);
}

}  // namespace

namespace {
// One thread: the step's status for the host, where no update kernel leaves it.
__global__ void k_report(const int *abort_, const SolveOut *out, const int *derr,
                         const unsigned long long *ts, unsigned seq, SolveReport *host) {
  leave_end(host, seq);
  leave_report(host, abort_ ? *out : SolveOut{}, abort_ ? *abort_ : 0, derr, ts, ts[8], seq);
}

SolveReport *report_of(wm_ctx *ctx) { return (SolveReport *)((char *)ctx->h_pin + WM_PIN_REPORT); }

// How long a solve waits for others of this process to end before it streams.
constexpr auto SLOT_WAIT = std::chrono::seconds(1);

Plan plan_of(const wm_ctx *ctx) {
  const XSide X = wm_xside(ctx);
  return make_plan(X.xb - X.xa + 1, ctx->g.ny, ctx->ncu);
}

void release(wm_ctx *ctx) {
  if (!ctx->tile_held) return;
  Slots &s = slots[ctx->device];
  {
    std::lock_guard<std::mutex> lk(s.m);
    s.used -= ctx->tile_held;
  }
  ctx->tile_held = 0;
  s.cv.notify_all();
}
}  // namespace

// Plain CG on a grid whose tiles run side by side; the recording of
// preconditioner pairs needs the iterates, so it streams.
bool wm_tiles_fit(wm_ctx *ctx, bool peek) {
  if (ctx->solver == WM_SOLVER_CG && ctx->bcf == WM_BC_PERIODIC && wm_pc_collecting(ctx))
    return false;
  if (ctx->device < 0 || ctx->device >= MAX_DEV) return false;
  if (!ctx->ncu) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, ctx->device) != hipSuccess)
      return false;
    ctx->ncu = n;
  }
  if (ctx->tile_rest > 0) {
    if (!peek) --ctx->tile_rest;
    return false;
  }
  return plan_of(ctx).R > 0;
}

// *ran: false where other contexts' solves hold too much of the device for too
// long (nothing is launched then).
int wm_k_tiles(wm_ctx *ctx, bool begins, bool *ran) {
  const Plan p = plan_of(ctx);
  const size_t n = (size_t)p.workgroups();
  *ran = false;
  if (n > ctx->tile_cap) {
    if (ctx->tile_sums) (void)hipFree(ctx->tile_sums);
    if (ctx->tile_edges) (void)hipFree(ctx->tile_edges);
    ctx->tile_sums = ctx->tile_edges = nullptr;
    ctx->tile_cap = 0;
    WM_HIP(hipMalloc((void **)&ctx->tile_sums, sizeof(u64) * n * 2 * 8));
    WM_HIP(hipMalloc((void **)&ctx->tile_edges, sizeof(u64) * n * 2 * 1024));
    WM_HIP(hipMemsetAsync(ctx->tile_sums, 0, sizeof(u64) * n * 2 * 8, ctx->stream));
    WM_HIP(hipMemsetAsync(ctx->tile_edges, 0, sizeof(u64) * n * 2 * 1024, ctx->stream));
    ctx->tile_cap = n;
  }
  if (!ctx->tile_abort) {
    WM_HIP(hipMalloc((void **)&ctx->tile_abort, sizeof(int)));
    WM_HIP(hipMalloc(&ctx->tile_out, sizeof(SolveOut)));
    WM_HIP(hipMemsetAsync(ctx->tile_out, 0, sizeof(SolveOut), ctx->stream));
  }
  SArgs A;
  A.fg = ctx->fg;
  A.f = make_fc(ctx->g);
  A.X = wm_xside(ctx);
  A.nbx = p.nbx;
  A.nby = p.nby;
  A.err = ctx->cg_err;
  A.ite_max = ctx->ite_max;
  A.uf = ctx->uf;
  A.uj = ctx->uj;
  A.df = ctx->df;
  A.b = ctx->gkl;
  A.r = ctx->cg_r;
  A.sums = ctx->tile_sums;
  A.edges = ctx->tile_edges;
  const unsigned need = 3u * (unsigned)(ctx->ite_max + 4);
  if (ctx->tile_tag > 0xFFFFFFFFu - need) {
    // the tags begin again: words that still carry one of them must not pass
    // for this solve's
    WM_HIP(hipMemsetAsync(ctx->tile_sums, 0, sizeof(u64) * ctx->tile_cap * 2 * 8, ctx->stream));
    WM_HIP(hipMemsetAsync(ctx->tile_edges, 0, sizeof(u64) * ctx->tile_cap * 2 * 1024, ctx->stream));
    ctx->tile_tag = 1;
  }
  A.tag0 = ctx->tile_tag;
  ctx->tile_tag += need;
  const bool forced = ctx->solve_gives_up > 0;
  if (forced) --ctx->solve_gives_up;
  A.patience = forced ? 0 : PATIENCE_MS * ctx->clock_khz;
  A.abort_ = ctx->tile_abort;
  A.abort0 = forced;
  A.out = (SolveOut *)ctx->tile_out;
  A.ts = ctx->ts;
  A.stamp = begins;
  {
    Slots &s = slots[ctx->device];
    std::unique_lock<std::mutex> lk(s.m);
    if (!s.cv.wait_for(lk, SLOT_WAIT, [&] { return s.used + (int)n <= ctx->ncu; })) return WM_OK;
    s.used += (int)n;
    ctx->tile_held = (int)n;
  }
  if (ctx->solve_fails > 0) {
    --ctx->solve_fails;
    wm_set_error(ctx, WM_ERR_HIP, "the field solve's launch failed");
    return WM_ERR_HIP;
  }
  hipLaunchKernelGGL(k_tile_start, dim3(wm_cdiv((long long)ctx->g.nx * ctx->g.ny, 256), 3),
                     dim3(256), 0, ctx->stream, A);
  switch (p.R) {
    case 4: launch_tiles<4>(p, A, ctx->stream); break;
    case 8: launch_tiles<8>(p, A, ctx->stream); break;
    default: launch_tiles<16>(p, A, ctx->stream); break;
  }
  WM_HIP(hipGetLastError());
  *ran = true;
  return WM_OK;
}

// A single row is its own neighbour above and below: its ghost rows hold what
// the reference's sequence of copies leaves there, which takes the separate
// kernels.
bool wm_fused_update(const wm_ctx *ctx) { return ctx->g.ny > 1; }

int wm_k_update_report(wm_ctx *ctx) {
  const FieldGeom &fg = ctx->fg;
  const int *abort_ = ctx->tile_held ? ctx->tile_abort : nullptr;
  ++ctx->seq;
  if (wm_fused_update(ctx)) {
    if (!ctx->uf2) WM_HIP(hipMalloc((void **)&ctx->uf2, sizeof(double) * 6 * fg.ps));
    const dim3 grid(wm_cdiv((long long)fg.gx * fg.gy, 256));
    const XSide X = wm_xside(ctx);
    if (X.wall)
      hipLaunchKernelGGL(k_walls_update, grid, dim3(256), 0, ctx->stream, fg, make_fc(ctx->g), X,
                         ctx->uf, ctx->uj, ctx->df, ctx->uf2, abort_,
                         (const SolveOut *)ctx->tile_out, ctx->derr, ctx->ts, ctx->seq,
                         report_of(ctx));
    else
      hipLaunchKernelGGL(k_field_update, grid, dim3(256), 0, ctx->stream, fg, make_fc(ctx->g),
                         ctx->uf, ctx->uj, ctx->df, ctx->uf2, abort_,
                         (const SolveOut *)ctx->tile_out, ctx->derr, ctx->ts, ctx->seq,
                         report_of(ctx));
    std::swap(ctx->uf, ctx->uf2);
    ctx->tile_swapped = ctx->tile_held != 0;
  } else {
    hipLaunchKernelGGL(k_report, dim3(1), dim3(1), 0, ctx->stream, abort_,
                       (const SolveOut *)ctx->tile_out, ctx->derr, ctx->ts, ctx->seq, report_of(ctx));
  }
  WM_HIP(hipGetLastError());
  return WM_OK;
}

// Waits for the last report asked for.  For a while by looking at it: a small
// grid's step is over in a tenth of a millisecond, of which waiting for the
// stream would take a tenth again.
int wm_report_wait(wm_ctx *ctx) {
  const SolveReport *r = report_of(ctx);
  const auto there = [&] { return __atomic_load_n(&r->seq, __ATOMIC_ACQUIRE) == ctx->seq; };
  const auto t0 = std::chrono::steady_clock::now();
  while (!there()) {
    for (int k = 0; k < 64 && !there(); ++k) __builtin_ia32_pause();
    if (std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(1)) break;
  }
  if (there()) return WM_OK;
  WM_HIP(hipStreamSynchronize(ctx->stream));
  if (there()) return WM_OK;
  wm_set_error(ctx, WM_ERR_HIP, "the step's report did not arrive");
  return WM_ERR_HIP;
}

// The clock as the update of report seq ended (this or the last report's).
unsigned long long wm_update_end(const wm_ctx *ctx, unsigned seq) {
  const SolveReport *r = (const SolveReport *)((const char *)ctx->h_pin + WM_PIN_REPORT);
  return __atomic_load_n(&r->end[seq & 1], __ATOMIC_ACQUIRE);
}

// After the report has been waited for.
int wm_tiles_result(wm_ctx *ctx, bool *gave_up, int *err, int *ite) {
  release(ctx);
  const SolveReport r = *report_of(ctx);
  *gave_up = r.abort_ != 0;
  *err = r.out.err[0] | r.out.err[1] | r.out.err[2];
  for (int l = 0; l < 3; ++l) ite[l] = r.out.ite[l];
  if ((*gave_up || *err) && ctx->tile_swapped) std::swap(ctx->uf, ctx->uf2);
  ctx->tile_swapped = false;
  if (*gave_up) {
    ctx->tile_rest = std::max(REST_FIRST, ctx->tile_rest_next);
    ctx->tile_rest_next = std::min(2 * (long long)ctx->tile_rest, (long long)REST_MOST);
  }
  return WM_OK;
}

void wm_field_release(wm_ctx *ctx) {
  if (!ctx->tile_held) return;
  (void)hipStreamSynchronize(ctx->stream);
  if (ctx->tile_swapped) {
    const SolveReport r = *report_of(ctx);
    if (r.abort_ || r.out.err[0] || r.out.err[1] || r.out.err[2]) std::swap(ctx->uf, ctx->uf2);
    ctx->tile_swapped = false;
  }
  release(ctx);
}

long long wm_debug_slots(wm_ctx *ctx, int add) {
  if (ctx->device < 0 || ctx->device >= MAX_DEV) return -1;
  Slots &s = slots[ctx->device];
  long long used;
  {
    std::lock_guard<std::mutex> lk(s.m);
    used = s.used += add;
  }
  if (add < 0) s.cv.notify_all();
  return used;
}
