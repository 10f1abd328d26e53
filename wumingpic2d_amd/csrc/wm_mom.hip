// wm_mom.hip -- the moment diagnostics of an output step on the device:
// mom_calc__accl's velocity update over half a step (mom_calc.f90:48-164),
// mom_calc__nvt's cloud-in-cell moments N, V, T (:167-249), fused per tile of
// cells, and boundary_periodic__mom's periodic fold
// (boundary_periodic.f90:571-636).
//
// One workgroup takes MC cells x MR rows of one species.  Sixteen lanes share a
// cell and take its particles in rounds of sixteen, one per lane: each lane
// stages its particle's weights at the 3 x 3 nodes around the cell (x - 1/2
// truncates to the cell or the one before it) and its moment values in LDS,
// and the cell's sums, moments x particles x nodes, are matrix products (4 x 4
// x 4, a block for each of the wavefront's four cells), particles in order.  A
// lane keeps three node rows' sums; when the cells of a row are done the lowest
// is complete for its column of cells.  At the end the columns go into the
// tile in ascending order.  The tiles overlap by two node columns and two node
// rows; a gather adds the (at most four) tiles of a node in a fixed order.
// Every sum has one order: the result does not depend on scheduling.
#include "wm_internal.h"

namespace {

constexpr int MC = 16;           // cells per workgroup along x
constexpr int MR = 4;            // rows per workgroup
constexpr int MG = 16;           // lanes per cell
constexpr int MW = MC + 2;       // tile columns: cells / nodes i0-1 .. i0+MC
constexpr int MH = MR + 2;       // tile rows: j0-1 .. j0+MR
constexpr int NMOM = 7;          // N, Vx, Vy, Vz, Txx, Tyy, Tzz
constexpr int NV = NMOM - 1;     // moment values staged (N's is 1)
constexpr int NST = NV + 9;      // staged per particle: 6 moment values, 9 weights
constexpr int CST = 8 * NST + 2;   // a cell's slots (padded against bank conflicts)
constexpr int CSZ = MH * 3 * NMOM;
constexpr int TSZ = NMOM * MH * MW;

struct MP {
  int nx, ny, nxgs, nys, nsp, nchunk, nrb, cap;
  double d_delx, c, delt;        // delt: the moment step, half the run's (mom_calc.f90:34)
  double q[WM_MAXSP], r[WM_MAXSP];
};

struct Pt {
  double x, y, ux, uy, uz;
};

// FP64 form: the records of cell i (local index) of a row, in cumcnt order.
struct Src64 {
  const double *x, *y, *ux, *uy, *uz;
  const int *cumcnt;
  __device__ void range(const MP &P, int s, int jl, int i, size_t &base, int &kb, int &ke) const {
    const size_t seg = (size_t)s * P.ny + jl;
    const int *cc = cumcnt + seg * (size_t)(P.nx + 1);
    kb = max(0, cc[i]);
    ke = min(P.cap, cc[i + 1]);
    base = seg * (size_t)P.cap;
  }
  static constexpr bool INDEXED = false;
  __device__ Pt load(size_t p, int, int) const { return Pt{x[p], y[p], ux[p], uy[p], uz[p]}; }
};

// The same between steps of the resident run, while the rows' order is an index
// into the species' planes (wm_order.hip).  Putting the rows in order first, as
// every other reader of whole rows does, moves 120 bytes a particle: a call after
// a step 1.93 ms at 512 x 512 with 64 per cell and species, 2.78 with that and 1.91
// where the rows lie in order (the index costs the kernel 0.64 to 0.62 ms).
struct Order64 {
  Src64 s;
  const unsigned *perm;
  size_t plane;                  // slots of a species' plane
  size_t seg0 = 0;               // the plane of the species at hand
  static constexpr bool INDEXED = true;
  __device__ void range(const MP &P, int sp, int jl, int i, size_t &base, int &kb, int &ke) {
    seg0 = sp * plane;
    s.range(P, sp, jl, i, base, kb, ke);
  }
  __device__ unsigned at(size_t p) const { return perm[p]; }
  __device__ Pt load(unsigned q, int i, int j) const { return s.load(seg0 + q, i, j); }
};

// FP32 form: the cell's bin.  The position is the cell's index plus the
// offset, in FP64, as the layout conversion to the reference arrays forms it.
struct Src32 {
  const float4 *q;
  const float *uz;
  const int *cnt;
  const int *bstart;
  __device__ void range(const MP &P, int s, int jl, int i, size_t &base, int &kb, int &ke) const {
    const size_t seg = (size_t)s * P.ny + jl;
    kb = 0;
    ke = cnt[seg * P.nx + i];
    base = seg * (size_t)P.cap + bstart[seg * (P.nx + 1) + i];
  }
  static constexpr bool INDEXED = false;
  __device__ Pt load(size_t p, int iabs, int jabs) const {
    const float4 v = q[p];
    return Pt{(double)iabs + (double)v.x, (double)jabs + (double)v.y, (double)v.z, (double)v.w,
              (double)uz[p]};
  }
};

__device__ inline void tsc(double dh, double &sm, double &s0, double &sp) {
  // mom_calc.f90:97-105
  sm = 0.5 * (0.5 - dh) * (0.5 - dh);
  s0 = 0.75 - dh * dh;
  sp = 0.5 * (0.5 + dh) * (0.5 + dh);
}

// mom_calc.f90:107-155: the Boris update of u over the moment step in the
// fields f; the position is not advanced.
__device__ inline void half_push(const double (&f)[6], const Pt &v, const MP &P, double fac1,
                                 double txxx, double fac2, double &ux, double &uy, double &uz) {
  const double bpx = f[0], bpy = f[1], bpz = f[2], epx = f[3], epy = f[4], epz = f[5];
  double uvm1 = v.ux + fac1 * epx;
  double uvm2 = v.uy + fac1 * epy;
  double uvm3 = v.uz + fac1 * epz;
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
  ux = uvm1 + fac1 * epx;
  uy = uvm2 + fac1 * epy;
  uz = uvm3 + fac1 * epz;
}

// The cell-centred fields, mom_calc.f90:68-81, of H rows of W cells from cell
// (a0, b0) (local indices): [field][row][column]; cell (a, b) is at (a+2, b+2)
// of a ghost-inclusive plane.
template <int W, int H>
__device__ inline void cell_fields(double *F, const MP &P, const FieldGeom &fg,
                                   const double *__restrict__ uf, int a0, int b0) {
  for (int t = threadIdx.x; t < 6 * H * W; t += blockDim.x) {
    const int col = t % W, row = (t / W) % H, k = t / (W * H);
    const int a = a0 + col, b = b0 + row;
    double v = 0.0;
    if (a <= P.nx && b <= P.ny) {
      const size_t gx = fg.gx, o = (size_t)(a + 2) + gx * (size_t)(b + 2);
      const double *U = uf + (size_t)k * fg.ps;
      switch (k) {
        case 0: v = 0.5 * (U[o] + U[o + gx]); break;
        case 1: v = 0.5 * (U[o] + U[o + 1]); break;
        case 2: v = 0.25 * (U[o] + U[o + 1] + U[o + gx] + U[o + gx + 1]); break;
        case 3: v = 0.5 * (U[o] + U[o + 1]); break;
        case 4: v = 0.5 * (U[o] + U[o + gx]); break;
        default: v = U[o]; break;
      }
    }
    F[t] = v;
  }
}

// mom_calc__accl on its own: workgroup (row, chunk, species), eight lanes a
// cell; the updated records go to the gp bank.
constexpr int AC = 32;           // cells of a workgroup
constexpr int AG = 8;            // lanes of a cell
constexpr int AW = AC + 2;
__global__ __launch_bounds__(AC * AG, 3) void k_accl(MP P, FieldGeom fg, const double *__restrict__ uf,
                                                  Src64 src, Rec64 gp) {
  __shared__ double F[6 * 3 * AW];
  const int jl = blockIdx.x, c0 = blockIdx.y * AC, s = blockIdx.z;
  cell_fields<AW, 3>(F, P, fg, uf, c0 - 1, jl - 1);
  __syncthreads();
  const int g = threadIdx.x / AG, i = c0 + g;
  if (i >= P.nx) return;
  const double q = P.q[s], rr = P.r[s];
  const double fac1 = q / rr * 0.5 * P.delt;     // mom_calc.f90:90-92
  const double txxx = fac1 * fac1;
  const double fac2 = q * P.delt / rr;
  const int iabs = P.nxgs + i, jabs = P.nys + jl;
  size_t base;
  int kb, ke;
  src.range(P, s, jl, i, base, kb, ke);
  for (int k = kb + threadIdx.x % AG; k < ke; k += AG) {
    const size_t p = base + (size_t)k;
    const Pt v = src.load(p, iabs, jabs);
    __asm__ volatile("" ::: "memory");           // the 54 values stay in LDS
    double sx0, sx1, sx2, sy0, sy1, sy2, f[6];
    tsc(v.x * P.d_delx - 0.5 - iabs, sx0, sx1, sx2);
    tsc(v.y * P.d_delx - 0.5 - jabs, sy0, sy1, sy2);
#pragma unroll
    for (int e = 0; e < 6; ++e) {
      const double *T = F + e * 3 * AW + g;
      f[e] = (T[0] * sx0 + T[1] * sx1 + T[2] * sx2) * sy0 +
             (T[AW] * sx0 + T[AW + 1] * sx1 + T[AW + 2] * sx2) * sy1 +
             (T[2 * AW] * sx0 + T[2 * AW + 1] * sx1 + T[2 * AW + 2] * sx2) * sy2;
    }
    double ux, uy, uz;
    half_push(f, v, P, fac1, txxx, fac2, ux, uy, uz);
    gp.x[p] = v.x;
    gp.y[p] = v.y;
    gp.ux[p] = ux;
    gp.uy[p] = uy;
    gp.uz[p] = uz;
  }
}

// The fields at a particle: sum over ij of C_ij ox^i oy^j, field k's nine
// coefficients in lane k of the particle's 16 lanes.  The row broadcast is the
// multiply-add's own operand modifier; all 64 lanes are active (the wait
// covers the modifier after a write of C).
__device__ inline void gather(double (&f)[6], const double (&C)[9], const double (&w)[9]) {
#define WM_B(N) " row_newbcast:" #N " row_mask:0xf bank_mask:0xf\n\t"
#define WM_6(C, W)                                                                          \
  "v_fmac_f64_dpp %0, %" #C ", %" #W WM_B(0) "v_fmac_f64_dpp %1, %" #C ", %" #W WM_B(1)     \
  "v_fmac_f64_dpp %2, %" #C ", %" #W WM_B(2) "v_fmac_f64_dpp %3, %" #C ", %" #W WM_B(3)     \
  "v_fmac_f64_dpp %4, %" #C ", %" #W WM_B(4) "v_fmac_f64_dpp %5, %" #C ", %" #W WM_B(5)
#pragma unroll
  for (int k = 0; k < 6; ++k) f[k] = 0.0;
  __asm__("s_nop 4\n\t" WM_6(6, 15) WM_6(7, 16) WM_6(8, 17) WM_6(9, 18) WM_6(10, 19) WM_6(11, 20)
          WM_6(12, 21) WM_6(13, 22) WM_6(14, 23)
          : "+&v"(f[0]), "+&v"(f[1]), "+&v"(f[2]), "+&v"(f[3]), "+&v"(f[4]), "+&v"(f[5])
          : "v"(C[0]), "v"(C[1]), "v"(C[2]), "v"(C[3]), "v"(C[4]), "v"(C[5]), "v"(C[6]),
            "v"(C[7]), "v"(C[8]), "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "v"(w[4]),
            "v"(w[5]), "v"(w[6]), "v"(w[7]), "v"(w[8]));
#undef WM_6
#undef WM_B
}

// The nine coefficients of a field in a cell from its 3 x 3 cells (T: rows of
// MW): the weights are w-(o) = 1/2 - o + o^2/2, w0(o) = 1/2 + o - o^2,
// w+(o) = o^2/2 of the offset o in the cell; C_ij at 3 i + j.
__device__ inline void coeffs(double (&C)[9], const double *T) {
  double R[3][3];
#pragma unroll
  for (int b = 0; b < 3; ++b) {
    const double m = T[b * MW], z = T[b * MW + 1], p = T[b * MW + 2];
    R[b][0] = 0.5 * (m + z);
    R[b][1] = z - m;
    R[b][2] = 0.5 * ((m - z) + (p - z));
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    C[3 * i] = 0.5 * (R[0][i] + R[1][i]);
    C[3 * i + 1] = R[1][i] - R[0][i];
    C[3 * i + 2] = 0.5 * ((R[0][i] - R[1][i]) + (R[2][i] - R[1][i]));
  }
}

// Workgroup (chunk, row block, species): see the file's head.  ACCL: update u
// over the moment step first.
//
// Bound by FP64 issue: about 390 vector instructions a round of a wavefront and
// 24 matrix products of 16 cycles, three quarters of the time at 512 x 512 cells
// with 64 particles per cell and species.  There 0.61 ms (0.79 with eight lanes a
// cell that read fields, weights and values from LDS, 123 reads and writes a
// round of 64 particles where these are 52, which kept LDS busy 74% of the time);
// 32 per cell 0.37 (0.48), 8 per cell 0.17 (0.21), 2 per cell 0.14 (0.13), 256 x
// 64 with 64: 62 us (95).  Half of the lanes' particles are staged at a time, for
// four wavefronts a SIMD instead of three: 0.64 -> 0.61 ms; loading a row's first
// particles during the row before gave nothing.
template <class S, bool ACCL>
__global__ __launch_bounds__(MC * MG, 4) void k_mom(MP P, FieldGeom fg,
                                                    const double *__restrict__ uf, S src,
                                                    double *__restrict__ part,
                                                    int *__restrict__ derr) {
  __shared__ double F[ACCL ? 6 * MH * MW : 1];
  // per cell, half of its 16 lanes' particles: moment values 1..6, weights 3 b + a
  __shared__ double St[MC * CST];
  __shared__ double Ct[MC * CSZ];                // per cell, its sums: [node row][a][moment]
  const int chunk = blockIdx.x, rb = blockIdx.y, s = blockIdx.z;
  const int c0 = chunk * MC, r0 = rb * MR;       // first cell, first row (local indices)
  if (ACCL) cell_fields<MW, MH>(F, P, fg, uf, c0 - 1, r0 - 1);
  __syncthreads();
  const int g = threadIdx.x / MG, sub = threadIdx.x % MG, lane = threadIdx.x & 63;
  const int i = c0 + g;
  const double q = P.q[s], rr = P.r[s];
  const double fac1 = q / rr * 0.5 * P.delt;     // mom_calc.f90:90-92
  const double txxx = fac1 * fac1;
  const double fac2 = q * P.delt / rr;
  const double ic2 = 1.0 / (P.c * P.c);
  bool bad = false;
  // The matrix products' operands: lane mi + 4 mb + 16 mk holds moment mi (of
  // four) and node column mi of cell mb (of the wavefront's four) and particle
  // mk (of four); of the result, moment mk and node column mi of cell mb.
  const int mi = lane & 3, mb = (lane >> 2) & 3, mk = lane >> 4;
  double *my = St + g * CST + (sub & 7) * NST;         // this lane's staging slot
  const double *rd = St + ((threadIdx.x >> 6) * 4 + mb) * CST + mk * NST;
  const double *rw = rd + NV + min(mi, 2);       // column 3 of a result is not used, nor is
  const double *r0v = rd + max(mi - 1, 0), *r1v = rd + min(3 + mi, NV - 1);   // moment 7
  double *out = Ct + ((threadIdx.x >> 6) * 4 + mb) * CSZ + mi * NMOM + mk;
  double acc[2][3] = {{0, 0, 0}, {0, 0, 0}};     // moments 0..3 and 4..6 at node rows rl + b
  for (int rl = 0; rl < MR; ++rl) {
    const int jl = r0 + rl;
    if (jl < P.ny) {                             // the same for the whole workgroup
      const int iabs = P.nxgs + i, jabs = P.nys + jl;
      size_t base = 0;
      int kb = 0, ke = 0;
      if (i < P.nx) src.range(P, s, jl, i, base, kb, ke);
      double C[9];
      if (ACCL) coeffs(C, F + (min(sub, 5) * MH + rl) * MW + g);
      // rounds of sixteen particles, one per lane; the next round's particle
      // is loaded while this one is computed, and where the one after that is
      int k = kb + sub;
      Pt nxt{0, 0, 0, 0, 0};
      unsigned at = 0;
      if constexpr (S::INDEXED) {
        if (k < ke) nxt = src.load(src.at(base + (size_t)k), iabs, jabs);
        if (k + MG < ke) at = src.at(base + (size_t)(k + MG));
      } else {
        if (k < ke) nxt = src.load(base + (size_t)k, iabs, jabs);
      }
      for (int k0 = kb; __ballot(k0 < ke) != 0ULL; k0 += MG, k += MG) {
        const Pt v = nxt;
        const bool live = k < ke;
        if constexpr (S::INDEXED) {
          if (k + MG < ke) nxt = src.load(at, iabs, jabs);
          if (k + 2 * MG < ke) at = src.at(base + (size_t)(k + 2 * MG));
        } else {
          if (k + MG < ke) nxt = src.load(base + (size_t)(k + MG), iabs, jabs);
        }
        double ux = v.ux, uy = v.uy, uz = v.uz;
        if (ACCL) {
          const double ox = v.x * P.d_delx - iabs, oy = v.y * P.d_delx - jabs;
          const double w[9] = {1.0,     oy,           oy * oy,      ox,         ox * oy,
                               ox * (oy * oy), ox * ox, (ox * ox) * oy, (ox * ox) * (oy * oy)};
          double f[6];
          gather(f, C, w);
          half_push(f, v, P, fac1, txxx, fac2, ux, uy, uz);
        }
        // mom_calc.f90:190-201: ih = int(x - 1/2) (truncation), the cell or
        // the one before it for a particle of this cell
        const double xs = v.x * P.d_delx - 0.5, ys = v.y * P.d_delx - 0.5;
        const int ih = (int)xs, jh = (int)ys;
        const int di = ih - iabs, dj = jh - jabs;
        const bool inside = di >= -1 && di <= 0 && dj >= -1 && dj <= 0;
        bad |= live && !inside;
        const bool on = live && inside;
        const double dx = xs - ih, dxm = 1.0 - dx, dy = ys - jh, dym = 1.0 - dy;
        // x weights of nodes i-1, i, i+1, y weights of nodes j-1, j, j+1
        const bool w0 = on && di < 0, w1 = on && di == 0, h0 = on && dj < 0, h1 = on && dj == 0;
        const double wx[3] = {w0 ? dxm : 0.0, w0 ? dx : (w1 ? dxm : 0.0), w1 ? dx : 0.0};
        const double wy[3] = {h0 ? dym : 0.0, h0 ? dy : (h1 ? dym : 0.0), h1 ? dy : 0.0};
        const double ig = 1.0 / sqrt(1.0 + (ux * ux + uy * uy + uz * uz) * ic2);
        // N, V, T: mom_calc.f90:203-243
        const double m[NV] = {ux * ig,      uy * ig,      uz * ig,
                              ux * ux * ig, uy * uy * ig, uz * uz * ig};
        const unsigned long long has = __ballot(live);
        // a cell's lanes are in one wavefront, whose LDS accesses complete in
        // order: the slots are written before any lane reads them, and read
        // before they are written again
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          if (h == 1 && !(has & 0xFF00FF00FF00FF00ULL)) continue;
          if (sub >> 3 == h) {
#pragma unroll
            for (int e = 0; e < NV; ++e) my[e] = on ? m[e] : 0.0;
#pragma unroll
            for (int e = 0; e < 9; ++e) my[NV + e] = wx[e % 3] * wy[e / 3];
          }
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
          __builtin_amdgcn_wave_barrier();
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
          for (int ks = 0; ks < 2; ++ks) {
            if (has & (0x000F000F000F000FULL << (4 * ks + 8 * h))) {
              const int o = ks * 4 * NST;
              const double a0 = mi == 0 ? 1.0 : r0v[o], a1 = r1v[o];
#pragma unroll
              for (int b = 0; b < 3; ++b) {
                const double wb = rw[o + 3 * b];
                acc[0][b] = __builtin_amdgcn_mfma_f64_4x4x4f64(a0, wb, acc[0][b], 0, 0, 0);
                acc[1][b] = __builtin_amdgcn_mfma_f64_4x4x4f64(a1, wb, acc[1][b], 0, 0, 0);
              }
            }
          }
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
          __builtin_amdgcn_wave_barrier();
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
      }
    }
    // node row rl has all of this column's cells
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      if (mi < 3 && 4 * e + mk < NMOM) out[rl * 3 * NMOM + 4 * e] = acc[e][0];
      acc[e][0] = acc[e][1];
      acc[e][1] = acc[e][2];
      acc[e][2] = 0.0;
    }
  }
#pragma unroll
  for (int e = 0; e < 2; ++e)
    if (mi < 3 && 4 * e + mk < NMOM) {
      out[MR * 3 * NMOM + 4 * e] = acc[e][0];
      out[(MR + 1) * 3 * NMOM + 4 * e] = acc[e][1];
    }
  __syncthreads();
  // node column c takes cells c-2, c-1, c in order
  double *T = part + (((size_t)s * P.nrb + rb) * P.nchunk + chunk) * TSZ;
  for (int t = threadIdx.x; t < TSZ; t += blockDim.x) {
    const int m = t % NMOM, c = (t / NMOM) % MW, r = t / (NMOM * MW);
    double sum = 0.0;
    for (int gg = max(0, c - 2); gg <= min(MC - 1, c); ++gg)
      sum += Ct[gg * CSZ + (r * 3 + (c - gg)) * NMOM + m];
    T[t] = sum;
  }
  if (bad) atomicOr(derr, DERR_RANGE);
}

// mom (7, nxgs-1:nxge+1, nys-1:nye+1, nsp) from the tiles: node (a, b)
// (offsets from nxgs-1, nys-1) is column a - ch*MC of chunk ch and row
// b - rb*MR of row block rb; the tiles add in ascending (rb, ch).  Block: the
// row, 256 of its values (moments fastest, as in the tiles), the species.
__global__ void k_mom_gather(MP P, const double *__restrict__ part, double *__restrict__ mom) {
  const int NXm = P.nx + 2, NYm = P.ny + 2;
  const int t = blockIdx.y * blockDim.x + threadIdx.x;
  if (t >= NMOM * NXm) return;
  const int m = t % NMOM, a = t / NMOM, b = blockIdx.x, s = blockIdx.z;
  double sum = 0.0;
  for (int rb = max(0, b / MR - 1); rb <= min(P.nrb - 1, b / MR); ++rb) {
    const int tr = b - rb * MR;
    if (tr >= MH) continue;
    for (int ch = max(0, a / MC - 1); ch <= min(P.nchunk - 1, a / MC); ++ch) {
      const int tc = a - ch * MC;
      if (tc >= MW) continue;
      sum += part[(((size_t)s * P.nrb + rb) * P.nchunk + ch) * TSZ + (tr * MW + tc) * NMOM + m];
    }
  }
  mom[((size_t)s * NYm + b) * (NMOM * NXm) + t] = sum;
}

// boundary_periodic.f90:579-584: the x ghosts into the opposite edge, every
// row; the wall families fold each into its own edge (boundary_shock.f90:
// 636-641, boundary_reconnection.f90:590-595).
__global__ void k_mom_fold_x(int nx, int ny, int nsp, double *mom, int wall) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= NMOM * (ny + 2) * nsp) return;
  const int m = t % NMOM, row = t / NMOM;        // row = b + (ny+2) * s
  double *r = mom + m + (size_t)NMOM * (nx + 2) * row;
  const double lo = r[0], hi = r[NMOM * (nx + 1)];
  r[NMOM * 1] += wall ? lo : hi;
  r[NMOM * nx] += wall ? hi : lo;
}

// boundary_periodic.f90:586-633 on one rank: row nys-1 into row nye, then
// row nye+1 into row nys, every column.
__global__ void k_mom_fold_y(int nx, int ny, int nsp, double *mom) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= NMOM * (nx + 2) * nsp) return;
  const int e = t % (NMOM * (nx + 2)), s = t / (NMOM * (nx + 2));
  const size_t rs = (size_t)NMOM * (nx + 2);
  double *c = mom + e + rs * (ny + 2) * s;
  c[rs * ny] += c[0];
  c[rs * 1] += c[rs * (ny + 1)];
}

MP make_mp(const wm_ctx *ctx) {
  const wm_grid &g = ctx->g;
  MP P;
  P.nx = g.nx;
  P.ny = g.ny;
  P.nxgs = g.nxgs;
  P.nys = g.nys;
  P.nsp = g.nsp;
  P.nchunk = wm_cdiv(g.nx, MC);
  P.nrb = wm_cdiv(g.ny, MR);
  P.cap = ctx->cap;
  P.d_delx = 1. / g.delx;
  P.c = g.c;
  P.delt = g.delt * 0.5;
  for (int s = 0; s < WM_MAXSP; ++s) {
    P.q[s] = s < g.nsp ? g.q[s] : 0.0;
    P.r[s] = s < g.nsp ? g.r[s] : 1.0;
  }
  return P;
}

template <class S, bool ACCL>
int launch_mom(wm_ctx *ctx, const MP &P, const S &src) {
  hipLaunchKernelGGL((k_mom<S, ACCL>), dim3(P.nchunk, P.nrb, P.nsp), dim3(MC * MG), 0, ctx->stream,
                     P, ctx->fg, ctx->uf, src, ctx->mom_part, ctx->derr);
  WM_HIP(hipGetLastError());
  return WM_OK;
}

}  // namespace

size_t wm_mom_elems(const wm_ctx *ctx) {
  return (size_t)NMOM * (ctx->g.nx + 2) * (ctx->g.ny + 2) * ctx->g.nsp;
}

int wm_mom_buffers(wm_ctx *ctx) {
  const MP P = make_mp(ctx);
  const size_t np = (size_t)P.nsp * P.nrb * P.nchunk * TSZ;
  if (!ctx->mom) WM_HIP(hipMalloc((void **)&ctx->mom, sizeof(double) * wm_mom_elems(ctx)));
  if (!ctx->mom_part) WM_HIP(hipMalloc((void **)&ctx->mom_part, sizeof(double) * np));
  return WM_OK;
}

// Into ctx->mom, allocated here on first use (read the pointer only after).
int wm_k_moments(wm_ctx *ctx, bool accl) {
  WM_TRY(wm_mom_buffers(ctx));
  const MP P = make_mp(ctx);
  if (ctx->form == WM_FORM_FP32) {
    if (!accl) return WM_ERR_ARG;
    const Src32 src{ctx->bins.q, ctx->bins.uz, ctx->bin_cnt, ctx->bstart};
    WM_TRY((launch_mom<Src32, true>(ctx, P, src)));
  } else {
    const PBank &A = ctx->bank[0];
    const Src64 src{A.x, A.y, A.ux, A.uy, A.uz, ctx->cumcnt};
    if (accl && ctx->perm_valid)
      WM_TRY((launch_mom<Order64, true>(
          ctx, P, Order64{src, ctx->perm, (size_t)ctx->g.ny * ctx->cap})));
    else if (accl)
      WM_TRY((launch_mom<Src64, true>(ctx, P, src)));
    else
      WM_TRY((launch_mom<Src64, false>(ctx, P, src)));
  }
  hipLaunchKernelGGL(k_mom_gather, dim3(P.ny + 2, wm_cdiv(NMOM * (P.nx + 2), 256), P.nsp), dim3(256),
                     0, ctx->stream, P,
                     ctx->mom_part, ctx->mom);
  WM_HIP(hipGetLastError());
  return WM_OK;
}

int wm_k_accl(wm_ctx *ctx, int src_bank, int dst_bank) {
  const MP P = make_mp(ctx);
  const PBank &A = ctx->bank[src_bank];
  const Src64 src{A.x, A.y, A.ux, A.uy, A.uz, ctx->cumcnt};
  hipLaunchKernelGGL(k_accl, dim3(P.ny, wm_cdiv(P.nx, AC), P.nsp), dim3(AC * AG), 0, ctx->stream, P,
                     ctx->fg, ctx->uf, src, ctx->bank[dst_bank]);
  WM_HIP(hipGetLastError());
  return WM_OK;
}

int wm_k_bc_mom(wm_ctx *ctx, double *mom) {
  const wm_grid &g = ctx->g;
  const int nxr = NMOM * (g.ny + 2) * g.nsp, nyr = NMOM * (g.nx + 2) * g.nsp;
  hipLaunchKernelGGL(k_mom_fold_x, dim3(wm_cdiv(nxr, 256)), dim3(256), 0, ctx->stream, g.nx, g.ny,
                     g.nsp, mom, ctx->bcf != WM_BC_PERIODIC);
  WM_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_mom_fold_y, dim3(wm_cdiv(nyr, 256)), dim3(256), 0, ctx->stream, g.nx, g.ny,
                     g.nsp, mom);
  WM_HIP(hipGetLastError());
  return WM_OK;
}
