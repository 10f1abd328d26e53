// wm_order.hip -- the row order between device-resident FP64 steps:
// particle_y and the sort (boundary_periodic.f90:99-248, sort.f90:36-82) as
// an index, not a move.
//
// The push leaves every particle where it found it in its row (sorted by old
// cell) with a 16-bit code: its new cell and whether it leaves the row.  The
// three kernels below turn the codes into the order the reference's
// particle_x, particle_y and sort__bucket would leave, as one 32-bit source
// index per new slot; the next push reads its particles through it and writes
// them sorted.  The IDs stay where they are until someone asks for them; a
// second index says which goes with which slot.  A step so reads and writes
// the 40 bytes of each particle's state once, plus about 20 of codes and
// indexes, where pushing in place, scanning for leavers and sorting moved 192
// bytes a particle.  Measured at 2048 x 2048, 64 particles per cell and
// species, beside the field solve: rows and merge 1.5, place 4.0 ms, where
// pass 1 took 6.0 and pass 2 with the sort 16.7 ms.
//
// The order.  Pass 1 lists a row's leavers (up, down) and their slots, the
// holes, in slot order.  Pass 2 puts arrival a (the neighbours' leavers,
// concatenated as the self-SENDRECVs do, :174-189) into hole a, or behind the
// row once the holes are used up; with fewer arrivals than holes the row's
// top m = holes - arrivals slots empty, their particles going, from the top,
// into the holes the arrivals leave (:193-236).  The sort is stable.  So the
// particles of new cell c are, in slot order, the row's own particles of old
// cells c-1, c, c+1 that now lie in c, merged by slot with the "displaced"
// ones, which pass 2 puts elsewhere than they were: arrivals and the top
// slots' particles.
//  k_order_rows:  per row, the leavers' lists and the holes, from the codes;
//  k_order_merge: per row, the displaced particles listed by new cell with
//                 the slots pass 2 puts them in, and the new cumcnt and np2
//                 (counts per old cell and kind of move come from the push);
//  k_order_place: per new cell, every particle's place: the number of the
//                 row's own particles of the cell before it (a ballot over
//                 the codes of three old cells) plus that of displaced ones.
#include "wm_internal.h"
#include "wm_order.h"

namespace {

constexpr int RT = 512;          // threads of a row's workgroup
constexpr int RW = RT / 64;

struct OP {
  int nx, ny, cap, mcap;
  int periodic;                  // x wraps
};

__device__ inline int wave_excl(int v, int &total) {
  const int lane = threadIdx.x & 63;
  int incl = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(incl, o, 64);
    if (lane >= o) incl += u;
  }
  total = __shfl(incl, 63, 64);
  return incl - v;
}

__device__ inline unsigned long long below_me() { return (1ULL << (threadIdx.x & 63)) - 1ULL; }

// The codes of slots k .. k + 7 (k a multiple of 8) in four words; slots past
// n read as staying.
__device__ inline uint4 codes8(const uint16_t *code, int k, int n) {
  uint4 v = make_uint4(0, 0, 0, 0);
  if (k < n) v = *(const uint4 *)(code + k);         // rows have a multiple of 16 slots
  if (k + 8 > n) {
    const int m = n - k;                             // codes that count
    v.x = m >= 2 ? v.x : (m == 1 ? v.x & 0xFFFFu : 0u);
    v.y = m >= 4 ? v.y : (m == 3 ? v.y & 0xFFFFu : 0u);
    v.z = m >= 6 ? v.z : (m == 5 ? v.z & 0xFFFFu : 0u);
    v.w = m == 7 ? v.w & 0xFFFFu : 0u;
  }
  return v;
}
// The low bits of each code of a word: bits 0 and 16 set where it goes up
// (down).
__device__ inline unsigned ups(unsigned w) { return w & ~(w >> 1) & 0x00010001u; }
__device__ inline unsigned downs(unsigned w) { return (w >> 1) & ~w & 0x00010001u; }

// Per row: its leavers (slot, new cell) up and down and its holes, ascending.
// Each wavefront walks an eighth of the row twice, 512 codes at a time: a
// count for the wavefronts' offsets, then the places.  2 bytes a particle.
__global__ __launch_bounds__(RT) void k_order_rows(OP P, const int *__restrict__ np2,
                                                   const uint16_t *__restrict__ code,
                                                   uint2 *__restrict__ lup, uint2 *__restrict__ ldn,
                                                   int *__restrict__ hole, int *__restrict__ nhole,
                                                   int *__restrict__ nup, int *__restrict__ ndn,
                                                   int *derr, unsigned long long *ts) {
  wm_stamp(ts, 5);
  __shared__ int su[RW], sd[RW];
  const int seg = blockIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int n = np2[seg];
  const uint16_t *cd = code + (size_t)seg * P.cap;
  const size_t mb = (size_t)seg * P.mcap;
  const int nch = (n + 511) / 512, per = (nch + RW - 1) / RW;
  const int c0 = min(nch, w * per), c1 = min(nch, c0 + per);
  int cu = 0, cdn = 0;
#pragma unroll 4
  for (int c = c0; c < c1; ++c) {
    const uint4 v = codes8(cd, c * 512 + lane * 8, n);
    cu += __popc(ups(v.x) | ups(v.y) << 1 | ups(v.z) << 2 | ups(v.w) << 3);
    cdn += __popc(downs(v.x) | downs(v.y) << 1 | downs(v.z) << 2 | downs(v.w) << 3);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    cu += __shfl_xor(cu, o, 64);
    cdn += __shfl_xor(cdn, o, 64);
  }
  if (lane == 0) {
    su[w] = cu;
    sd[w] = cdn;
  }
  __syncthreads();
  int bu = 0, bd = 0, tu = 0, td = 0;
#pragma unroll
  for (int v = 0; v < RW; ++v) {
    bu += v < w ? su[v] : 0;
    bd += v < w ? sd[v] : 0;
    tu += su[v];
    td += sd[v];
  }
  bool over = false;
#pragma unroll 4
  for (int c = c0; c < c1; ++c) {
    const int k = c * 512 + lane * 8;
    const uint4 q = codes8(cd, k, n);
    const int nu = __popc(ups(q.x) | ups(q.y) << 1 | ups(q.z) << 2 | ups(q.w) << 3);
    const int nd = __popc(downs(q.x) | downs(q.y) << 1 | downs(q.z) << 2 | downs(q.w) << 3);
    const int mine = nu | nd << 16;                  // at most 512 of either in a chunk
    if (__ballot(mine != 0) == 0ULL) continue;
    int tot;
    const int ex = wave_excl(mine, tot);
    int pu = bu + (ex & 0xFFFF), pd = bd + (ex >> 16);
    if (mine) {
      const unsigned v[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        const unsigned e = (v[b >> 1] >> (16 * (b & 1))) & 0xFFFFu, d = e & 3u;
        if (d != WM_CODE_UP && d != WM_CODE_DOWN) continue;
        if (pu + pd < 2 * P.mcap) hole[2 * mb + pu + pd] = k + b;
        else over = true;
        const int pos = d == WM_CODE_UP ? pu++ : pd++;
        if (pos < P.mcap) (d == WM_CODE_UP ? lup : ldn)[mb + pos] = make_uint2(k + b, e >> 2);
        else over = true;
      }
    }
    bu += tot & 0xFFFF;
    bd += tot >> 16;
  }
  if (threadIdx.x == 0) {
    nhole[seg] = min(tu + td, 2 * P.mcap);
    nup[seg] = min(tu, P.mcap);
    ndn[seg] = min(td, P.mcap);
  }
  if (over) atomicOr(derr, DERR_MOVER_OVER);
}

// Workgroup-wide exclusive prefix over the row's cells, thread th owning a
// run of them: value(i) in ascending order, emit(i, prefix).  Returns the
// total.  Every thread calls it; ends with a barrier.
template <class V, class E>
__device__ int cell_prefix(int nx, int *wsum, V value, E emit) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int per = (nx + RT - 1) / RT;
  const int lo = min(nx, (int)threadIdx.x * per), hi = min(nx, lo + per);
  int sum = 0;
  for (int i = lo; i < hi; ++i) sum += value(i);
  int tot64;
  const int ex = wave_excl(sum, tot64);
  if (lane == 63) wsum[w] = ex + sum;
  __syncthreads();
  int pre = 0, tot = 0;
#pragma unroll
  for (int v = 0; v < RW; ++v) {
    pre += v < w ? wsum[v] : 0;
    tot += wsum[v];
  }
  int run = pre + ex;
  for (int i = lo; i < hi; ++i) {
    const int c = value(i);
    emit(i, run);
    run += c;
  }
  __syncthreads();
  return tot;
}

// Per row: the new cumcnt and np2 from the push's counts per old cell and the
// arrivals, and the displaced particles listed by new cell, each with the
// slot pass 2 puts it in and the species-plane index it comes from.  The
// order inside a cell's list is left to k_order_place.
__global__ __launch_bounds__(RT) void k_order_merge(
    OP P, int *__restrict__ np2, int *__restrict__ nold, const uint16_t *__restrict__ code,
    const int4 *__restrict__ kind, int *__restrict__ farcnt, const int *__restrict__ far,
    const uint2 *__restrict__ lup, const uint2 *__restrict__ ldn, const int *__restrict__ hole,
    const int *__restrict__ nhole, const int *__restrict__ nup, const int *__restrict__ ndn,
    int *__restrict__ cumnew, uint2 *__restrict__ disp, int *__restrict__ dstart,
    int *__restrict__ rowok, int *derr) {
  extern __shared__ int dc[];                        // nx: displaced per new cell
  __shared__ int wsum[RW];
  const int seg = blockIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int s = seg / P.ny, jl = seg % P.ny;
  const int jb = jl == 0 ? P.ny - 1 : jl - 1, ja = jl == P.ny - 1 ? 0 : jl + 1;
  const bool first_row = jl == 0;                    // arrival order: see the file's head
  const int Fj = first_row ? ja : jb, Sj = first_row ? jb : ja;
  const int Fseg = s * P.ny + Fj, Sseg = s * P.ny + Sj;
  const uint2 *F = (first_row ? ldn : lup) + (size_t)Fseg * P.mcap;
  const uint2 *S = (first_row ? lup : ldn) + (size_t)Sseg * P.mcap;
  const int nF = first_row ? ndn[Fseg] : nup[Fseg], nS = first_row ? nup[Sseg] : ndn[Sseg];
  const int A = nF + nS, H = nhole[seg], N = np2[seg];
  const int newn = N + A - H, m = H - A;
  const int *hl = hole + 2 * (size_t)seg * P.mcap;
  const uint16_t *cd = code + (size_t)seg * P.cap;
  const int4 *kd = kind + (size_t)seg * P.nx;
  int *fc = farcnt + (size_t)seg * P.nx;
  const bool wide = far[seg] != 0;
  const bool fits = newn <= P.cap && newn >= 0;
  if (threadIdx.x == 0) {
    rowok[seg] = fits;
    nold[seg] = N;
    if (!fits) atomicOr(derr, DERR_NP_OVER);
  }
  if (!fits) {
    if (wide)
      for (int i = threadIdx.x; i < P.nx; i += RT) fc[i] = 0;
    return;
  }
  for (int i = threadIdx.x; i < P.nx; i += RT) dc[i] = 0;
  __syncthreads();
  auto arrival = [&](int a) { return a < nF ? F[a] : S[a - nF]; };
  for (int a = threadIdx.x; a < A; a += RT) atomicAdd(&dc[arrival(a).y], 1);
  __syncthreads();
  // cumcnt: the row's own particles of new cell i, by kind of move from the
  // cells around it, and the arrivals
  {
    int *cc = cumnew + (size_t)seg * (P.nx + 1);
    const int tot = cell_prefix(
        P.nx, wsum,
        [&](int i) {
          const int l = i > 0 ? i - 1 : (P.periodic ? P.nx - 1 : -1);
          const int r = i + 1 < P.nx ? i + 1 : (P.periodic ? 0 : -1);
          int c = kd[i].y + dc[i];
          if (l >= 0) c += kd[l].z;
          if (r >= 0) c += kd[r].x;
          if (wide) c += fc[i];
          return c;
        },
        [&](int i, int run) { cc[i] = run; });
    if (threadIdx.x == 0) {
      cc[P.nx] = tot;
      if (tot != newn) atomicOr(derr, DERR_RANGE);   // a particle outside the row's cells
    }
  }
  if (wide)
    for (int i = threadIdx.x; i < P.nx; i += RT) fc[i] = 0;   // zero again for the next step
  // the top slots' particles: the r-th from the top that stays goes to hole
  // A + r; f(slot, r) for each, every thread of the workgroup calls it
  auto vacated = [&](auto f) {
    int run = 0;
    for (int q0 = 0; q0 < m; q0 += RT) {
      const int slot = N - 1 - (q0 + (int)threadIdx.x);
      unsigned d = WM_CODE_UP;
      if (q0 + (int)threadIdx.x < m) d = cd[slot] & 3u;
      const bool stays = d != WM_CODE_UP && d != WM_CODE_DOWN;
      const unsigned long long bm = __ballot(stays);
      if (lane == 0) wsum[w] = __popcll(bm);
      __syncthreads();
      int pre = 0, tot = 0;
#pragma unroll
      for (int v = 0; v < RW; ++v) {
        pre += v < w ? wsum[v] : 0;
        tot += wsum[v];
      }
      const int r = run + pre + __popcll(bm & below_me());
      if (stays && A + r < H) f(slot, r);
      run += tot;
      __syncthreads();
    }
  };
  vacated([&](int slot, int) { atomicAdd(&dc[cd[slot] >> 2], 1); });
  __syncthreads();
  {
    int *ds = dstart + (size_t)seg * (P.nx + 1);
    // dc becomes each cell's running place in the list (a thread's own cells)
    const int tot = cell_prefix(
        P.nx, wsum, [&](int i) { return dc[i]; },
        [&](int i, int run) {
          ds[i] = run;
          dc[i] = run;
        });
    if (threadIdx.x == 0) ds[P.nx] = tot;
  }
  uint2 *dl = disp + 2 * (size_t)seg * P.mcap;       // at most max(A, H) entries
  const unsigned Fb = (unsigned)Fj * (unsigned)P.cap, Sb = (unsigned)Sj * (unsigned)P.cap;
  const unsigned own = (unsigned)jl * (unsigned)P.cap;
  for (int a = threadIdx.x; a < A; a += RT) {
    const uint2 e = arrival(a);
    const int p = atomicAdd(&dc[e.y], 1);
    dl[p] = make_uint2(a < H ? hl[a] : N + (a - H), (a < nF ? Fb : Sb) + e.x);
  }
  vacated([&](int slot, int r) {
    const int p = atomicAdd(&dc[cd[slot] >> 2], 1);
    dl[p] = make_uint2(hl[A + r], own + (unsigned)slot);
  });
  if (threadIdx.x == 0) np2[seg] = newn;
}

struct Place {
  const int *nold, *rowok, *cumold, *cumnew, *far, *dstart;
  const uint16_t *code;
  const int4 *kind;
  const uint2 *disp;
  unsigned *perm;
  const unsigned *oid;           // whose ID each slot's particle has (null: its own)
  unsigned *oidd;
};

// A row with particles that crossed more than one cell (mirrored by a wall
// from a cell beyond it, at most in a run's first step): the places of the
// particles of new cell c by one wavefront, which looks for them in the whole
// row, 64 codes at a time.
__device__ bool place_wide(const OP &P, const Place &R, int seg, int c) {
  const int lane = threadIdx.x & 63;
  const int jl = seg % P.ny;
  const size_t base = (size_t)seg * P.cap, plane = base - (size_t)jl * P.cap;
  const unsigned own = (unsigned)jl * (unsigned)P.cap;
  const uint16_t *cd = R.code + base;
  const int *cn = R.cumnew + (size_t)seg * (P.nx + 1), *ds = R.dstart + (size_t)seg * (P.nx + 1);
  const uint2 *dl = R.disp + 2 * (size_t)seg * P.mcap;
  const int newn = cn[P.nx], keep = min(R.nold[seg], newn);
  const int start = cn[c], d0 = ds[c], D = ds[c + 1] - d0;
  bool bad = false;
  // displaced particles 64 at a time (one lane each); the row's own are placed
  // in the first round
  for (int e0 = 0; e0 == 0 || e0 < D; e0 += 64) {
    const bool mine = e0 + lane < D;
    uint2 de = make_uint2(0u, 0u);
    if (mine) de = dl[d0 + e0 + lane];
    int nb = 0, run = 0;                             // own particles below the displaced one; so far
    for (int k0 = 0; k0 < keep; k0 += 64) {
      const int k = k0 + lane;
      const unsigned v = k < keep ? cd[k] : 0u;
      const bool hit = k < keep && (int)(v >> 2) == c &&
                       ((v & 3u) == WM_CODE_STAY || (v & 3u) == WM_CODE_FAR);
      const unsigned long long bm = __ballot(hit);
      const int below = (int)de.x - k0;
      if (mine) nb += below <= 0 ? 0 : __popcll(below >= 64 ? bm : bm & ((1ULL << below) - 1ULL));
      if (e0 == 0 && hit) {
        int dst = start + run + __popcll(bm & below_me());
        for (int i = 0; i < D; ++i) dst += (int)dl[d0 + i].x < k;
        if (dst < newn) {
          R.perm[base + dst] = own + (unsigned)k;
          R.oidd[base + dst] = R.oid ? R.oid[base + k] : own + (unsigned)k;
        } else {
          bad = true;
        }
      }
      run += __popcll(bm);
    }
    if (mine) {
      int dst = start + nb;
      for (int i = 0; i < D; ++i) dst += (int)dl[d0 + i].x < (int)de.x;
      if (dst < newn) {
        R.perm[base + dst] = de.y;
        R.oidd[base + dst] = R.oid ? R.oid[plane + de.y] : de.y;
      } else {
        bad = true;
      }
    }
  }
  return bad;
}

// The place of every particle, as the index it comes from, and whose ID it has
// (an index into the IDs, which stay where they are until the rows are read as
// rows).  A group of 16 lanes per cell o, in two parts.
//
// The row's own particles of old cell o (16 codes at a time, ballots): one
// that goes to cell c in {o-1, o, o+1} comes after the particles of lower
// cells that go to c (counted by the push), after those of its own cell with
// lower slots that go the same way, and after the displaced particles of c
// with lower slots.  Where some of the latter have slots among the cell's own
// (near a row's ends), bitmaps of those slots are made in LDS, 512 slots at a
// time, and each window adds the bits below it.
//
// The displaced particles of new cell o: after the row's own of the cell with
// lower slots -- whole cells' counts, or the part of a cell before the slot
// from the tables that its group left (per window: the particles that stay,
// go right, go left, and how many before it) -- and the displaced ones with
// lower slots.
//
// 2 B of code, 4 B of index and 8 B of ID index per particle, three dependent round
// trips to memory a cell, which bound it; six wavefronts a SIMD hide most.  Where
// a plasma has pinched (256 x 64 cells, 407 particles in the densest at a mean
// of 64) the longest cells set the time: 42 us, and 124 where every window
// compared itself with each displaced particle and each of those searched the
// codes again.
constexpr int PG = 16;           // lanes of a cell
constexpr int PT = 256;
constexpr int PCELL = PT / PG;   // cells of a workgroup
constexpr int PWIN = 4;          // windows of a cell in flight
constexpr int PD = 64;           // displaced particles of a cell ranked from LDS at a time
constexpr int PWT = 32;          // windows of a cell in the tables and bitmaps
__global__ __launch_bounds__(PT, 6) void k_order_place(OP P, Place R, int *derr,
                                                     unsigned long long *ts) {
  wm_stamp(ts, 6);
  __shared__ __attribute__((aligned(16))) int slots[PCELL][PD];
  __shared__ unsigned tab[3][PCELL][PWT];            // stay, right, left: count << 16 | lanes
  __shared__ unsigned bits[3][PCELL][PWT / 2];       // displaced of o, r, l by slot - ks
  constexpr int NONE = 0x7FFFFFFF;
  const int seg = blockIdx.y;
  const int sub = threadIdx.x % PG, g = threadIdx.x / PG, gsh = (threadIdx.x & 63) / PG * PG;
  const int nx = P.nx, jl = seg % P.ny;
  const bool act = (int)blockIdx.x * PCELL + g < nx;
  const int o = min(nx - 1, (int)blockIdx.x * PCELL + g);
  const size_t base = (size_t)seg * P.cap, plane = base - (size_t)jl * P.cap;
  const unsigned own = (unsigned)jl * (unsigned)P.cap;
  const uint16_t *cd = R.code + base;
  const int *co = R.cumold + (size_t)seg * (nx + 1), *cn = R.cumnew + (size_t)seg * (nx + 1);
  const int *ds = R.dstart + (size_t)seg * (nx + 1);
  const int4 *kd = R.kind + (size_t)seg * nx;
  const uint2 *dl = R.disp + 2 * (size_t)seg * P.mcap;
  // first round trip: everything about the cell and its neighbours (walls
  // have none beyond the ends: their counts are zero)
  const bool hasl = o > 0 || P.periodic, hasr = o + 1 < nx || P.periodic;
  const int l = o > 0 ? o - 1 : nx - 1, r = o + 1 < nx ? o + 1 : 0, ll = o > 1 ? o - 2 : 0;
  const int rowok = R.rowok[seg], far = R.far[seg], nold = R.nold[seg], newn = cn[nx];
  const int kb = max(0, co[o]), ke = act ? min(P.cap, co[o + 1]) : kb;
  const int start = cn[o], sl = cn[l], sr = cn[r];
  const int d0 = ds[o], d1 = ds[o + 1], dl0 = ds[l], dl1 = ds[l + 1], dr0 = ds[r], dr1 = ds[r + 1];
  const int4 ko = kd[o], kl_ = kd[l], kr_ = kd[r], kll_ = kd[ll], k0_ = kd[0], k1_ = kd[1];
  if (!rowok) return;
  bool bad = false;
  if (far) {
    const int c1 = min(nx, (int)(blockIdx.x + 1) * PCELL);
    for (int c = blockIdx.x * PCELL + (threadIdx.x >> 6); c < c1; c += PT / 64)
      bad |= place_wide(P, R, seg, c);
    if (bad) atomicOr(derr, DERR_RANGE);
    return;
  }
  const int keep = min(nold, newn);
  const int toR = ko.z, toL = ko.x;                  // the cell's particles that go right, left
  const int fromL = hasl ? kl_.z : 0, fromR = hasr ? kr_.x : 0;   // the neighbours' that come here
  const int D = act ? d1 - d0 : 0;
  const int Dl = act && toL > 0 ? dl1 - dl0 : 0, Dr = act && toR > 0 ? dr1 - dr0 : 0;
  const bool tabled = ke - kb <= PG * PWT;
  // second round trip: the first codes and IDs, the displaced particles (the
  // first 16 of each list in registers)
  unsigned cv[PWIN], iv[PWIN];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int w = 0; w < PWIN; ++w) {
      const int k = k0 + w * PG + sub;
      cv[w] = 0xFFFFFFFFu;
      iv[w] = 0;
      if (k < ke) {
        cv[w] = cd[k];
        iv[w] = R.oid ? R.oid[base + k] : own + (unsigned)k;
      }
    }
  };
  const uint2 de0 = sub < D ? dl[d0 + sub] : make_uint2(NONE, 0u);
  const int pL = sub < Dl ? (int)dl[dl0 + sub].x : NONE, pR = sub < Dr ? (int)dl[dr0 + sub].x : NONE;
  fetch(kb);
  const unsigned di0 = sub < D && R.oid ? R.oid[plane + de0.y] : de0.y;   // (the third)
  auto ballot16 = [&](bool b) { return (unsigned)(__ballot(b) >> gsh) & 0xFFFFu; };
  const unsigned below = (1u << sub) - 1u;
  auto low16 = [](int n) { return n <= 0 ? 0u : n >= 16 ? 0xFFFFu : (1u << n) - 1u; };
  // f(slot) for each displaced particle of a list (its first 16 in p)
  auto each = [&](int p, int f0, int n, auto f) {
    f(p);
    for (int i0 = PG; i0 < n; i0 += PG) f(i0 + sub < n ? (int)dl[f0 + i0 + sub].x : NONE);
  };
  // how many of them have slots below kb; do any inside [kb, ke)
  bool in = false;
  auto lower = [&](int p, int f0, int n) {
    int c = 0;
    each(p, f0, n, [&](int q) {
      c += __popc(ballot16(q < kb));
      in |= ballot16(q >= kb && q < ke) != 0u;
    });
    return c;
  };
  // first place of the cell's particles that stay, go right, go left
  const int wrapL = P.periodic && o == nx - 1 ? k0_.x : 0;   // cell 0's that come to the last cell
  int bS = start + (o > 0 ? fromL : 0) + wrapL + lower((int)de0.x, d0, D);
  int bR = sr + (o < nx - 1 ? (P.periodic && o + 1 == nx - 1 ? k0_.x : 0) : k0_.y + k1_.x) +
           lower(pR, dr0, Dr);
  int bL = sl + (o > 0 ? (o > 1 ? kll_.z : 0) + kl_.y : 0) + lower(pL, dl0, Dl);
  int cS = 0, cR = 0, cL = 0;                        // the cell's own so far
  for (int k0 = kb; k0 < ke; k0 += PWIN * PG) {
    if (k0 > kb) fetch(k0);
    const int seg0 = (k0 - kb) & (PG * PWT - 1);     // within the bitmaps' 512 slots
    if (in && seg0 == 0) {
      __builtin_amdgcn_wave_barrier();               // what was there has been read
      for (int i = sub; i < PWT / 2; i += PG) bits[0][g][i] = bits[1][g][i] = bits[2][g][i] = 0u;
      __builtin_amdgcn_wave_barrier();
      auto mark = [&](unsigned *b, int p, int f0, int n) {
        each(p, f0, n, [&](int q) {
          const int at = q - k0;
          if (at >= 0 && at < PG * PWT && q < ke) atomicOr(b + (at >> 5), 1u << (at & 31));
        });
      };
      mark(bits[0][g], (int)de0.x, d0, D);
      mark(bits[1][g], pR, dr0, Dr);
      mark(bits[2][g], pL, dl0, Dl);
      __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (int w = 0; w < PWIN; ++w) {
      const int k = k0 + w * PG + sub;
      if (k - sub >= ke) break;
      const int c = (int)(cv[w] >> 2);
      const bool own_ = k < keep && (cv[w] & 3u) == WM_CODE_STAY;   // (none past ke: all bits set)
      const bool moves = own_ && c != o, right = c == r;
      const unsigned mS = ballot16(own_ && c == o), mM = ballot16(moves);
      unsigned mR = 0, mL = 0;
      int dst = bS + cS + __popc(mS & below);
      if (mM) {                                      // uniform over the group
        mR = ballot16(moves && right);
        mL = mM & ~mR;
        if (moves) dst = right ? bR + cR + __popc(mR & below) : bL + cL + __popc(mL & below);
      }
      if (in) {                                      // displaced slots among the cell's own
        const int at = seg0 + w * PG;
        unsigned d[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) d[q] = (bits[q][g][at >> 5] >> (at & 31)) & 0xFFFFu;
        dst += __popc((!moves ? d[0] : (right ? d[1] : d[2])) & below);
        bS += __popc(d[0]);
        bR += __popc(d[1]);
        bL += __popc(d[2]);
      }
      if (tabled && sub < 3)
        tab[sub][g][(k - sub - kb) / PG] =
            sub == 0 ? (unsigned)cS << 16 | mS : (sub == 1 ? (unsigned)cR << 16 | mR : (unsigned)cL << 16 | mL);
      cS += __popc(mS);
      cR += __popc(mR);
      cL += __popc(mL);
      if (own_) {
        if (dst < newn) {
          R.perm[base + dst] = own + (unsigned)k;
          R.oidd[base + dst] = iv[w];
        } else {
          bad = true;
        }
      }
    }
  }
  __syncthreads();                                   // the neighbours' tables
  // the displaced particles of cell o, 16 at a time, each ranked among all
  // (more than 16: their slots in LDS, PD at a time, padded to fours)
  int *const sl_ = slots[g];
  auto stage = [&](int f) {
    __builtin_amdgcn_wave_barrier();                 // what was there has been read
    for (int i = sub; i < min(PD, (D - f + 3) & ~3); i += PG)
      sl_[i] = f + i < D ? (int)dl[d0 + f + i].x : NONE;
    __builtin_amdgcn_wave_barrier();
  };
  if (D > PG && D <= PD) stage(0);
  const int lb = max(0, co[l]), le = min(P.cap, co[l + 1]), rb = max(0, co[r]), re = min(P.cap, co[r + 1]);
  for (int i0 = 0; i0 < D; i0 += PG) {
    const bool mine = i0 + sub < D;
    uint2 de = de0;
    unsigned v = di0;
    if (i0 > 0) {
      de = mine ? dl[d0 + i0 + sub] : make_uint2(NONE, 0u);
      v = mine && R.oid ? R.oid[plane + de.y] : de.y;
    }
    const int p = (int)de.x;
    int dst = start;
    if (D <= PG) {
      for (int i = 0; i < D; ++i) dst += __shfl(p, gsh + i, 64) < p;
    } else {
      for (int f = 0; f < D; f += PD) {
        if (D > PD) stage(f);
        for (int i = 0; i < min(PD, D - f); i += 4) {
          const int4 q = *(const int4 *)(sl_ + i);
          dst += (q.x < p) + (q.y < p) + (q.z < p) + (q.w < p);
        }
      }
    }
    // the row's own particles with lower slots, by the cell [b, e) they come
    // from: a whole cell's count n, or what its table t has up to the slot;
    // without one (another workgroup's cell, a long one), its codes
    auto from = [&](int b, int e, int n, const unsigned *t) {
      const bool part = mine && p > b && p < e;
      if (mine && p >= e) dst += n;
      if (ballot16(part) == 0u) return;
      if (t && e - b <= PG * PWT) {
        if (part) {
          const unsigned q = t[(p - b) / PG];
          dst += (int)(q >> 16) + __popc(q & low16((p - b) % PG));
        }
        return;
      }
      const unsigned way = (unsigned)o << 2 | WM_CODE_STAY;
      const int upto = part ? p : b;
      for (int k0 = b; k0 < e; k0 += PWIN * PG) {
        unsigned c[PWIN];
#pragma unroll
        for (int w = 0; w < PWIN; ++w) {
          const int k = k0 + w * PG + sub;
          c[w] = k < e ? cd[k] : 0xFFFFFFFFu;
        }
#pragma unroll
        for (int w = 0; w < PWIN; ++w)
          dst += __popc(ballot16(c[w] == way) & low16(upto - (k0 + w * PG)));
      }
    };
    from(kb, ke, ko.y, tab[0][g]);
    if (fromL) from(lb, le, fromL, g > 0 ? tab[1][g - 1] : nullptr);
    if (fromR) from(rb, re, fromR, g + 1 < PCELL && o + 1 < nx ? tab[2][g + 1] : nullptr);
    if (mine) {
      if (dst < newn) {
        R.perm[base + dst] = de.y;
        R.oidd[base + dst] = v;
      } else {
        bad = true;
      }
    }
  }
  if (bad) atomicOr(derr, DERR_RANGE);
  // the end: of a row's last workgroup, every 16th row's and the last's
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0 &&
      ((blockIdx.y & 15) == 15 || blockIdx.y == gridDim.y - 1))
    atomicMax(ts + 7, (unsigned long long)wall_clock64());
}

// The rows in their order: slot k of the result is what the index gives it.
__global__ __launch_bounds__(256) void k_order_apply(int cap, int ny, const int *__restrict__ np2,
                                                     const unsigned *__restrict__ perm, Rec64 A,
                                                     Rec64 B) {
  const int seg = blockIdx.y, n = np2[seg];
  const size_t base = (size_t)seg * cap, plane = (size_t)(seg / ny) * ny * cap;
  for (int k = blockIdx.x * 256 + threadIdx.x; k < n; k += 256 * gridDim.x)
    B.store(base + k, A.load(plane + perm[base + k]));
}
// Their IDs: gathered (an index that a row without a place left is kept inside
// the plane), then put in place.
__global__ __launch_bounds__(256) void k_ids_gather(int cap, int ny, const int *__restrict__ np2,
                                                    const unsigned *__restrict__ oid,
                                                    const int64_t *__restrict__ id,
                                                    int64_t *__restrict__ to) {
  const int seg = blockIdx.y, n = np2[seg];
  const size_t len = (size_t)ny * cap;
  const size_t base = (size_t)seg * cap, plane = (size_t)(seg / ny) * len;
  for (int k = blockIdx.x * 256 + threadIdx.x; k < n; k += 256 * gridDim.x)
    to[base + k] = id[plane + min((size_t)oid[base + k], len - 1)];
}
__global__ __launch_bounds__(256) void k_ids_put(int cap, const int *__restrict__ np2,
                                                 const int64_t *__restrict__ from,
                                                 int64_t *__restrict__ id) {
  const int seg = blockIdx.y, n = np2[seg];
  const size_t base = (size_t)seg * cap;
  for (int k = blockIdx.x * 256 + threadIdx.x; k < n; k += 256 * gridDim.x)
    id[base + k] = from[base + k];
}

}  // namespace

// particle_y and the sort of the pushed rows (bank 0, in the slots the push
// read them from): the order of the rows into ctx->perm, the IDs, cumcnt and
// np2 moved on.
int wm_k_order(wm_ctx *ctx) {
  const wm_grid &g = ctx->g;
  const OP P{g.nx, g.ny, ctx->cap, ctx->mcap, ctx->bcf == WM_BC_PERIODIC};
  const int nseg = g.nsp * g.ny;
  const size_t lds = sizeof(int) * (size_t)g.nx;
  if (ctx->form == WM_FORM_FP32 || lds > 65536) {
    wm_set_error(ctx, WM_ERR_ARG, "particle_y + sort: FP64 rows of at most 16384 cells");
    return WM_ERR_ARG;
  }
  hipLaunchKernelGGL(k_order_rows, dim3(nseg), dim3(RT), 0, ctx->stream, P, ctx->np2, ctx->code,
                     ctx->lup, ctx->ldn, ctx->hole, ctx->nhole, ctx->nup, ctx->ndn, ctx->derr,
                     ctx->ts);
  hipLaunchKernelGGL(k_order_merge, dim3(nseg), dim3(RT), lds, ctx->stream, P, ctx->np2, ctx->nold,
                     ctx->code, ctx->kind, ctx->farcnt, ctx->far, ctx->lup, ctx->ldn, ctx->hole,
                     ctx->nhole, ctx->nup, ctx->ndn, ctx->cumnew, ctx->disp, ctx->dstart,
                     ctx->rowok, ctx->derr);
  // the IDs' indexes of this order and the last share the spare ID array
  unsigned *const o = (unsigned *)ctx->id[1 - ctx->idcur];
  const size_t slots = (size_t)nseg * ctx->cap;
  const int now = ctx->perm_valid ? ctx->oidcur : 1;
  const Place R{ctx->nold, ctx->rowok, ctx->cumcnt, ctx->cumnew, ctx->far, ctx->dstart, ctx->code,
                ctx->kind, ctx->disp, ctx->perm, ctx->perm_valid ? o + now * slots : nullptr,
                o + (1 - now) * slots};
  hipLaunchKernelGGL(k_order_place, dim3(wm_cdiv(g.nx, PCELL), nseg), dim3(PT), 0, ctx->stream, P,
                     R, ctx->derr, ctx->ts);
  WM_HIP(hipGetLastError());
  ctx->oidcur = 1 - now;
  std::swap(ctx->cumcnt, ctx->cumnew);
  ctx->perm_valid = true;
  return WM_OK;
}

// Where the particles' IDs are (species-plane indexes by slot) while the IDs lie
// as they did when the order began.
const unsigned *wm_order_ids(const wm_ctx *ctx) {
  if (!ctx->perm_valid) return nullptr;
  return (const unsigned *)ctx->id[1 - ctx->idcur] +
         (size_t)ctx->oidcur * ctx->g.nsp * ctx->g.ny * ctx->cap;
}

// Bank 0 put in its order (for whoever reads the rows as rows).
int wm_order_apply(wm_ctx *ctx) {
  if (!ctx->perm_valid) return WM_OK;
  const wm_grid &g = ctx->g;
  const dim3 grid(std::max(1, std::min(64, wm_cdiv(ctx->cap, 1024))), g.nsp * g.ny);
  hipLaunchKernelGGL(k_order_apply, grid, dim3(256), 0, ctx->stream, ctx->cap, g.ny, ctx->np2,
                     ctx->perm, ctx->bank[0], ctx->bank[1]);
  // (bank 0's records have moved: its space holds the IDs on their way)
  const unsigned *oid = wm_order_ids(ctx);
  int64_t *const tmp = (int64_t *)ctx->bank[0].x;
  hipLaunchKernelGGL(k_ids_gather, grid, dim3(256), 0, ctx->stream, ctx->cap, g.ny, ctx->np2, oid,
                     ctx->id[ctx->idcur], tmp);
  hipLaunchKernelGGL(k_ids_put, grid, dim3(256), 0, ctx->stream, ctx->cap, ctx->np2, tmp,
                     ctx->id[ctx->idcur]);
  WM_HIP(hipGetLastError());
  std::swap(ctx->bank[0], ctx->bank[1]);
  ctx->perm_valid = false;
  return WM_OK;
}
