// Short row segments of the batched step: the speed pass and the update of a
// step with too few patches to fill the GPU by marching.
//
// Such a step is bound by latency, not by HBM: a wavefront of the row march
// (pc_kernels.hpp) walks at least 8 rows one after another, a dependent chain
// of FP64 operations per row and one row of loads in flight, after a chain of
// about ten dependent descriptor loads.  Here a wavefront takes at most R
// rows of its patches (R a template parameter), issues the loads of all its
// rows at once, and does all its edges as straight-line code, so the chains
// of the rows overlap; everything a patch needs besides its cells is in one
// record (SegDesc).  The x-edges between two segments are solved by both
// (the same operands, so the same bits).  The step is two launches, exact
// speeds and update; the update takes its dt from the speed pass's block
// minima itself, so there is no reduction launch and none for a fallback.
// 9 x 9 patches of 16^2, f-wave: 34.7 -> 13.9 us a step (speeds 5.4, update
// 5.6, the rest launches; five launches before, update 16.9); 24 x 24 of
// 32^2: 40.6 -> 28.0 us; 16 x 16 of 32^2, augmented: 182 -> 57 us.
//
// Results are those of the row march bit for bit: the same operations per
// edge and the same order of accumulation per cell (x-left, x-right, y-up,
// y-down).
#pragma once

#include "pc_kernels.hpp"

namespace pcamd {

// Everything the segment kernels read of a patch besides its cells.
//   gx[s]: index of column 0 of the row across x side s: the neighbour's
//          boundary row, the own boundary row (wall) or the own ghost row;
//   gy[s]: index, in row 0, of the cell across y side s (row r: + r stride);
//   neg:   bit k set: side k (x-, x+, y-, y+) is a wall, its normal momentum
//          negated.
struct SegDesc {
  long long off;
  long long gx[2];
  long long gy[2];
  int nx, ny, stride, neg;
  int slot, scn;
  double dx, dy, dxinv, dyinv;
};

// What one wavefront reads first: records recs[wave * group .. + nseg) of the
// patches of its task with the rows it takes.  A kernel starts on cold caches
// (another XCD wrote what it reads), every dependent load costs 0.7-0.9 us,
// and a record's place follows from the wavefront's number alone, so cells
// are one load away instead of three (task -> patch list -> patch).
struct alignas(128) SegRec {
  SegDesc d;
  int r0, r1, sidx, nseg;
};

// The records of a launch.  lanes: lanes per patch (columns rounded up to a
// power of two) where it is the same for all, else 0; scn: likewise the
// scenario, else -1.
struct SegList {
  const SegRec* recs;
  int group, lanes, scn;
};

// Records from tasks and patch descriptions, one thread per record.
__global__ void __launch_bounds__(256)
k_seg_records(const Task* __restrict__ tasks, const SegDesc* __restrict__ desc, int n, int group,
              SegRec* __restrict__ recs) {
  const int k = blockIdx.x * 256 + threadIdx.x;
  if (k >= n) return;
  const Task t = tasks[k / group];
  const int s = k % group;
  SegRec r;
  r.d = desc[t.first + (s < t.nseg ? s : 0)];
  r.r0 = t.r0;
  r.r1 = t.r1;
  r.sidx = t.sidx;
  r.nseg = t.nseg;
  recs[k] = r;
}

// Slots per patch of the segments' speed maxima (nx <= 64 rows).
constexpr int kSegSlots = 64;
constexpr int kSegWaves = 4;  // wavefronts (independent tasks) per workgroup
constexpr double kNoLimit = 1.7976931348623157e308;

// Segments of a patch with nx rows, at most R rows each.
__host__ __device__ __forceinline__ int seg_count(int nx, int R) { return (nx + R - 1) / R; }

// Net updates of one f-wave edge of two wet cells before they are handed to
// the cells on its sides.
struct WetEdge {
  double s1, s2, b1, b2;
};

__device__ __forceinline__ WetEdge wet_edge(const CellQ& L, const CellQ& R) {
  WetEdge e;
  wave_speeds_wet(L, R, e.s1, e.s2);
  const double d0 = R.q - L.q;
  const double d1 = (R.f - L.f) + (kHalfG * (L.h + R.h)) * (R.b - L.b);
  const double inv = div_nr(1.0, e.s2 - e.s1);
  e.b1 = (e.s2 * d0 - d1) * inv;
  e.b2 = (d1 - e.s1 * d0) * inv;
  return e;
}

// The edge's four shares.  `sub`: every edge of the wavefront is subsonic
// (wave 1 goes left, wave 2 right); the signs of zeros that may differ from
// the general sums do not reach a cell (see edge_solve_wet).
__device__ __forceinline__ void wet_shares(const WetEdge& e, bool sub, double& dhL, double& dhR,
                                           double& dqL, double& dqR) {
  const double z1 = e.b1 * e.s1, z2 = e.b2 * e.s2;
  if (sub) {
    dhL = e.b1; dqL = z1; dhR = e.b2; dqR = z2;
    return;
  }
  double a = 0.0, b = 0.0, c = 0.0, d = 0.0;
  if (e.s1 < -kZeroTol) {
    a += e.b1; c += z1;
  } else if (e.s1 > kZeroTol) {
    b += e.b1; d += z1;
  } else {
    a += 0.5 * e.b1; c += 0.5 * z1;
    b += 0.5 * e.b1; d += 0.5 * z1;
  }
  if (e.s2 < -kZeroTol) {
    a += e.b2; c += z2;
  } else if (e.s2 > kZeroTol) {
    b += e.b2; d += z2;
  } else {
    a += 0.5 * e.b2; c += 0.5 * z2;
    b += 0.5 * e.b2; d += 0.5 * z2;
  }
  dhL = a; dhR = b; dqL = c; dqR = d;
}

__device__ __forceinline__ CellQ left_cell(const CellQ& c) {
  CellQ l;
  l.h = from_left(c.h); l.q = from_left(c.q); l.b = from_left(c.b);
  l.u = from_left(c.u); l.sq = from_left(c.sq); l.c = from_left(c.c);
  l.f = from_left(c.f);
  return l;
}

// The rows of one wavefront and the lanes' places in them.
struct SegLane {
  const SegRec* recs;    // of this wavefront
  int ra, rb, rows;      // interior rows ra..rb of the patch
  int nx, ny, nseg, sidx;
  int lanes;             // per patch
  int seg, col;          // patch of the task, 1-based interior column
  bool segok, active;
};

__device__ __forceinline__ SegLane seg_lane(const SegList& A, int wave) {
  SegLane g;
  const int lane = threadIdx.x & 63;
  g.recs = A.recs + (long long)wave * A.group;
  g.ra = gl(&g.recs->r0);
  g.rb = gl(&g.recs->r1);
  g.sidx = gl(&g.recs->sidx);
  g.nseg = gl(&g.recs->nseg);
  g.nx = gl(&g.recs->d.nx);
  g.ny = gl(&g.recs->d.ny);
  g.rows = g.rb - g.ra + 1;
  g.lanes = A.lanes ? A.lanes : pow2ceil(g.ny);
  g.seg = lane / g.lanes;
  g.col = lane - g.seg * g.lanes + 1;
  g.segok = g.seg < g.nseg;
  g.active = g.segok && g.col <= g.ny;
  return g;
}

// The lane's patch (read without waiting for the wavefront's record: its
// place needs the number of lanes only).
__device__ __forceinline__ SegDesc seg_desc(const SegList& A, const SegLane& g) {
  return gl(&(g.recs + (g.seg < A.group ? g.seg : 0))->d);
}

// This thread's wavefront among those of the launch's workgroups, uniform.
__device__ __forceinline__ int seg_wave(int waves) {
  return __builtin_amdgcn_readfirstlane((int)blockIdx.x * waves + (int)(threadIdx.x >> 6));
}

// h, hu, hv of one state.
struct State {
  const double *h, *hu, *hv;
};
__device__ __forceinline__ State state_of(const Fields& F, int s) {
  return State{F.H(s), F.HU(s), F.HV(s)};
}

// Cells of rows ra-1 .. ra+R of the lane's column (rows past `last` and lanes
// without a cell: a wet cell at rest).  hv of a ghost row is not used.
// Interior and ghost rows can be loaded apart, the ghosts from another state.
enum RowPart { kRowsInterior = 1, kRowsGhost = 2, kRowsAll = 3 };
template <int R, bool B>
struct SegRows {
  double h[R + 2], hu[R + 2], hv[R + 2], b[R + 2];
  template <int PART>
  __device__ __forceinline__ void load(const SegDesc& D, const SegLane& g, const State& S,
                                       const double* Bf, int last) {
#pragma unroll
    for (int k = 0; k < R + 2; ++k) {
      const int r = g.ra - 1 + k;
      const bool ghost = r == 0 || r == D.nx + 1;
      if (PART & kRowsInterior) {
        h[k] = 1.0; hu[k] = 0.0; hv[k] = 0.0; b[k] = 0.0;
      }
      if (!g.active || r > last) continue;
      const long long i = D.off + (long long)r * D.stride + g.col;
      const long long j = r == 0 ? D.gx[0] + g.col : (r == D.nx + 1 ? D.gx[1] + g.col : i);
      if ((PART & kRowsInterior) && B) b[k] = gl(Bf + i);
      if (PART == kRowsInterior && ghost) continue;
      if (PART == kRowsGhost && !ghost) continue;
      h[k] = gl(S.h + j);
      hu[k] = gl(S.hu + j);
      hv[k] = gl(S.hv + j);
    }
    if (PART & kRowsGhost) {
#pragma unroll
      for (int k = 0; k < R + 2; ++k) {
        const int r = g.ra - 1 + k;
        if ((r == 0 && (D.neg & 1)) || (r == D.nx + 1 && (D.neg & 2))) hu[k] = -hu[k];
      }
    }
  }
};

// The y-edges that touch the ghost columns, two per row and patch, one per
// lane: entry e is side e & 1 of row ra + (e >> 1) % rows of patch
// (e >> 1) / rows.  Own cells and ghosts may come from two states.
struct SegSide {
  int slot, side;
  double hL, hvL, bL, hR, hvR, bR, dyinv;
  template <bool B>
  __device__ __forceinline__ void load(const SegLane& g, int e, const State& S,
                                       const State& G, const double* Bf) {
    side = e & 1;
    const int s = (e >> 1) / g.rows;
    const int row = g.ra + (e >> 1) - s * g.rows;
    slot = e >> 1;
    const SegDesc Q = gl(&(g.recs + s)->d);
    dyinv = Q.dyinv;
    const long long at = Q.off + (long long)row * Q.stride;
    const long long io = at + (side ? Q.ny : 1);
    const long long ig = (side ? Q.gy[1] : Q.gy[0]) + (long long)row * Q.stride;
    const double ho = gl(S.h + io), hvo = gl(S.hv + io);
    double hg = gl(G.h + ig), hvg = gl(G.hv + ig);
    if (Q.neg & (side ? 8 : 4)) hvg = -hvg;
    const double bo = B ? gl(Bf + io) : 0.0;
    const double bg = B ? gl(Bf + at + (side ? Q.ny + 1 : 0)) : 0.0;
    hL = side ? ho : hg; hvL = side ? hvo : hvg; bL = side ? bo : bg;
    hR = side ? hg : ho; hvR = side ? hvg : hvo; bR = side ? bg : bo;
  }
};

// Largest speed of the segment's edges per patch, in every lane of the
// patch.  `pre`: this wavefront's LDS.  The edge below the last row belongs
// to the next segment (`last`: the last row loaded).
template <int R, int SOLVER, class Rows>
__device__ __forceinline__ double seg_speeds(const SegLane& g,
                                             const Rows& q, int last,
                                             const State& S, const State& G, const double* Bf,
                                             double (*pre)[64]) {
  using ES = EdgeSolver<SOLVER>;
  constexpr bool B = SOLVER != 0;  // the f-wave's speeds do not depend on b
  const int npre = g.nseg * g.rows * 2;
  for (int e = threadIdx.x & 63; e < npre; e += 64) {
    SegSide s;
    s.load<B>(g, e, S, G, Bf);
    const CellQ cl = cell_dir(cell_base(s.hL, s.bL), s.hvL);
    const CellQ cr = cell_dir(cell_base(s.hR, s.bR), s.hvR);
    pre[s.side][s.slot] = ES::speed(cl, cr);
  }
  CellBase cb[R + 2];
  CellQ cx[R + 2];
  bool wet = true;
#pragma unroll
  for (int k = 0; k < R + 2; ++k) {
    cb[k] = cell_base(q.h[k], q.b[k]);
    cx[k] = cell_dir(cb[k], q.hu[k]);
    wet = wet && q.h[k] >= kDryTol;
  }
  double sm = 0.0;
  if (SOLVER == 0 && wave_all(wet)) {
#pragma unroll
    for (int k = 1; k < R + 2; ++k) {
      const double sx = edge_speed_wet(cx[k - 1], cx[k]);
      if (g.ra - 1 + k <= last) sm = dmax(sm, sx);
      if (k > R) break;
      const CellQ cy = cell_dir(cb[k], q.hv[k]);
      const double sy = edge_speed_wet(left_cell(cy), cy);
      if (g.col >= 2 && k <= g.rows) sm = dmax(sm, sy);
    }
  } else {
#pragma unroll
    for (int k = 1; k < R + 2; ++k) {
      if (g.ra - 1 + k <= last) sm = dmax(sm, ES::speed(cx[k - 1], cx[k]));
      if (k > R || k > g.rows) continue;
      const CellQ cy = cell_dir(cb[k], q.hv[k]);
      const double sy = ES::speed(left_cell(cy), cy);
      if (g.col >= 2) sm = dmax(sm, sy);
    }
  }
  wave_sync();
  if (g.active && (g.col == 1 || g.col == g.ny))
    for (int k = 0; k < g.rows; ++k) {
      if (g.col == 1) sm = dmax(sm, pre[0][g.seg * g.rows + k]);
      if (g.col == g.ny) sm = dmax(sm, pre[1][g.seg * g.rows + k]);
    }
  double v = g.active ? sm : 0.0;
  for (int m = g.lanes >> 1; m >= 1; m >>= 1) v = dmax(v, __shfl_xor(v, m));
  return v;
}

// Shares of the segment's ghost-column y-edges, into this wavefront's LDS.
template <int SOLVER>
__device__ __forceinline__ void seg_side_shares(const SegLane& g, const State& S,
                                                const double* Bf, double (*pre)[64]) {
  const int npre = g.nseg * g.rows * 2;
  for (int e = threadIdx.x & 63; e < npre; e += 64) {
    SegSide s;
    s.load<true>(g, e, S, S, Bf);
    const CellQ cl = cell_dir(cell_base(s.hL, s.bL), s.hvL);
    const CellQ cr = cell_dir(cell_base(s.hR, s.bR), s.hvR);
    double dhL, dhR, dqL, dqR;
    EdgeSolver<SOLVER>::solve(cl, cr, dhL, dhR, dqL, dqR);
    // side 0: the right cell (row,1) takes the "upwards" part;
    // side 1: the left cell (row,ny) takes the "downwards" part.
    pre[s.side * 2 + 0][s.slot] = s.dyinv * (s.side ? dhL : dhR);
    pre[s.side * 2 + 1][s.slot] = s.dyinv * (s.side ? dqL : dqR);
  }
}

// Update of the segment's rows by dt, written to (Hd, HUd, HVd); `pre` holds
// seg_side_shares.
template <int R, int SOLVER>
__device__ __forceinline__ void seg_update_rows(const SegLane& g, const SegDesc& D,
                                                const SegRows<R, true>& q,
                                                double dt, double (*pre)[64],
                                                double* __restrict__ Hd,
                                                double* __restrict__ HUd,
                                                double* __restrict__ HVd) {
  using ES = EdgeSolver<SOLVER>;
  bool wet = true;
#pragma unroll
  for (int k = 0; k < R + 2; ++k) wet = wet && q.h[k] >= kDryTol;
  const bool fast = SOLVER == 0 && wave_all(wet);
  const unsigned long long col1 = __builtin_amdgcn_ballot_w64(g.col == 1);
  const double dxinv = D.dxinv, dyinv = D.dyinv;
  // Chunks of rows: the edges below the chunk's rows (x-edge k | k+1, y-edges
  // of row k+1) in straight-line code, one vote, then the rows they complete.
  // Few rows go in one chunk (most overlap); with more, two by two, for the
  // registers.
  constexpr int C = R <= 2 ? R + 1 : 1;
  CellBase cb = cell_base(q.h[0], q.b[0]);
  CellQ cx = cell_dir(cb, q.hu[0]);
  double accH = 0.0, accHu = 0.0, uph = 0.0, upq = 0.0, dnh = 0.0, dnq = 0.0;
#pragma unroll
  for (int k0 = 0; k0 <= R; k0 += C) {
    if (k0 > g.rows) break;
    double xhL[C], xhR[C], xqL[C], xqR[C], yhL[C], yhR[C], yqL[C], yqR[C];
    if (fast) {
      WetEdge ex[C], ey[C];
      bool sub = true, suby = true;
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const int k = k0 + c;
        const CellBase nb = cell_base(q.h[k + 1], q.b[k + 1]);
        const CellQ nx = cell_dir(nb, q.hu[k + 1]);
        ex[c] = wet_edge(cx, nx);
        sub = sub && ex[c].s1 < -kZeroTol && ex[c].s2 > kZeroTol;
        if (k < R) {
          const CellQ cy = cell_dir(nb, q.hv[k + 1]);
          ey[c] = wet_edge(left_cell(cy), cy);
          suby = suby && ey[c].s1 < -kZeroTol && ey[c].s2 > kZeroTol;
        }
        cx = nx;
      }
      const bool all = (__builtin_amdgcn_ballot_w64(sub) &
                        (__builtin_amdgcn_ballot_w64(suby) | col1)) ==
                       __builtin_amdgcn_read_exec();
#pragma unroll
      for (int c = 0; c < C; ++c) {
        wet_shares(ex[c], all, xhL[c], xhR[c], xqL[c], xqR[c]);
        if (k0 + c < R) wet_shares(ey[c], all, yhL[c], yhR[c], yqL[c], yqR[c]);
      }
    } else {
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const int k = k0 + c;
        xhL[c] = xhR[c] = xqL[c] = xqR[c] = 0.0;
        yhL[c] = yhR[c] = yqL[c] = yqR[c] = 0.0;
        if (k > g.rows) continue;
        const CellBase nb = cell_base(q.h[k + 1], q.b[k + 1]);
        const CellQ nx = cell_dir(nb, q.hu[k + 1]);
        ES::solve(cx, nx, xhL[c], xhR[c], xqL[c], xqR[c]);
        if (k < R) {
          const CellQ cy = cell_dir(nb, q.hv[k + 1]);
          ES::solve(left_cell(cy), cy, yhL[c], yhR[c], yqL[c], yqR[c]);
        }
        cx = nx;
      }
    }
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int k = k0 + c;
      if (k > g.rows) break;
      if (k >= 1) {
        // row k: x-left (in acc), x-right, y-up, y-down
        double nH = accH + dxinv * xhL[c];
        double nHu = accHu + dxinv * xqL[c];
        nH = nH + uph;
        nH = nH + dnh;
        double nHv = 0.0 + upq;
        nHv = nHv + dnq;
        double h1 = q.h[k] - dt * nH;
        double hu1 = q.hu[k] - dt * nHu;
        double hv1 = q.hv[k] - dt * nHv;
        if (h1 < kClampH) { hu1 = 0.0; hv1 = 0.0; }
        if (h1 < 0.0) h1 = 0.0;
        if (g.active) {
          const long long o = D.off + (long long)(g.ra - 1 + k) * D.stride + g.col;
          gs(Hd + o, h1);
          gs(HUd + o, hu1);
          gs(HVd + o, hv1);
        }
      }
      accH = 0.0 + dxinv * xhR[c];
      accHu = 0.0 + dxinv * xqR[c];
      if (k < R) {
        // shares of the y-edges of row k + 1; the lower neighbour's is
        // handed down one lane
        uph = dyinv * yhR[c];
        upq = dyinv * yqR[c];
        dnh = from_right(dyinv * yhL[c]);
        dnq = from_right(dyinv * yqL[c]);
        const int slot = g.seg * g.rows + k;
        if (k < g.rows && g.active && g.col == 1) {
          uph = pre[0][slot];
          upq = pre[1][slot];
        }
        if (k < g.rows && g.active && g.col == g.ny) {
          dnh = pre[2][slot];
          dnq = pre[3][slot];
        }
      }
    }
  }
}

// Minimum of v over the workgroup (every thread calls it), in thread 0.
__device__ __forceinline__ double block_min(double v, double* red) {
  for (int o = 32; o >= 1; o >>= 1) v = dmin(v, __shfl_xor(v, o));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0)
    for (int k = 1; k < (int)blockDim.x / 64; ++k) v = dmin(v, red[k]);
  return v;
}

// Exact edge speeds of the current state: one maximum per row segment in
// smax_seg[slot * kSegSlots + segment] (for the patches' own estimates), and
// per workgroup the smallest CFL step of its segments.  The CFL step falls
// with the speed, so the minimum over segments is the minimum over patches.
template <int R, int SOLVER>
__global__ void __launch_bounds__(64 * kSegWaves)
k_seg_speed(const SegRec* recs, const ScnDev* __restrict__ scn, int group, int lanes, int one,
            double* __restrict__ cfl_block, double* __restrict__ smax_seg, Fields F) {
  const SegList A{recs, group, lanes, one};
  __shared__ double pre[kSegWaves][2][64];
  __shared__ double red[kSegWaves];
  const int w = threadIdx.x >> 6;
  const SegLane g = seg_lane(A, seg_wave(kSegWaves));
  const SegDesc D = seg_desc(A, g);
  const int s = A.scn >= 0 ? A.scn : gl(&g.recs->d.scn);
  const State S = state_of(F, gl(&scn[s].stepc) & 1);
  const int last = g.rb == g.nx ? g.rb + 1 : g.rb;
  SegRows<R, SOLVER != 0> q;
  q.template load<kRowsAll>(D, g, S, F.b, last);
  const double v = seg_speeds<R, SOLVER>(g, q, last, S, S, F.b, pre[w]);
  if (g.segok && g.col == 1) gs(smax_seg + (long long)D.slot * kSegSlots + g.sidx, v);
  const double c = block_min(g.segok ? max_timestep(v, D.dx, D.dy) : kNoLimit, red);
  if (threadIdx.x == 0) gs(cfl_block + blockIdx.x, c);
}

// Every patch's own CFL step from its segments' speed maxima.
__global__ void __launch_bounds__(64)
k_seg_estimates(const SegDesc* __restrict__ desc, int n, int R,
                const double* __restrict__ smax_seg, double* __restrict__ est) {
  const int k = blockIdx.x * 64 + threadIdx.x;
  if (k >= n) return;
  const SegDesc D = gl(desc + k);
  double s = 0.0;
  for (int j = 0; j < seg_count(D.nx, R); ++j)
    s = dmax(s, gl(smax_seg + (long long)D.slot * kSegSlots + j));
  est[D.slot] = max_timestep(s, D.dx, D.dy);
}

// Blocks [first, last) of the segment kernels hold the tasks of a scenario.
struct SegRange {
  int first, last;
};

// This thread's share of a scenario's CFL step: the minimum over every
// `stride`-th of its blocks from the `at`-th on.
__device__ __forceinline__ double cfl_share(const SegRange& r,
                                            const double* __restrict__ cfl_block, int at,
                                            int stride) {
  double v = kNoLimit;
  for (int k = r.first + at; k < r.last; k += stride) v = dmin(v, gl(cfl_block + k));
  for (int o = 32; o >= 1; o >>= 1) v = dmin(v, __shfl_xor(v, o));
  return v;
}

// Workgroups at the end of the update's launch that advance the clocks, a
// wavefront per scenario: its chain of dependent loads (range, minima, clock)
// takes 2 us or more, so the scenarios' chains stand side by side.  Four at a
// time in one workgroup, a step of 128 scenarios (2 x 2 patches of 32^2 each)
// took 44.9 us, so 23.7 us; of 64: 23.6 us, so 16.8.
__host__ __device__ __forceinline__ int seg_clock_groups(int nscn) {
  return (nscn + kSegWaves - 1) / kSegWaves;
}

// The update of the same segments, current state -> other state.  Every
// workgroup takes its scenario's step from the blocks' minima and the clock
// `in`; the workgroups from `blocks` on (seg_clock_groups) advance the clocks of
// the scenarios into `out` (the next step's `in`), so no launch is needed between
// the speeds and the update.
template <int R, int SOLVER>
__global__ void __launch_bounds__(64 * kSegWaves)
__attribute__((amdgpu_waves_per_eu(R == 4 ? 3 : 2, 8)))
k_seg_update(const SegRec* recs, const ScnDev* __restrict__ in, int group, int lanes, int one,
             int nscn, int blocks, const SegRange* __restrict__ ranges, const double* __restrict__ cfl_block,
             ScnDev* __restrict__ out, Fields F) {
  const SegList A{recs, group, lanes, one};
  __shared__ double pre[kSegWaves][4][64];
  __shared__ double red[kSegWaves];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if ((int)blockIdx.x >= blocks) {
    const int s = ((int)blockIdx.x - blocks) * kSegWaves + w;
    if (s >= nscn) return;
    const double cfl = cfl_share(gl(ranges + s), cfl_block, lane, 64);
    if (lane == 0) {
      ScnDev S = in[s];
      dt_final_one(S, cfl, 0, nullptr, 1.0);
      out[s] = S;
    }
    return;
  }
  const SegLane g = seg_lane(A, seg_wave(kSegWaves));
  const SegDesc D = seg_desc(A, g);
  const int s = A.scn >= 0 ? A.scn : gl(&g.recs->d.scn);  // one per workgroup
  const ScnDev* C = in + s;
  const double max_dt = gl(&C->end_time) - (gl(&C->time) + gl(&C->dt));
  if (!(max_dt - 0.0 > kLaEps)) return;
  const int par = gl(&C->stepc) & 1;
  const State S = state_of(F, par);
  SegRows<R, true> q;
  q.template load<kRowsAll>(D, g, S, F.b, g.rb + 1);
  const double share = cfl_share(gl(ranges + s), cfl_block, (int)threadIdx.x,
                                 64 * kSegWaves);
  if (lane == 0) red[w] = share;
  seg_side_shares<SOLVER>(g, S, F.b, pre[w]);
  __syncthreads();
  double dt = max_dt;
  for (int k = 0; k < kSegWaves; ++k) dt = fmin(red[k], dt);
  if (g.nseg == 0) return;
  seg_update_rows<R, SOLVER>(g, D, q, dt, pre[w], F.H(1 - par), F.HU(1 - par),
                             F.HV(1 - par));
}

}  // namespace pcamd
