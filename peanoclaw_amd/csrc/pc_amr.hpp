// Batched step of an adaptive patch grid (included at the end of
// pc_abi.hip; uses the pool internals).
//
// The per-call form of a global AMR step is a long sequence of Numerics
// calls: restriction of every leaf into each virtual patch containing it
// (GridLevelTransfer::restrictToOverlappingVirtualSubgrids,
// GridLevelTransfer.cpp:140-198, with SWEKernel::restrictSolution and
// postProcessRestriction, SWEKernel.cpp:288-316), copyUNewToUOld of every
// leaf, a ghost-layer fill of every leaf face by transferGhostlayer from
// the same-level patch or interpolateSolution from the coarser leaf
// (GhostlayerCompositorFunctors.cpp:59-69; SWEKernel.cpp:239-286), walls
// (SolveTimestep.cpp:87-142), the global CFL minimum and solveTimestep of
// every leaf.  Here the host hands over that plan once (a device-side
// table rebuilt only when the grid changes) and every step is three
// launches over all patches at once:
//
//   restrict the contributions of the leaves covering every virtual-patch
//            cell, then h+b -> h
//   fill     one workgroup per task of leaves: uNew -> uOld, the ghost
//            layer of every face (copy with time factor, or d-linear
//            interpolation from the coarser leaf: h+b, back to h with the
//            destination's b), the walls in call order, then the exact edge
//            speeds of the leaves and the smallest CFL step of the workgroup
//   update   of every leaf, uOld -> uNew, with the smallest of those steps
//            bounded by the end time; one workgroup advances the clock
//
// (and a fourth between the last two where there are more than kCflFold
// workgroups' steps: k_cfl_fold).
//
// These grids hold a few hundred thousand cells, so latency bounds them: the
// fill loads a leaf's cells once for the copy and the speeds, and neither
// the copy, the walls nor the reduction of dt is a launch of its own.  The
// launches are issued one by one: graph launches left 5-8 us between steps.
// A workgroup's first loads (clock, task, records, ghost map) stand side by
// side and a ghost entry is read whole: a dependent load costs 0.7 to 0.9 us
// on the cold L2 a launch starts with.  Against checks and fields one behind
// the other: 67.8 -> 66.1 us a step of the 3-level grid of 729 27^2 leaves,
// 533 -> 516 us for 16 iterations of local time stepping on the 2-level grid.
//
// Every phase checks the step bound end_time - (time + dt); a step past the
// end time does nothing.
//
// The level transfers read h + b instead of transforming the source in
// place and back: the reference's round trip (h + b) - b can move a depth
// by one ulp, which the per-call entry points reproduce and this form does
// not (results agree to ~1e-14 relative; both are checked against the
// oracle's matching drivers).  Every other operation is the per-call
// arithmetic in the same order.
#pragma once

#include <unordered_map>

#include "pc_seg_kernels.hpp"

namespace {

struct AmrClock {
  double time, dt;  // the leaves' clock (time, timestep_size)
  double end_time;
  double bound;     // dt of the step being run
  int advance;      // the last step ran
  int pad;
  long long steps;
};

// end_time - (time + dt) > tolerance (AMR driver's step condition)
__device__ __forceinline__ bool amr_advance(const AmrClock& c) {
  const double maxdt = c.end_time - (c.time + c.dt);
  return maxdt - 0.0 > kLaEps;
}

// Local time stepping: per-slot clocks of the leaves (indexed by slot id).
struct AmrLts {
  double* t;        // time (start of the current interval)
  double* dt;       // timestep size
  int* adv;         // the leaf advances in this iteration
  double* stepdt;   // the step an advancing leaf takes
  int* iter;        // leaves advancing in this iteration
  unsigned long long* steps;  // leaf steps taken
  int* itn;         // iteration number
  int* need;        // virtual patch: iteration in which an advancing leaf reads it
};

// Gate of a phase: global steps run while the shared clock may advance;
// local time stepping while some leaf advances in this iteration.
template <bool LTS>
__device__ __forceinline__ bool amr_phase_runs(const AmrClock* clock, const AmrLts& L) {
  if (LTS) return *L.iter > 0;
  return amr_advance(*clock);
}

// The restriction kernel's lanes per virtual-patch cell, cells per workgroup
// (one AmrVBlock) and contributions per cell held in LDS at a time.
constexpr int kRestrictLanes = 16;
constexpr int kRestrictCells = 256 / kRestrictLanes;
constexpr int kRestrictChunk = 2 * kRestrictLanes;

// kRestrictCells consecutive cells of one virtual patch
struct AmrVBlock {
  long long off;     // its tile
  double dstRegion;  // area of its cells
  int slot;
  int cell0;  // first cell (x * ny + y)
  int base;   // index of cell 0 of this patch in the per-cell lists
  int nx, ny, stride;
};

// One fine cell of a leaf inside a virtual-patch cell: where it is
// (kContribBits bits: index in the field arrays; above: the leaf's place in
// the plan) and the area they share.
constexpr int kContribBits = 40;
struct AmrContrib {
  unsigned long long at;
  double region;
};

// Restriction of the whole leaf `src` into one virtual patch
// (DefaultRestriction.cpph:16-106 over region (0, n)).
struct AmrRestrict {
  int src, leaf;  // slot, place in the plan's leaves
  int rSize[2];
  int dOff[2], dSize[2];
  double srcSub[2], dstSub[2], dstRegion;
  double spos[2], dpos[2];
};

enum AmrGhostKind { kAmrTransferLeaf = 0, kAmrTransferVirtual = 1, kAmrInterpolate = 2 };

struct AmrGhost {
  int kind, src, dst;
  int sx, sy, sox, soy, dox, doy;
  int sn[2];
  int cell0;  // its first cell among the ghost cells of its task's leaves
  // tile rows: first cell of the source region (interpolation: cell (0, 0)
  // of the source), first cell of the destination region
  long long sbase, dbase;
  int sstride, dstride;
  double spos[2], ssub[2], sinv[2], dpos[2], dsub[2];
};

// walls[first .. first + count) of a leaf as (dim, upper) pairs
struct AmrWalls {
  int first, count;
};

// One task of leaves in the fill (workgroup b): its row segments are
// wavefronts [b max_waves, + nwaves) of the plan's records, its ghost cells'
// entries gmap[b max_cells .. + max_cells) (-1: none).
struct AmrBlock {
  int nwaves, leaf0, nseg;  // leaf0: place of its first leaf in task order
  int nx, ny;
  int nwalls;  // most walls of one of its leaves
  int pad[2];
};

// Restriction time factors of a leaf source on the [0, 1] basis
// (DefaultRestriction.cpph:46-52).
__device__ __forceinline__ void amr_restrict_factors(const AmrClock& c, double& tfOld,
                                                     double& tfNew) {
  tfOld = 1.0;
  tfNew = 1.0;
  if (c.dt - 0.0 > kLaEps) {
    const double sOld = c.time, sNew = c.time + c.dt;
    tfOld = (0.0 - sOld) / (sNew - sOld);
    tfNew = (1.0 - sOld) / (sNew - sOld);
  }
}

// Fine cells of a leaf under row (d = 0) or column (d = 1) `di` of a virtual
// patch: [o, o + n) (DefaultRestriction.cpph:60-83).
__host__ __device__ __forceinline__ void amr_fine_span(const AmrRestrict& a, int d, int di,
                                                       int& o, int& n) {
  const double eps = 1e-12;
  const double dp = a.dpos[d] + (double)di * a.dstSub[d];
  double ot = (dp - a.spos[d] + eps);
  ot /= a.srcSub[d];
  const int first = (int)ot;
  double st = dp + a.dstSub[d] - a.spos[d] - eps;
  st /= a.srcSub[d];
  st -= ot;
  st += 1.0;
  const int upper = first + (int)st, rUpper = a.rSize[d];
  o = first > 0 ? first : 0;
  n = (upper < rUpper ? upper : rUpper) - o;
  if (n < 0) n = 0;
}

// Area that cell (s0, s1) of the leaf shares with the virtual patch's cell
// whose lower corner is dp.
__device__ __forceinline__ double amr_shared_area(const AmrRestrict& a, const double* dp, int s0,
                                                  int s1) {
  const double sp[2] = {a.spos[0] + (double)s0 * a.srcSub[0],
                        a.spos[1] + (double)s1 * a.srcSub[1]};
  double region = 1.0;
  for (int d = 0; d < 2; ++d) {
    const double hi = dmin(dp[d] + a.dstSub[d], sp[d] + a.srcSub[d]);
    const double lo = dmax(dp[d], sp[d]);
    region *= hi - lo;
    region = dmax(region, 0.0);
  }
  return region;
}

// The plan's contributions, one thread per virtual-patch cell, in the order
// of the per-call sequence (pairs in plan order, fine cells x outer, y
// inner): contribs[xptr[cell] ..].  Runs once per plan.  `cptr`/`cpairs`
// list, per cell, the restriction pairs whose destination region holds it.
__global__ void __launch_bounds__(256)
k_amr_contribs(const AmrVBlock* __restrict__ blocks, const int* __restrict__ cptr,
               const int* __restrict__ cpairs, const int* __restrict__ xptr,
               const AmrRestrict* __restrict__ pairs, const PatchDev* __restrict__ pd,
               AmrContrib* __restrict__ contribs) {
  const AmrVBlock B = blocks[blockIdx.x * (256 / kRestrictCells) + threadIdx.x / kRestrictCells];
  const int k = B.cell0 + (int)threadIdx.x % kRestrictCells;
  if (k >= B.nx * B.ny) return;
  const int d0 = k / B.ny, d1 = k - d0 * B.ny;
  AmrContrib* out = contribs + xptr[B.base + k];
  for (int j = cptr[B.base + k]; j < cptr[B.base + k + 1]; ++j) {
    const AmrRestrict& a = pairs[cpairs[j]];
    const PatchDev S = pd[a.src];
    const double dp[2] = {a.dpos[0] + (double)d0 * a.dstSub[0],
                          a.dpos[1] + (double)d1 * a.dstSub[1]};
    int o[2], n[2];
    amr_fine_span(a, 0, d0, o[0], n[0]);
    amr_fine_span(a, 1, d1, o[1], n[1]);
    for (int x = 0; x < n[0]; ++x)
      for (int y = 0; y < n[1]; ++y) {
        out->at = (unsigned long long)tile_index(S, o[0] + x, o[1] + y) |
                  ((unsigned long long)a.leaf << kContribBits);
        out->region = amr_shared_area(a, dp, o[0] + x, o[1] + y);
        ++out;
      }
  }
}

// Restriction (DefaultRestriction.cpph:16-106, SWEKernel::
// postProcessRestriction): kRestrictLanes lanes per virtual-patch cell take
// its contributions in turn; lane q < 6 sums one of the six quantities (h +
// b, hu, hv in both states) in the order of the per-call sequence, so the
// sums equal the sequential ones bit for bit.
//
// Bound by latency: geometry, source cells and shared areas come from the
// plan's contribution list (16 bytes each), so a cell's chain is block ->
// list bounds -> list -> cells; deriving them per step, behind four
// divisions and five more dependent loads, took 15.7 us on the 2-level grid
// of 1129 16^2 leaves and 24.8 us on the 3-level grid of 729 27^2 leaves, so
// 6.3 and 18.0 us.  On the latter its bytes bound it (about 0.95 M
// contributions of 72 bytes): loading them two rounds ahead gave nothing.
template <bool LTS>
__global__ void __launch_bounds__(256)
k_amr_restrict(const AmrVBlock* __restrict__ blocks, const int* __restrict__ xptr,
               const AmrContrib* __restrict__ contribs, const int* __restrict__ leaves,
               Fields F, int cur, const AmrClock* clock, AmrLts L) {
  constexpr int K = kRestrictLanes, N = kRestrictChunk;
  __shared__ double con[kRestrictCells][6][N + 1];
  const AmrClock c = *clock;
  const AmrVBlock B = blocks[blockIdx.x];
  const int g = (int)threadIdx.x / K, sub = (int)threadIdx.x - g * K;
  const int k = B.cell0 + g;
  const bool cellok = k < B.nx * B.ny;
  const int beg = cellok ? gl(xptr + B.base + k) : 0;
  const int n = cellok ? gl(xptr + B.base + k + 1) - beg : 0;
  if (!amr_phase_runs<LTS>(clock, L)) return;
  // local time stepping: only the virtual patches an advancing leaf reads
  if (LTS && L.need[B.slot] != *L.itn) return;
  double tfOld, tfNew;
  amr_restrict_factors(c, tfOld, tfNew);
  const State O = state_of(F, 1 - cur), W = state_of(F, cur);
  int most = n;  // of the wavefront's cells
  for (int o = 32; o >= K; o >>= 1) most = max(most, __shfl_xor(most, o));
  double acc = 0.0;
  for (int r0 = 0; r0 < most; r0 += N) {
#pragma unroll
    for (int half = 0; half < N; half += K) {
      const int m = r0 + half + sub;
      if (m >= n) continue;
      const AmrContrib a = gl(contribs + beg + m);
      const long long i = (long long)(a.at & ((1ull << kContribBits) - 1));
      if (LTS) {
        // each leaf restricts on its own interval
        const int s = gl(leaves + (a.at >> kContribBits));
        AmrClock cs = c;
        cs.time = L.t[s];
        cs.dt = L.dt[s];
        amr_restrict_factors(cs, tfOld, tfNew);
      }
      const double bv = gl(F.b + i);
      const double vo[3] = {gl(O.h + i) + 1.0 * bv, gl(O.hu + i), gl(O.hv + i)};
      const double vn[3] = {gl(W.h + i) + 1.0 * bv, gl(W.hu + i), gl(W.hv + i)};
      for (int q = 0; q < 3; ++q) {
        con[g][q][half + sub] =
            (vo[q] * (1.0 - tfOld) + vn[q] * tfOld) * a.region / B.dstRegion;
        con[g][3 + q][half + sub] =
            (vo[q] * (1.0 - tfNew) + vn[q] * tfNew) * a.region / B.dstRegion;
      }
    }
    wave_sync();
    if (sub < 6) {
      const int cnt = n - r0 < N ? n - r0 : N;
      for (int i = 0; i < cnt; ++i) acc = acc + con[g][sub][i];
    }
    wave_sync();
  }
  if (!cellok || sub >= 6) return;
  const int x = k / B.ny, y = k - x * B.ny;
  const long long di = B.off + (long long)(x + 1) * B.stride + (y + 1);
  const int q = sub % 3, st = sub < 3 ? 1 - cur : cur;
  // h + b -> h with the virtual patch's b
  if (q == 0)
    gs(F.H(st) + di, acc + (-1.0) * gl(F.b + di));
  else
    gs((q == 1 ? F.HU(st) : F.HV(st)) + di, acc);
}

// The same for plans without a contribution list (amr_list_fits): every lane
// derives its fine cell and their shared area from the cell's pairs.
template <bool LTS>
__global__ void __launch_bounds__(256)
k_amr_restrict_pairs(const AmrVBlock* __restrict__ blocks, const int* __restrict__ cptr,
                     const int* __restrict__ cpairs, const AmrRestrict* __restrict__ pairs,
                     const PatchDev* __restrict__ pd, Fields F, int cur, const AmrClock* clock,
                     AmrLts L) {
  constexpr int K = kRestrictLanes;
  __shared__ double con[kRestrictCells][6][K + 1];
  const AmrClock c = *clock;
  const AmrVBlock B = blocks[blockIdx.x];
  const int g = (int)threadIdx.x / K, sub = (int)threadIdx.x - g * K;
  const int k = B.cell0 + g;
  const bool cellok = k < B.nx * B.ny;
  if (!amr_phase_runs<LTS>(clock, L)) return;
  if (LTS && L.need[B.slot] != *L.itn) return;
  double tfOld, tfNew;
  amr_restrict_factors(c, tfOld, tfNew);
  const State O = state_of(F, 1 - cur), W = state_of(F, cur);
  const int d0 = cellok ? k / B.ny : 0, d1 = cellok ? k - d0 * B.ny : 0;
  const int jb = cellok ? cptr[B.base + k] : 0, je = cellok ? cptr[B.base + k + 1] : 0;
  double acc = 0.0;
  for (int j = jb; j < je; ++j) {  // the same for the lanes of a cell
    const AmrRestrict a = pairs[cpairs[j]];
    const PatchDev S = pd[a.src];
    if (LTS) {
      // each leaf restricts on its own interval
      AmrClock cs = c;
      cs.time = L.t[a.src];
      cs.dt = L.dt[a.src];
      amr_restrict_factors(cs, tfOld, tfNew);
    }
    const double dp[2] = {a.dpos[0] + (double)d0 * a.dstSub[0],
                          a.dpos[1] + (double)d1 * a.dstSub[1]};
    int o[2], n[2];
    amr_fine_span(a, 0, d0, o[0], n[0]);
    amr_fine_span(a, 1, d1, o[1], n[1]);
    const int nfine = n[0] * n[1];
    for (int r0 = 0; r0 < nfine; r0 += K) {
      const int m = r0 + sub;
      if (m < nfine) {
        const int s0 = o[0] + m / n[1], s1 = o[1] + m % n[1];
        const long long i = tile_index(S, s0, s1);
        const double region = amr_shared_area(a, dp, s0, s1), bv = gl(F.b + i);
        const double vo[3] = {gl(O.h + i) + 1.0 * bv, gl(O.hu + i), gl(O.hv + i)};
        const double vn[3] = {gl(W.h + i) + 1.0 * bv, gl(W.hu + i), gl(W.hv + i)};
        for (int q = 0; q < 3; ++q) {
          con[g][q][sub] = (vo[q] * (1.0 - tfOld) + vn[q] * tfOld) * region / B.dstRegion;
          con[g][3 + q][sub] = (vo[q] * (1.0 - tfNew) + vn[q] * tfNew) * region / B.dstRegion;
        }
      }
      wave_sync();
      if (sub < 6) {
        const int cnt = nfine - r0 < K ? nfine - r0 : K;
        for (int i = 0; i < cnt; ++i) acc = acc + con[g][sub][i];
      }
      wave_sync();
    }
  }
  if (!cellok || sub >= 6) return;
  const long long di = B.off + (long long)(d0 + 1) * B.stride + (d1 + 1);
  const int q = sub % 3, st = sub < 3 ? 1 - cur : cur;
  if (q == 0)
    gs(F.H(st) + di, acc + (-1.0) * gl(F.b + di));
  else
    gs((q == 1 ? F.HU(st) : F.HV(st)) + di, acc);
}

// Cell k of a ghost entry.  LTS: every leaf runs on its own clock, and only
// an advancing one's ghosts are written.  Else all leaves run on (time, dt),
// and a leaf's uOld is its uNew (copied in the same launch, so not read here).
// The entry comes in registers: its fields' loads are one level of the chain.
template <bool LTS>
__device__ __forceinline__ void amr_ghost_cell(const AmrGhost g, int k,
                                               const Fields& F, int cur, const AmrClock& c,
                                               const AmrLts& L) {
  const int oldSt = 1 - cur;
  const int kind = g.kind;
  const bool go = !LTS || L.adv[g.dst] != 0;
  const double dTime = LTS ? L.t[g.dst] : c.time, dDt = LTS ? L.dt[g.dst] : c.dt;
  const double sTime = (LTS && kind != kAmrTransferVirtual) ? L.t[g.src] : c.time;
  const double sDt = (LTS && kind != kAmrTransferVirtual) ? L.dt[g.src] : c.dt;
  const double dstTimeUNew = dTime + dDt;
  const int x = k / g.sy, y = k - (k / g.sy) * g.sy;
  const long long di = g.dbase + (long long)x * g.dstride + y;
  const int srcOld = LTS || kind == kAmrTransferVirtual ? oldSt : cur;
  if (kind != kAmrInterpolate) {
    // DefaultTransfer.cpph:27-51
    double tf;
    if (kind == kAmrTransferVirtual) {
      tf = (dstTimeUNew - 0.0) / 1.0;
    } else {
      const double sNew = sTime + sDt, sOld = sTime;
      tf = (sNew - sOld - 0.0 > kLaEps) ? (dstTimeUNew - sOld) / (sNew - sOld) : 1.0;
    }
    const double inv = 1.0 - tf;
    const long long si = g.sbase + (long long)x * g.sstride + y;
    const double h = F.H(cur)[si] * tf + F.H(srcOld)[si] * inv;
    const double hu = F.HU(cur)[si] * tf + F.HU(srcOld)[si] * inv;
    const double hv = F.HV(cur)[si] * tf + F.HV(srcOld)[si] * inv;
    if (!go) return;
    F.H(oldSt)[di] = h;
    F.HU(oldSt)[di] = hu;
    F.HV(oldSt)[di] = hv;
    return;
  }
  // DefaultInterpolation.cpph:45-67 (toCurrentTime = 0, useTimeUNewOrUOld = 1)
  double tf;
  if (fabs(sDt - 0.0) <= kLaEps) {
    tf = 1.0;
  } else {
    const double sOld = sTime, sNew = sTime + sDt;
    tf = (dstTimeUNew - sOld) / (sNew - sOld);
  }
  tf = dmax(0.0, dmin(1.0, tf));
  const double bd = F.b[di];
  double acc[3] = {0.0, 0.0, 0.0};
  double cc[2];
  cc[0] = g.dpos[0] + g.dsub[0] * (double)(g.dox + x) + g.dsub[0] * 0.5;
  cc[1] = g.dpos[1] + g.dsub[1] * (double)(g.doy + y) + g.dsub[1] * 0.5;
  int si[2];
  for (int d = 0; d < 2; ++d) {
    const double base = g.spos[d] + g.ssub[d] * 0.5;
    const double loc = cc[d] - base;
    int v = (int)floor(loc * g.sinv[d]);
    v = v < g.sn[d] - 2 ? v : g.sn[d] - 2;
    v = v > 0 ? v : 0;
    si[d] = v;
  }
  for (int o = 0; o < 4; ++o) {
    const int off[2] = {o & 1, (o >> 1) & 1};
    const int nb[2] = {si[0] + off[0], si[1] + off[1]};
    double np[2];
    np[0] = g.spos[0] + g.ssub[0] * (double)nb[0] + g.ssub[0] * 0.5;
    np[1] = g.spos[1] + g.ssub[1] * (double)nb[1] + g.ssub[1] * 0.5;
    double sf = 1.0;
    for (int d = 0; d < 2; ++d) {
      const double sign = (double)(1 - 2 * off[d]);
      sf *= 1.0 - (sign * (cc[d] - np[d])) * g.sinv[d];
    }
    const long long sidx = g.sbase + (long long)nb[0] * g.sstride + nb[1];
    const double bv = F.b[sidx];
    const double vo[3] = {F.H(srcOld)[sidx] + 1.0 * bv, F.HU(srcOld)[sidx], F.HV(srcOld)[sidx]};
    const double vn[3] = {F.H(cur)[sidx] + 1.0 * bv, F.HU(cur)[sidx], F.HV(cur)[sidx]};
    for (int q = 0; q < 3; ++q) acc[q] = acc[q] + sf * (vo[q] * (1.0 - tf) + vn[q] * tf);
  }
  if (!go) return;
  F.H(oldSt)[di] = acc[0] + (-1.0) * bd;
  F.HU(oldSt)[di] = acc[1];
  F.HV(oldSt)[di] = acc[2];
}

// The plan's ghost map (-1 where no entry writes one): every entry's cells, a
// wavefront per entry; task: the entries' tasks.  Runs once per plan.
__global__ void __launch_bounds__(256)
k_amr_ghost_map(const AmrGhost* __restrict__ ghosts, const int* __restrict__ task, int n,
                int max_cells, int* __restrict__ gmap) {
  const int e = blockIdx.x * 4 + (int)(threadIdx.x >> 6);
  if (e >= n) return;
  const int cells = ghosts[e].sx * ghosts[e].sy;
  int* const out = gmap + (long long)task[e] * max_cells + ghosts[e].cell0;
  for (int k = threadIdx.x & 63; k < cells; k += 64) out[k] = e;
}

// Local time stepping: the ghost cells of the advancing leaves, before any
// leaf changes (one thread per ghost cell of the plan).
__global__ void __launch_bounds__(256)
k_lts_ghosts(const int* __restrict__ gmap, int max_cells, int ncells,
             const AmrGhost* __restrict__ ghosts, Fields F, int cur, const AmrClock* clock,
             AmrLts L) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= ncells) return;
  const int e = gl(gmap + c), advancing = gl(L.iter);
  const AmrClock now = gl(clock);
  if (e < 0 || advancing == 0) return;
  const AmrGhost g = gl(ghosts + e);
  amr_ghost_cell<true>(g, c % max_cells - g.cell0, F, cur, now, L);
}

// SWEKernel::fillBoundaryLayer (SWEKernel.cpp:176-237) of the leaves of a
// task, their walls in call order (corner cells read what the previous wall
// wrote); `adv` null: all of them.
__device__ __forceinline__ void amr_walls(const AmrBlock& K, const SegRec* __restrict__ recs,
                                          const AmrWalls* __restrict__ walls,
                                          const int* __restrict__ dims, const Fields& F, int st,
                                          const int* adv) {
  const int len = (K.nx > K.ny ? K.nx : K.ny) + 2;
  for (int w = 0; w < K.nwalls; ++w) {
    for (int i = threadIdx.x; i < K.nseg * len; i += blockDim.x) {
      const int s = i / len, k = i - s * len - 1;
      const AmrWalls W = walls[K.leaf0 + s];
      if (w >= W.count) continue;
      const int dim = dims[2 * (W.first + w)], upper = dims[2 * (W.first + w) + 1];
      const SegDesc P = recs[s].d;
      if (k >= (dim == 0 ? P.ny : P.nx) + 1 || (adv && !adv[P.slot])) continue;
      int dx, dy, sx, sy;
      if (dim == 0) {
        dx = upper ? P.nx : -1;
        sx = dx + (upper ? -1 : 1);
        dy = sy = k;
      } else {
        dy = upper ? P.ny : -1;
        sy = dy + (upper ? -1 : 1);
        dx = sx = k;
      }
      const long long d = P.off + (long long)(dx + 1) * P.stride + (dy + 1);
      const long long q = P.off + (long long)(sx + 1) * P.stride + (sy + 1);
      const double h = F.H(st)[q], hu = F.HU(st)[q], hv = F.HV(st)[q];
      F.H(st)[d] = h;
      F.HU(st)[d] = dim == 0 ? -hu : hu;
      F.HV(st)[d] = dim == 1 ? -hv : hv;
    }
    __syncthreads();
  }
}

// After a call's iterations of local time stepping: the leaves' clocks and
// the leaf steps taken, into pinned host memory (time and step of leaf k at
// host[2 k + 1]; the count, reset here, at host[0]).
__global__ void __launch_bounds__(256)
k_lts_report(const int* __restrict__ leaves, int nleaves, AmrLts L, double* host) {
  const int k = blockIdx.x * 256 + threadIdx.x;
  if (k == 0) {
    *reinterpret_cast<unsigned long long*>(host) = *L.steps;
    *L.steps = 0;
  }
  if (k >= nleaves) return;
  host[2 * k + 1] = L.t[leaves[k]];
  host[2 * k + 2] = L.dt[leaves[k]];
}

// What the fill and the update read of the plan.
struct AmrPlanDev {
  SegList list;  // ghosts in the own tile
  int max_waves, max_cells;
  const AmrBlock* blocks;
  const int* gmap;
  const AmrGhost* ghosts;
  const AmrWalls* walls;  // per leaf in task order
  const int* dims;
};

// The fill of one task of leaves (see the top of this file), one wavefront
// per row segment.  Global steps: the workgroup's smallest CFL step goes to
// cfl_block.  Local time stepping: the leaves that advance only, their ghost
// cells filled before (k_lts_ghosts), and each leaf's step fmin(own CFL step,
// end - (t + dt)) (SWEKernel.cpp:60-68) to L.stepdt.
// MAXT: most threads of a workgroup (the register budget).
template <int R, int SOLVER, bool LTS, int MAXT>
__global__ void __launch_bounds__(MAXT)
__attribute__((amdgpu_waves_per_eu(4, 8)))
k_amr_fill(AmrPlanDev A, Fields F, int cur, const AmrClock* clock,
           double* __restrict__ cfl_block, AmrLts L) {
  __shared__ double pre[MAXT / 64][2][64];
  __shared__ double red[MAXT / 64];
  __shared__ double leaf_max[LTS ? MAXT / 64 : 1][64];
  // the first loads side by side: clock, task, records, ghost map
  const AmrClock c = gl(clock);
  const AmrBlock K = gl(A.blocks + blockIdx.x);
  const int* const gmap = A.gmap + (long long)blockIdx.x * A.max_cells;
  int ghost = -1;
  if (!LTS && (int)threadIdx.x < A.max_cells) ghost = gl(gmap + threadIdx.x);
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const SegRec* const recs = A.list.recs + (long long)blockIdx.x * A.max_waves * A.list.group;
  if (LTS && !amr_phase_runs<LTS>(clock, L)) return;
  if (LTS) {
    const bool go = lane < K.nseg && L.adv[recs[lane].d.slot] != 0;
    if (__builtin_amdgcn_ballot_w64(go) == 0) return;  // the same in every wavefront
  }
  SegLane g = seg_lane(A.list, seg_wave(A.max_waves));
  const SegDesc D = seg_desc(A.list, g);
  if (LTS && g.segok && !L.adv[D.slot]) g.active = false;
  if (!LTS && !amr_advance(c)) return;
  const State N = state_of(F, cur), O = state_of(F, 1 - cur);
  const int last = g.rb == g.nx ? g.rb + 1 : g.rb;
  SegRows<R, SOLVER != 0> q;
  q.template load<kRowsInterior>(D, g, N, F.b, last);
  if (!LTS)
    for (int i = threadIdx.x; i < A.max_cells; i += blockDim.x) {
      const int k = i == (int)threadIdx.x ? ghost : gl(gmap + i);
      if (k < 0) continue;
      const AmrGhost e = gl(A.ghosts + k);
      amr_ghost_cell<false>(e, i - e.cell0, F, cur, c, L);
    }
  // uNew -> uOld (DefaultTransfer::copyUNewToUOld)
#pragma unroll
  for (int k = 1; k <= R; ++k) {
    if (!g.active || k > g.rows) continue;
    const long long o = D.off + (long long)(g.ra - 1 + k) * D.stride + g.col;
    gs(F.H(1 - cur) + o, q.h[k]);
    gs(F.HU(1 - cur) + o, q.hu[k]);
    gs(F.HV(1 - cur) + o, q.hv[k]);
  }
  __syncthreads();
  amr_walls(K, recs, A.walls, A.dims, F, 1 - cur, LTS ? L.adv : nullptr);
  q.template load<kRowsGhost>(D, g, O, F.b, last);
  const double v = seg_speeds<R, SOLVER>(g, q, last, N, O, F.b, pre[w]);
  if (!LTS) {
    const double m = block_min(g.segok ? max_timestep(v, D.dx, D.dy) : kNoLimit, red);
    if (threadIdx.x == 0) gs(cfl_block + blockIdx.x, m);
    return;
  }
  if (g.segok && g.col == 1) leaf_max[w][g.seg] = v;
  __syncthreads();
  if ((int)threadIdx.x < K.nseg) {
    const SegDesc P = gl(&(recs + threadIdx.x)->d);
    if (L.adv[P.slot]) {
      double m = leaf_max[0][threadIdx.x];
      for (int k = 1; k < K.nwaves; ++k) m = dmax(m, leaf_max[k][threadIdx.x]);
      const double md = c.end_time - (L.t[P.slot] + L.dt[P.slot]);
      L.stepdt[P.slot] = fmin(max_timestep(m, P.dx, P.dy), md);
    }
  }
}

// Local time stepping of one task of leaves in one launch, where its row
// segments are at most 8 wavefronts (the register budget holds a wavefront's
// rows from the speeds to the update): the fill of the advancing leaves, each
// leaf's step, its update and clock.  No workgroup reads what another writes:
// the ghost cells were filled before.  As two launches, fill and update took
// 11.1 + 8.0 us an iteration on the 2-level grid of 1129 16^2 leaves, so 14.2.
template <int R, int SOLVER>
__global__ void __launch_bounds__(512)
k_lts_leaves(AmrPlanDev A, Fields F, int cur, const AmrClock* clock, AmrLts L) {
  constexpr int kWaves = 8;
  __shared__ double pre[kWaves][4][64];
  __shared__ double leaf_max[kWaves][64];
  __shared__ double leaf_dt[64];
  const AmrBlock K = gl(A.blocks + blockIdx.x);
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const SegRec* const recs = A.list.recs + (long long)blockIdx.x * A.max_waves * A.list.group;
  SegLane g = seg_lane(A.list, seg_wave(A.max_waves));
  const SegDesc D = seg_desc(A.list, g);
  if (blockIdx.x == 0 && threadIdx.x == 0) {  // not read in this launch
    *L.iter = 0;
    *L.itn = *L.itn + 1;
  }
  // the rows of all leaves next to their flags, not behind them
  const int leaf_slot = gl(&(recs + (lane < K.nseg ? lane : 0))->d.slot);
  const State N = state_of(F, cur), O = state_of(F, 1 - cur);
  SegRows<R, true> q;
  q.template load<kRowsInterior>(D, g, N, F.b, g.rb + 1);
  const bool go = lane < K.nseg && gl(L.adv + leaf_slot) != 0;
  if (g.segok && !gl(L.adv + D.slot)) g.active = false;
  const unsigned long long advancing = __builtin_amdgcn_ballot_w64(go);
  if (advancing == 0) return;  // the same in every wavefront
  // uNew -> uOld (DefaultTransfer::copyUNewToUOld)
#pragma unroll
  for (int k = 1; k <= R; ++k) {
    if (!g.active || k > g.rows) continue;
    const long long o = D.off + (long long)(g.ra - 1 + k) * D.stride + g.col;
    gs(F.H(1 - cur) + o, q.h[k]);
    gs(F.HU(1 - cur) + o, q.hu[k]);
    gs(F.HV(1 - cur) + o, q.hv[k]);
  }
  __syncthreads();
  amr_walls(K, recs, A.walls, A.dims, F, 1 - cur, L.adv);
  q.template load<kRowsGhost>(D, g, O, F.b, g.rb + 1);
  const double v = seg_speeds<R, SOLVER>(g, q, g.rb == g.nx ? g.rb + 1 : g.rb, N, O, F.b, pre[w]);
  if (g.segok && g.col == 1) leaf_max[w][g.seg] = v;
  wave_sync();
  seg_side_shares<SOLVER>(g, O, F.b, pre[w]);
  __syncthreads();
  if (w == 0 && go) {
    const SegDesc P = gl(&(recs + lane)->d);
    double m = leaf_max[0][lane];
    for (int k = 1; k < K.nwaves; ++k) m = dmax(m, leaf_max[k][lane]);
    const double t = L.t[leaf_slot], dt0 = L.dt[leaf_slot];
    const double md = clock->end_time - (t + dt0);
    const double dt = fmin(max_timestep(m, P.dx, P.dy), md);  // SWEKernel.cpp:60-68
    leaf_dt[lane] = dt;
    if (dt - 0.0 > kLaEps) {  // SWEKernel.cpp:83-87
      L.t[leaf_slot] = t + dt0;
      L.dt[leaf_slot] = dt;
    }
  }
  if (threadIdx.x == 0) atomicAdd(L.steps, (unsigned long long)__popcll(advancing));
  __syncthreads();
  seg_update_rows<R, SOLVER>(g, D, q, g.active ? leaf_dt[g.seg] : 0.0, pre[w], F.H(cur),
                             F.HU(cur), F.HV(cur));
}

// The smallest of many workgroups' CFL steps, where the update's workgroups
// would otherwise each read more than kCflFold of them.
constexpr int kCflFold = 1024;
__global__ void __launch_bounds__(1024)
k_cfl_fold(const double* __restrict__ cfl_block, int n, double* __restrict__ out) {
  __shared__ double red[16];
  double v = kNoLimit;
  for (int k = threadIdx.x; k < n; k += 1024) v = dmin(v, gl(cfl_block + k));
  v = block_min(v, red);
  if (threadIdx.x == 0) *out = v;
}

// The update of every leaf, uOld -> uNew, after the fill; the last workgroup
// does the clocks.  Global steps: the step is the smallest of cfl[0 .. ncfl)
// bounded by the step left to the end time (every leaf's fmin(own CFL step,
// bound) equals it), the clock goes from `in` to `out` and, with the last
// step of a call, to pinned host memory (`host`).  Local time stepping:
// the advancing leaves by their own steps, their clocks (SWEKernel.cpp:83-87)
// by their first segment.
template <int R, int SOLVER, bool LTS>
__global__ void __launch_bounds__(64 * kSegWaves)
__attribute__((amdgpu_waves_per_eu(R == 4 ? 3 : 2, 8)))
k_amr_update(AmrPlanDev A, Fields F, int cur, const AmrClock* in, AmrClock* out,
             AmrClock* host, const double* __restrict__ cfl, int ncfl, AmrLts L) {
  __shared__ double pre[kSegWaves][4][64];
  __shared__ double red[kSegWaves];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const bool tail = blockIdx.x == gridDim.x - 1;
  double dt = 0.0;
  bool adv = true;
  if (LTS) {
    if (tail) {  // no other workgroup of this launch reads them
      if (threadIdx.x == 0) {
        *L.iter = 0;
        *L.itn = *L.itn + 1;
      }
      return;
    }
  } else {
    const AmrClock c = gl(in);
    adv = amr_advance(c);
    const SegRange all{0, ncfl};
    if (tail) {
      if (w) return;
      const double m = cfl_share(all, cfl, lane, 64);
      if (lane) return;
      AmrClock n = c;
      n.advance = adv ? 1 : 0;
      if (adv) {
        const double md = c.end_time - (c.time + c.dt);
        n.bound = md < m ? md : m;
        // SWEKernel.cpp:83-87 for every leaf
        if (n.bound - 0.0 > kLaEps) {
          n.time = c.time + c.dt;
          n.dt = n.bound;
        }
        n.steps = c.steps + 1;
      }
      *out = n;
      if (host) *host = n;
      return;
    }
    dt = c.end_time - (c.time + c.dt);
    const double m = cfl_share(all, cfl, (int)threadIdx.x, 64 * kSegWaves);
    if (lane == 0) red[w] = m;
  }
  SegLane g = seg_lane(A.list, seg_wave(kSegWaves));
  const SegDesc D = seg_desc(A.list, g);
  if (!adv) return;  // behind the first loads, not before them
  const State O = state_of(F, 1 - cur);
  if (LTS) {
    const bool go = g.segok && L.adv[D.slot] != 0;
    g.active = g.active && go;
    if (__builtin_amdgcn_ballot_w64(go) == 0) return;  // LTS has no workgroup barrier
    dt = go ? L.stepdt[D.slot] : 0.0;
  }
  SegRows<R, true> q;
  q.template load<kRowsAll>(D, g, O, F.b, g.rb + 1);
  seg_side_shares<SOLVER>(g, O, F.b, pre[w]);
  if (LTS) {
    wave_sync();
  } else {
    __syncthreads();
    for (int k = 0; k < kSegWaves; ++k) dt = red[k] < dt ? red[k] : dt;
    if (g.nseg == 0) return;
  }
  seg_update_rows<R, SOLVER>(g, D, q, dt, pre[w], F.H(cur), F.HU(cur), F.HV(cur));
  if (LTS && g.active && g.col == 1 && g.sidx == 0) {
    if (dt - 0.0 > kLaEps) {
      L.t[D.slot] = L.t[D.slot] + L.dt[D.slot];
      L.dt[D.slot] = dt;
    }
    atomicAdd(L.steps, 1ull);
  }
}

// End time of every virtual patch: the minimum over the leaves below it
// (vleaf[vptr[v] .. vptr[v + 1])), a wavefront each.
__global__ void __launch_bounds__(256)
k_lts_virtual_ends(const int* __restrict__ vptr, const int* __restrict__ vleaf, int nvirt,
                   AmrLts L, double* __restrict__ vend) {
  const int v = blockIdx.x * 4 + (int)(threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (v >= nvirt) return;
  double m = kNoLimit;
  for (int i = vptr[v] + lane; i < vptr[v + 1]; i += 64) {
    const int x = vleaf[i];
    m = dmin(m, L.t[x] + L.dt[x]);
  }
  for (int o = 32; o >= 1; o >>= 1) m = dmin(m, __shfl_xor(m, o));
  if (lane == 0) vend[v] = m;
}

// TimeIntervals::isAllowedToAdvanceInTime (TimeIntervals.cpp:24-84) of each
// leaf: the step bound end - (t + dt) > 1e-8 and t + dt - constraint <= 1e-8,
// the constraint being the minimal end time over the neighbours listed in
// nptr/nbr (>= 0: a leaf slot; < 0: -1 - the slot of a virtual patch, whose
// end time is vend[vidx[slot]], from k_lts_virtual_ends).  Counts the
// advancing leaves into *iter (zeroed by the last launch of the previous
// iteration) and stamps the virtual patches they read with the iteration
// number.
//
// For plans past the limits of k_lts_flags_block: an iteration of 4681 8^2
// leaves on five levels (16,407 leaves below virtual patches) takes 34.1 us;
// with every leaf walking the leaves below its virtual neighbours it took 582.
__global__ void __launch_bounds__(256)
k_lts_flags(const int* __restrict__ leaves, int nleaves, const int* __restrict__ nptr,
            const int* __restrict__ nbr, const double* __restrict__ vend,
            const int* __restrict__ vidx, const int* __restrict__ rptr,
            const int* __restrict__ rsrc, const AmrClock* clock, AmrLts L) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nleaves) return;
  const int s = leaves[k];
  const double e = L.t[s] + L.dt[s];
  const double md = clock->end_time - e;
  double c = kNoLimit;
  for (int j = nptr[k]; j < nptr[k + 1]; ++j) {
    const int q = nbr[j];
    c = dmin(c, q >= 0 ? L.t[q] + L.dt[q] : vend[vidx[-1 - q]]);
  }
  const int adv = (md - 0.0 > kLaEps) && !(e - c > kLaEps);
  L.adv[s] = adv;
  if (adv) {
    atomicAdd(L.iter, 1);
    // the virtual patches its ghost faces read (rsrc[rptr[k] .. rptr[k+1]))
    const int stamp = *L.itn;
    for (int j = rptr[k]; j < rptr[k + 1]; ++j) L.need[rsrc[j]] = stamp;
  }
}

// A double as an unsigned integer of the same order, and back.
__device__ __forceinline__ unsigned long long order_key(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  return b ^ ((unsigned long long)((long long)b >> 63) | 0x8000000000000000ull);
}
__device__ __forceinline__ double from_order_key(unsigned long long k) {
  return __longlong_as_double(
      (long long)(k ^ ((k >> 63) ? 0x8000000000000000ull : 0xFFFFFFFFFFFFFFFFull)));
}

// The same decision for plans of up to kLtsBlockVirtuals virtual patches and
// kLtsBlockPairs leaves below them whose leaves have at most kLtsNeighbours
// neighbours: every workgroup first takes the virtual patches' end times in
// LDS (a thread per leaf below one, LDS minima), while its own leaves' data
// is on the way, then decides one leaf per thread.  neighbours[k *
// kLtsNeighbours ..]: leaf slots, -1 - v for the virtual patch of index v,
// the leaf itself in free places.
//
// Latency-bound: about four dependent loads.  One workgroup of 1024 threads
// with offset lists (eight dependent loads, two rounds of 1129 leaves, an
// atomic per advancing leaf) took 12.7 us an iteration, this form 5.2.
constexpr int kLtsBlockVirtuals = 4096;  // 32 KiB of LDS
// Every workgroup walks all pairs: us an iteration, this form / two launches,
// 1157 pairs 22.3 / 25.2, 3158: 26.4 / 28.3, 4857: 28.2 / 28.6, 12,358: 54.6 /
// 36.2, 48,229: 145 / 58.6.
constexpr int kLtsBlockPairs = 4096;
constexpr int kLtsNeighbours = 8;
__global__ void __launch_bounds__(256)
k_lts_flags_block(const int* __restrict__ leaves, int nleaves,
                  const int* __restrict__ neighbours, const int* __restrict__ vleaf,
                  const int* __restrict__ vowner, int npairs, int nvirt,
                  const int* __restrict__ rptr, const int* __restrict__ rsrc,
                  const AmrClock* clock, AmrLts L) {
  extern __shared__ unsigned long long vend[];
  for (int v = threadIdx.x; v < nvirt; v += 256) vend[v] = order_key(kNoLimit);
  const int k = blockIdx.x * 256 + threadIdx.x;
  const bool ok = k < nleaves;
  const int s = ok ? leaves[k] : 0;
  int q[kLtsNeighbours];
#pragma unroll
  for (int j = 0; j < kLtsNeighbours; ++j)
    q[j] = ok ? gl(neighbours + k * kLtsNeighbours + j) : -1;
  const int r0 = ok ? rptr[k] : 0, r1 = ok ? rptr[k + 1] : 0;
  double c = kNoLimit, e = 0.0;
  if (ok) {
    e = gl(L.t + s) + gl(L.dt + s);
#pragma unroll
    for (int j = 0; j < kLtsNeighbours; ++j)
      if (q[j] >= 0) c = dmin(c, gl(L.t + q[j]) + gl(L.dt + q[j]));
  }
  __syncthreads();
  for (int i = threadIdx.x; i < npairs; i += 256) {
    const int x = vleaf[i];
    atomicMin(&vend[vowner[i]], order_key(gl(L.t + x) + gl(L.dt + x)));
  }
  __syncthreads();
  const double md = clock->end_time - e;
#pragma unroll
  for (int j = 0; j < kLtsNeighbours; ++j)
    if (ok && q[j] < 0) c = dmin(c, from_order_key(vend[-1 - q[j]]));
  const bool adv = ok && (md - 0.0 > kLaEps) && !(e - c > kLaEps);
  if (ok) L.adv[s] = adv ? 1 : 0;
  const unsigned long long m = __builtin_amdgcn_ballot_w64(adv);
  if (m && (threadIdx.x & 63) == 0) atomicAdd(L.iter, (int)__popcll(m));
  if (adv && r1 > r0) {
    const int stamp = *L.itn;
    for (int j = r0; j < r1; ++j) L.need[rsrc[j]] = stamp;
  }
}

}  // namespace

// A slot as the plan's tables know it.
struct AmrPlace {
  long long off;   // its tile
  double size[2];  // of the patch
  int nx, ny;
};

struct pc_amr {
  pc_pool* pool = nullptr;
  std::vector<int> leaves, virtuals, plan_slots;
  std::vector<int> leaf_nx, leaf_ny;
  int nvblocks = 0, nghosts = 0;
  // what the tables hold of the plan's slots (amr_follow_slots), and the tables
  // themselves where they depend on it
  unsigned long long layout = 0;  // of the pool, as these follow it
  std::vector<AmrPlace> places;  // per plan slot
  std::vector<SegDesc> h_desc;   // per leaf in task order
  std::vector<AmrVBlock> h_vblocks;
  std::vector<AmrGhost> h_ghosts;
  Task* d_tasks = nullptr;  // row segments of the tasks
  SegDesc* d_desc = nullptr;
  int nrec = 0;  // records made of them
  int* d_cptr = nullptr;
  int* d_cpairs = nullptr;
  AmrRestrict* d_pairs = nullptr;
  // tasks of leaves, their row segments (at most seg_rows rows), and what
  // the fill reads (AmrPlanDev)
  int seg_rows = 4, nblocks = 0, nsegs = 0, max_waves = 1, max_cells = 0;
  AmrBlock* d_blocks = nullptr;
  SegList list{};
  int* d_gmap = nullptr;
  double* d_cfl = nullptr;  // per block, then the folded one
  int* d_leaves = nullptr;
  AmrVBlock* d_vblocks = nullptr;
  int* d_xptr = nullptr;  // per virtual cell: its contributions
  AmrContrib* d_contribs = nullptr;  // nullptr: no list (amr_list_fits)
  AmrGhost* d_ghosts = nullptr;
  AmrWalls* d_walls = nullptr;  // per leaf in task order
  int* d_wall_dims = nullptr;
  AmrClock* d_clock = nullptr;
  AmrClock* d_clock_next = nullptr;  // the clock a global step writes
  AmrClock h_clock{};                // as after the last call
  char* d_tables = nullptr;  // one allocation holding every d_* table above
  size_t tables_cap = 0;
  double last_dt = 0.0;
  bool shared_clock = true;  // all leaves on one clock (global steps allowed)
  // local time stepping: per-slot clocks and flags, neighbour lists of the
  // leaves, leaves below each virtual patch
  std::vector<std::vector<int>> vleaves;  // per virtual patch, plan order
  bool lts_ready = false;
  AmrLts lts{};
  int* d_vidx = nullptr;   // per slot: index of the virtual patch, -1 otherwise
  int* d_rptr = nullptr;   // per leaf (plan order): the virtual patches its faces read
  int* d_rsrc = nullptr;
  int* d_vptr = nullptr;
  int* d_vleaf = nullptr;
  int* d_nptr = nullptr;
  int* d_nbr = nullptr;
  double* d_vend = nullptr;     // end times of the virtual patches (k_lts_virtual_ends)
  int* d_vowner = nullptr;      // per entry of d_vleaf: its virtual patch's index
  int* d_neighbours = nullptr;  // k_lts_flags_block's table, where the plan fits it
  int npairs = 0;
};

namespace {

template <class T>
int amr_upload(T** d, const std::vector<T>& h) {
  HIPCHK(hipMalloc(d, std::max<size_t>(h.size(), 1) * sizeof(T)));
  if (!h.empty()) HIPCHK(hipMemcpy(*d, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice));
  return PC_OK;
}

void amr_free(pc_amr* a) {
  // the table buffer goes back to the pool for the next plan (the caller
  // has synchronised the stream)
  if (a->d_tables && !a->pool->amr_tables) {
    a->pool->amr_tables = a->d_tables;
    a->pool->amr_tables_cap = a->tables_cap;
  } else if (a->d_tables) {
    hipFree(a->d_tables);
  }
  a->d_tables = nullptr;
  void* lts[] = {a->lts.t,   a->lts.dt,   a->lts.adv, a->lts.stepdt, a->lts.iter, a->lts.steps,
                 a->lts.itn, a->lts.need, a->d_vidx,  a->d_vptr,     a->d_vleaf,  a->d_nptr,
                 a->d_nbr,   a->d_rptr,   a->d_rsrc, a->d_vowner, a->d_neighbours, a->d_vend};
  for (void* q : lts) hipFree(q);
}

// Leaves per task: their ghost-column edges (two per row) fit the segments'
// LDS at 4 rows.
constexpr int kAmrTaskLeaves = 16;

// Rows per segment of the plan's leaves: 2 while that gives at most 2.5
// wavefronts a SIMD (2-level grid of 1129 16^2 leaves, 2264 wavefronts: 44.3
// us a step against 45.1 with 4 rows), else 4 (3-level grid of 729 27^2
// leaves, 5110 wavefronts: 66.7 us against 74.5).
int amr_seg_rows(const std::vector<Task>& tasks) {
  long long n = 0;
  for (const Task& t : tasks) {
    n += seg_count(t.nx, 2);
    if (t.nx > 32) return 4;  // at most 16 wavefronts per workgroup
  }
  return n <= 2560 ? 2 : 4;
}

// Whether a plan keeps its list of n contributions: it counts them in 32 bits,
// and the list (16 bytes a fine cell and virtual patch above it, next to 56
// bytes a cell of the pool's fields) must fit what the fields leave of the
// pool's budget.  Lists of up to kContribListFloor bytes are always made.  A
// step that derives the contributions instead restricts in 22.8 us rather than
// 18.6 on the 3-level grid of 729 27^2 leaves, 13.7 rather than 6.2 on the
// 2-level grid of 1129 16^2 leaves.
constexpr long long kContribListFloor = 64ll << 20;
bool amr_list_fits(const pc_pool* p, long long n) {
  const long long left = (long long)p->budget - p->cap_cells * (long long)kBytesPerCell;
  return n <= INT_MAX && n * (long long)sizeof(AmrContrib) <= std::max(left, kContribListFloor);
}

// The plan's slots must still be live with the same role and numbers of cells.
int amr_check_slots(pc_amr* a) {
  pc_pool* p = a->pool;
  for (size_t i = 0; i < a->plan_slots.size(); ++i) {
    const bool virt = i >= a->leaves.size();
    const int s = a->plan_slots[i];
    if (!valid_slot(p, s) || (p->slots[s].desc.is_virtual != 0) != virt ||
        p->slots[s].desc.subdivision_factor[0] != a->places[i].nx ||
        p->slots[s].desc.subdivision_factor[1] != a->places[i].ny)
      return fail(PC_E_INVALID,
                  virt ? "a virtual patch of the AMR plan changed or was released"
                       : "a leaf of the AMR plan changed or was released");
  }
  return PC_OK;
}

AmrPlace amr_place(const Slot& s) {
  return AmrPlace{s.off, {s.desc.size[0], s.desc.size[1]}, s.desc.subdivision_factor[0],
                  s.desc.subdivision_factor[1]};
}

// A leaf as the fill and the update read it: ghosts in its own tile.
SegDesc amr_seg_desc(const pc_pool* p, int slot) {
  const PatchDev P = make_patchdev(p->slots[slot]);
  SegDesc d{};
  d.off = P.off;
  d.gx[0] = P.off;
  d.gx[1] = P.off + (long long)(P.nx + 1) * P.stride;
  d.gy[0] = P.off;
  d.gy[1] = P.off + P.ny + 1;
  d.nx = P.nx; d.ny = P.ny; d.stride = P.stride;
  d.slot = slot;
  d.scn = P.scn;
  d.dx = P.dx; d.dy = P.dy; d.dxinv = P.dxinv; d.dyinv = P.dyinv;
  return d;
}

// Where a ghost entry's source and destination regions begin.
void amr_ghost_places(const pc_pool* p, AmrGhost& g) {
  const Slot &ss = p->slots[g.src], &ds = p->slots[g.dst];
  g.sbase = ss.off + (long long)(g.sox + 1) * ss.stride + (g.soy + 1);
  g.dbase = ds.off + (long long)(g.dox + 1) * ds.stride + (g.doy + 1);
  g.sstride = ss.stride;
  g.dstride = ds.stride;
}

// The tables the device makes itself: the leaves' records and, with
// `places`, the restriction's contributions (their cells' places).
int amr_device_tables(pc_amr* a, bool places) {
  pc_pool* p = a->pool;
  hipLaunchKernelGGL(k_seg_records, dim3((a->nrec + 255) / 256), dim3(256), 0, p->stream,
                     a->d_tasks, a->d_desc, a->nrec, a->list.group,
                     const_cast<SegRec*>(a->list.recs));
  if (places && a->d_contribs && !a->h_vblocks.empty())
    hipLaunchKernelGGL(k_amr_contribs,
                       dim3((unsigned)(a->h_vblocks.size() * kRestrictCells / 256)), dim3(256), 0,
                       p->stream, a->d_vblocks, a->d_cptr, a->d_cpairs, a->d_xptr, a->d_pairs,
                       p->d_pd, a->d_contribs);
  HIPCHK(hipGetLastError());
  return PC_OK;
}

// The plan's tables follow its slots: the tile of a slot moves when it is
// released and registered again, and pc_patch_set_description may give a live
// patch another size.  Steps and speeds take the cells' size as it is now; the
// transfers between patches keep the geometry they were created with.  Called
// ahead of every step call, after prepare (the slots' tiles on the device).
int amr_follow_slots(pc_amr* a) {
  pc_pool* p = a->pool;
  if (a->layout == p->layout) return PC_OK;
  CHK(amr_check_slots(a));
  bool moved = false, sized = false;
  for (size_t i = 0; i < a->plan_slots.size(); ++i) {
    const Slot& s = p->slots[a->plan_slots[i]];
    const AmrPlace& q = a->places[i];
    moved = moved || s.off != q.off;
    sized = sized || s.desc.size[0] != q.size[0] || s.desc.size[1] != q.size[1];
  }
  if (!moved && !sized) {
    a->layout = p->layout;
    return PC_OK;
  }
  for (SegDesc& d : a->h_desc) d = amr_seg_desc(p, d.slot);
  HIPCHK(hipMemcpyAsync(a->d_desc, a->h_desc.data(), a->h_desc.size() * sizeof(SegDesc),
                        hipMemcpyHostToDevice, p->stream));
  if (moved) {
    for (AmrVBlock& B : a->h_vblocks) B.off = p->slots[B.slot].off;
    for (AmrGhost& g : a->h_ghosts) amr_ghost_places(p, g);
    if (!a->h_vblocks.empty())
      HIPCHK(hipMemcpyAsync(a->d_vblocks, a->h_vblocks.data(),
                            a->h_vblocks.size() * sizeof(AmrVBlock), hipMemcpyHostToDevice,
                            p->stream));
    if (!a->h_ghosts.empty())
      HIPCHK(hipMemcpyAsync(a->d_ghosts, a->h_ghosts.data(),
                            a->h_ghosts.size() * sizeof(AmrGhost), hipMemcpyHostToDevice,
                            p->stream));
  }
  CHK(amr_device_tables(a, moved));
  HIPCHK(hipStreamSynchronize(p->stream));
  for (size_t i = 0; i < a->plan_slots.size(); ++i)
    a->places[i] = amr_place(p->slots[a->plan_slots[i]]);
  a->layout = p->layout;
  return PC_OK;
}

int amr_cur(pc_amr* a, int* cur) {
  pc_pool* p = a->pool;
  const int c = cur_of(p, a->plan_slots[0]);
  for (int s : a->plan_slots)
    if (cur_of(p, s) != c)
      return fail(PC_E_INVALID, "AMR patches must share one state parity (one scenario)");
  *cur = c;
  return PC_OK;
}

}  // namespace

extern "C" {

int pc_amr_create(pc_pool* p, const int32_t* leaves, int nleaves, const int32_t* virtuals,
                  int nvirtuals, const int32_t* restrictions, int nrestrictions,
                  const pc_amr_ghost* ghosts, int nghosts, const pc_amr_wall* walls,
                  int nwalls, pc_amr** out) {
  if (!p || !out || nleaves < 1 || nvirtuals < 0 || nrestrictions < 0 || nghosts < 0 ||
      nwalls < 0 || !leaves || (nvirtuals && !virtuals) || (nrestrictions && !restrictions) ||
      (nghosts && !ghosts) || (nwalls && !walls))
    return fail(PC_E_INVALID, "invalid argument");
  hipSetDevice(p->device);
  CHK(prepare(p));
  std::vector<char> role(p->slots.size(), 0);  // 1 leaf, 2 virtual
  for (int i = 0; i < nleaves; ++i) {
    const int s = leaves[i];
    if (!valid_slot(p, s) || p->slots[s].desc.is_virtual || role[s])
      return fail(PC_E_INVALID, "leaves must be distinct live non-virtual patches");
    role[s] = 1;
  }
  for (int i = 0; i < nvirtuals; ++i) {
    const int s = virtuals[i];
    if (!valid_slot(p, s) || !p->slots[s].desc.is_virtual || role[s])
      return fail(PC_E_INVALID, "virtual patches must be distinct live virtual patches");
    role[s] = 2;
  }
  pc_amr* a = new pc_amr;
  a->pool = p;
  a->leaves.assign(leaves, leaves + nleaves);
  a->virtuals.assign(virtuals, virtuals + nvirtuals);
  a->plan_slots = a->leaves;
  a->plan_slots.insert(a->plan_slots.end(), a->virtuals.begin(), a->virtuals.end());
  for (int s : a->plan_slots) a->places.push_back(amr_place(p->slots[s]));
  a->layout = p->layout;
  // leaf clock: every leaf on one clock
  double t0, dt0;
  slot_clock(p, leaves[0], &t0, &dt0);
  for (int s : a->leaves) {
    double t, dt;
    slot_clock(p, s, &t, &dt);
    if (t != t0 || dt != dt0) a->shared_clock = false;
  }
  auto bail = [&](const char* msg) {
    amr_free(a);
    delete a;
    return fail(PC_E_INVALID, msg);
  };
  // leaf tasks: runs of equal-size leaves packed 64 / pow2(ny) per wavefront
  std::vector<Task> tasks;
  std::vector<int> plist;
  for (int s : a->leaves) {
    const auto& d = p->slots[s].desc;
    a->leaf_nx.push_back(d.subdivision_factor[0]);
    a->leaf_ny.push_back(d.subdivision_factor[1]);
    if (d.subdivision_factor[1] > 64) return bail("leaf patches must have ny <= 64");
  }
  for (size_t i = 0; i < a->leaves.size();) {
    const int nx = a->leaf_nx[i], ny = a->leaf_ny[i];
    int w = 1;
    while (w < ny) w <<= 1;
    const int per = std::min(64 / w, kAmrTaskLeaves);
    Task t{(int)plist.size(), 0, nx, ny};
    while (i < a->leaves.size() && t.nseg < per && a->leaf_nx[i] == nx && a->leaf_ny[i] == ny) {
      plist.push_back(a->leaves[i]);
      ++t.nseg;
      ++i;
    }
    tasks.push_back(t);
  }
  // row segments: short ones while they are few (latency), else longer ones
  // (work); per task a workgroup of the fill
  a->seg_rows = amr_seg_rows(tasks);
  std::vector<Task> segs;
  std::vector<AmrBlock> blocks;
  std::vector<SegDesc> desc;
  std::vector<int> pos(p->slots.size(), -1);  // place of a leaf in plist
  for (size_t k = 0; k < plist.size(); ++k) {
    desc.push_back(amr_seg_desc(p, plist[k]));
    pos[plist[k]] = (int)k;
  }
  for (const Task& t : tasks) {
    AmrBlock B{};
    B.nwaves = seg_count(t.nx, a->seg_rows);
    B.leaf0 = t.first;
    B.nseg = t.nseg;
    B.nx = t.nx;
    B.ny = t.ny;
    a->max_waves = std::max(a->max_waves, B.nwaves);
    blocks.push_back(B);
  }
  for (size_t b = 0; b < blocks.size(); ++b)
    for (int k = 0; k < a->max_waves; ++k) {
      Task u = tasks[b];
      const int n = blocks[b].nwaves;
      u.r0 = k < n ? seg_first_row(k, u.nx, n) : 1;
      u.r1 = k < n ? seg_first_row(k + 1, u.nx, n) - 1 : 1;
      u.sidx = k;
      if (k >= n) u.nseg = 0;
      segs.push_back(u);
    }
  while (segs.size() % kSegWaves) {
    Task u = segs.back();
    u.nseg = 0;
    segs.push_back(u);
  }
  a->list.lanes = 1;
  while (a->list.lanes < tasks[0].ny) a->list.lanes <<= 1;
  a->list.group = 1;
  for (const Task& t : tasks) {
    a->list.group = std::max(a->list.group, t.nseg);
    if (a->list.lanes && (t.ny > a->list.lanes || 2 * t.ny <= a->list.lanes)) a->list.lanes = 0;
  }
  a->nblocks = (int)blocks.size();
  a->nsegs = (int)segs.size();
  // restriction pairs grouped by virtual patch, in the given order; per
  // virtual cell the list of pairs covering it
  std::vector<AmrVBlock> vblocks;
  std::vector<int> cptr{0}, cpairs, xptr{0};
  long long ncontribs = 0;
  std::vector<AmrRestrict> pairs;
  std::vector<int> leaf_at(role.size(), -1);
  for (int k = 0; k < nleaves; ++k) leaf_at[leaves[k]] = k;
  // the restrictions of each destination slot, in the given order
  std::vector<int> rbeg(role.size() + 1, 0), rlist(nrestrictions);
  for (int r = 0; r < nrestrictions; ++r) {
    const int v = restrictions[2 * r + 1];
    if (v >= 0 && v < (int)role.size()) ++rbeg[v + 1];
  }
  for (size_t k = 1; k < rbeg.size(); ++k) rbeg[k] += rbeg[k - 1];
  {
    std::vector<int> fill(rbeg.begin(), rbeg.end() - 1);
    for (int r = 0; r < nrestrictions; ++r) {
      const int v = restrictions[2 * r + 1];
      if (v >= 0 && v < (int)role.size()) rlist[fill[v]++] = r;
    }
  }
  std::vector<int> ccount, xcount, span0, span1;
  {
    size_t cells = 1;
    for (int vi = 0; vi < nvirtuals; ++vi)
      cells += (size_t)p->slots[virtuals[vi]].desc.subdivision_factor[0] *
               p->slots[virtuals[vi]].desc.subdivision_factor[1];
    cptr.reserve(cells);
    xptr.reserve(cells);
    vblocks.reserve(cells / kRestrictCells + nvirtuals + 256);
    pairs.reserve(nrestrictions);
  }
  for (int vi = 0; vi < nvirtuals; ++vi) {
    const int v = virtuals[vi];
    const int pbeg = (int)pairs.size();
    const auto& dd = p->slots[v].desc;
    const PatchDev D = make_patchdev(p->slots[v]);
    for (int ri = rbeg[v]; ri < rbeg[v + 1]; ++ri) {
      const int r = rlist[ri];
      const int s = restrictions[2 * r];
      if (s < 0 || s >= (int)role.size() || role[s] != 1)
        return bail("a restriction source is not a leaf of the plan");
      const auto& sd = p->slots[s].desc;
      const PatchDev S = make_patchdev(p->slots[s]);
      AmrRestrict R{};
      R.src = s;
      R.leaf = leaf_at[s];
      const int z[2] = {0, 0};
      const int sn[2] = {sd.subdivision_factor[0], sd.subdivision_factor[1]};
      const int dn[2] = {dd.subdivision_factor[0], dd.subdivision_factor[1]};
      map_to_patch(z, sn, S, sd, D, dd, 1e-12, R.dOff, R.dSize);
      for (int d = 0; d < 2; ++d) {
        if (R.dOff[d] < 0 || R.dOff[d] + R.dSize[d] > dn[d])
          return bail("restriction source is not inside the destination");
        R.rSize[d] = sn[d];
        R.srcSub[d] = sd.size[d] * (1.0 / (double)sn[d]);
        R.dstSub[d] = dd.size[d] * (1.0 / (double)dn[d]);
        R.spos[d] = sd.position[d];
        R.dpos[d] = dd.position[d];
      }
      R.dstRegion = R.dstSub[0] * R.dstSub[1];
      pairs.push_back(R);
    }
    a->vleaves.emplace_back();
    for (int pi = pbeg; pi < (int)pairs.size(); ++pi) a->vleaves.back().push_back(pairs[pi].src);
    const int nx = dd.subdivision_factor[0], ny = dd.subdivision_factor[1];
    const int base = (int)cptr.size() - 1;
    const double area = (dd.size[0] * (1.0 / (double)nx)) * (dd.size[1] * (1.0 / (double)ny));
    for (int c0 = 0; c0 < nx * ny; c0 += kRestrictCells)
      vblocks.push_back(AmrVBlock{D.off, area, v, c0, base, nx, ny, D.stride});
    // per cell the pairs whose region covers it, in pair order: count, then
    // fill pair by pair (each pair marks its region's cells)
    ccount.assign((size_t)nx * ny, 0);
    xcount.assign((size_t)nx * ny, 0);
    for (int pi = pbeg; pi < (int)pairs.size(); ++pi) {
      const AmrRestrict& R = pairs[pi];
      int o;
      span0.resize(R.dSize[0] > 0 ? R.dSize[0] : 0);
      span1.resize(R.dSize[1] > 0 ? R.dSize[1] : 0);
      for (size_t k = 0; k < span0.size(); ++k) amr_fine_span(R, 0, R.dOff[0] + (int)k, o, span0[k]);
      for (size_t k = 0; k < span1.size(); ++k) amr_fine_span(R, 1, R.dOff[1] + (int)k, o, span1[k]);
      for (int x = 0; x < R.dSize[0]; ++x) {
        const size_t row = (size_t)(R.dOff[0] + x) * ny + R.dOff[1];
        int *const cc = ccount.data() + row, *const xc = xcount.data() + row, n0 = span0[x];
        for (int y = 0; y < R.dSize[1]; ++y) {
          ++cc[y];
          xc[y] += n0 * span1[y];
        }
      }
    }
    const size_t cbeg = cpairs.size();
    cptr.resize(cptr.size() + (size_t)nx * ny);
    xptr.resize(cptr.size());
    for (int c = 0; c < nx * ny; ++c) {
      cptr[base + c + 1] = cptr[base + c] + ccount[c];
      ncontribs += xcount[c];
      xptr[base + c + 1] = (int)std::min<long long>(ncontribs, INT_MAX);
    }
    cpairs.resize(cptr.back());
    for (int c = 0; c < nx * ny; ++c) ccount[c] = cptr[base + c] - (int)cbeg;  // cursors
    for (int pi = pbeg; pi < (int)pairs.size(); ++pi) {
      const AmrRestrict& R = pairs[pi];
      for (int x = 0; x < R.dSize[0]; ++x) {
        int* const cc = ccount.data() + (size_t)(R.dOff[0] + x) * ny + R.dOff[1];
        for (int y = 0; y < R.dSize[1]; ++y) cpairs[cbeg + cc[y]++] = pi;
      }
    }
  }
  for (int r = 0; r < nrestrictions; ++r) {
    const int v = restrictions[2 * r + 1];
    if (v < 0 || v >= (int)role.size() || role[v] != 2)
      return bail("a restriction destination is not a virtual patch of the plan");
  }
  a->nvblocks = (int)vblocks.size();
  // ghost faces
  std::vector<AmrGhost> gh;
  gh.reserve(nghosts);
  for (int i = 0; i < nghosts; ++i) {
    const pc_amr_ghost& G = ghosts[i];
    const int s = G.src, d = G.dst;
    if (s < 0 || d < 0 || s >= (int)role.size() || d >= (int)role.size() || role[d] != 1 ||
        !role[s])
      return bail("a ghost entry needs a leaf destination and a plan source");
    const auto& sd = p->slots[s].desc;
    const auto& dd = p->slots[d].desc;
    AmrGhost g{};
    g.src = s;
    g.dst = d;
    g.sx = G.size[0];
    g.sy = G.size[1];
    g.dox = G.dst_offset[0];
    g.doy = G.dst_offset[1];
    for (int k = 0; k < 2; ++k)
      if (G.size[k] < 0 || G.dst_offset[k] < -1 ||
          G.dst_offset[k] + G.size[k] > dd.subdivision_factor[k] + 1)
        return bail("ghost destination region out of bounds");
    // destinations are strips of the ghost ring (entries run concurrently
    // and read interior cells only)
    bool ring = false;
    for (int k = 0; k < 2; ++k)
      ring = ring || (G.size[k] == 1 && (G.dst_offset[k] == -1 ||
                                         G.dst_offset[k] == dd.subdivision_factor[k]));
    if (!ring) return bail("ghost destination must be a strip of the ghost layer");
    if (G.kind == 0) {
      g.kind = sd.is_virtual ? kAmrTransferVirtual : kAmrTransferLeaf;
      g.sox = G.src_offset[0];
      g.soy = G.src_offset[1];
      for (int k = 0; k < 2; ++k)
        if (G.src_offset[k] < 0 || G.src_offset[k] + G.size[k] > sd.subdivision_factor[k])
          return bail("transfer source region out of bounds");
    } else if (G.kind == 1) {
      if (role[s] != 1) return bail("interpolation sources must be leaves");
      g.kind = kAmrInterpolate;
      const PatchDev S = make_patchdev(p->slots[s]), D = make_patchdev(p->slots[d]);
      // the cells read (the grown source region, SWEKernel.cpp:252-263)
      // must lie in the source
      int so[2], ss[2];
      map_to_patch(G.dst_offset, G.size, D, dd, S, sd, 1e-12, so, ss);
      for (int k = 0; k < 2; ++k) {
        const int n = sd.subdivision_factor[k];
        if (so[k] > 0) {
          so[k] = so[k] - 1;
          ss[k] = std::min(n, ss[k] + 2);
        } else {
          ss[k] = std::min(n, ss[k] + 1);
        }
        if (so[k] < 0 || so[k] + ss[k] > n + 1 || n < 2)
          return bail("interpolation region is not covered by the source patch");
        g.sn[k] = n;
      }
      g.spos[0] = sd.position[0];
      g.spos[1] = sd.position[1];
      g.ssub[0] = S.dx;
      g.ssub[1] = S.dy;
      g.sinv[0] = 1.0 / S.dx;
      g.sinv[1] = 1.0 / S.dy;
      g.dpos[0] = dd.position[0];
      g.dpos[1] = dd.position[1];
      g.dsub[0] = D.dx;
      g.dsub[1] = D.dy;
    } else {
      return bail("ghost kind must be 0 (transfer) or 1 (interpolation)");
    }
    amr_ghost_places(p, g);
    gh.push_back(g);
  }
  a->nghosts = (int)gh.size();
  // the ghost cells of every task, one after another
  std::vector<int> block_of(plist.size());
  for (size_t b = 0; b < blocks.size(); ++b)
    for (int k = 0; k < blocks[b].nseg; ++k) block_of[blocks[b].leaf0 + k] = (int)b;
  std::vector<int> b_of(gh.size());
  {
    std::vector<int> ncells(blocks.size(), 0);
    for (size_t e = 0; e < gh.size(); ++e) {
      b_of[e] = block_of[pos[gh[e].dst]];
      int& n = ncells[b_of[e]];
      gh[e].cell0 = n;
      n += gh[e].sx * gh[e].sy;
      a->max_cells = std::max(a->max_cells, n);
    }
  }
  // walls grouped per leaf in call order
  std::vector<AmrWalls> wl(plist.size(), AmrWalls{0, 0});
  for (int i = 0; i < nwalls; ++i) {
    const int s = walls[i].slot;
    if (s < 0 || s >= (int)role.size() || role[s] != 1) return bail("walls belong to leaves");
    if ((walls[i].dimension != 0 && walls[i].dimension != 1) ||
        (walls[i].upper != 0 && walls[i].upper != 1))
      return bail("wall dimension and side must be 0 or 1");
    ++wl[pos[s]].count;
  }
  std::vector<int> wdims(2 * (size_t)nwalls), wnext(plist.size());
  for (size_t k = 0, top = 0; k < wl.size(); ++k) {
    wl[k].first = wnext[k] = (int)top;
    top += wl[k].count;
    AmrBlock& B = blocks[block_of[k]];
    B.nwalls = std::max(B.nwalls, wl[k].count);
  }
  for (int i = 0; i < nwalls; ++i) {
    const int w = wnext[pos[walls[i].slot]]++;
    wdims[2 * w] = walls[i].dimension;
    wdims[2 * w + 1] = walls[i].upper;
  }
  AmrClock c{};
  c.time = t0;
  c.dt = dt0;
  // every table in one device allocation, filled by one copy (a regrid
  // makes a new plan: one allocation, usually the previous plan's, and one
  // DMA instead of fifteen of each)
  PinnedTables st;
  const size_t o_blocks = st.add(blocks), o_tasks = st.add(segs), o_desc = st.add(desc);
  const size_t o_cfl = st.add(nullptr, (blocks.size() + 1) * sizeof(double));
  const size_t o_leaves = st.add(a->leaves);
  // (whole workgroups of the kernel that lists the contributions)
  while (vblocks.size() % (256 / kRestrictCells)) {
    vblocks.push_back(vblocks.back());
    vblocks.back().nx = 0;
  }
  const size_t o_vblocks = st.add(vblocks), o_cptr = st.add(cptr), o_cpairs = st.add(cpairs);
  const size_t o_xptr = st.add(xptr);
  const size_t o_pairs = st.add(pairs), o_ghosts = st.add(gh), o_walls = st.add(wl);
  const size_t o_wall_dims = st.add(wdims), o_ghost_task = st.add(b_of);
  c.end_time = INFINITY;
  a->h_clock = c;
  const std::vector<AmrClock> clk{c};
  const size_t o_clock = st.add(clk), o_next = st.add(clk);
  // the records, the ghost map and the contributions follow, made on the device
  a->nrec = (int)segs.size() * a->list.group;
  const size_t o_recs = (st.total + 255) / 256 * 256;
  const size_t o_gmap = o_recs + (size_t)a->nrec * sizeof(SegRec);
  const size_t gmap_bytes = blocks.size() * (size_t)a->max_cells * sizeof(int);
  const size_t o_contribs = (o_gmap + gmap_bytes + 255) / 256 * 256;
  bool listed = amr_list_fits(p, ncontribs);
  auto bytes = [&]() {
    return o_contribs + (listed ? (size_t)ncontribs * sizeof(AmrContrib) : 0) + 16;
  };
  hipError_t e = hipSuccess;
  if (p->amr_tables && p->amr_tables_cap >= bytes()) {
    a->d_tables = p->amr_tables;  // idle: its plan was destroyed after a sync
    a->tables_cap = p->amr_tables_cap;
    p->amr_tables = nullptr;
    p->amr_tables_cap = 0;
  } else {
    for (;;) {
      // room for a grown grid
      a->tables_cap = bytes() + std::min<size_t>(bytes(), kContribListFloor);
      e = hipMalloc(&a->d_tables, a->tables_cap);
      if (e == hipSuccess || !listed) break;
      (void)hipGetLastError();
      listed = false;
    }
  }
  if (e != hipSuccess) {
    amr_free(a);
    delete a;
    return fail(PC_E_HIP, std::string("plan tables: ") + hipGetErrorString(e));
  }
  const int urc = st.upload(p, a->d_tables);
  if (urc != PC_OK) {
    amr_free(a);
    delete a;
    return urc;
  }
  char* const base = a->d_tables;
  a->d_blocks = reinterpret_cast<AmrBlock*>(base + o_blocks);
  a->d_gmap = reinterpret_cast<int*>(base + o_gmap);
  a->d_cfl = reinterpret_cast<double*>(base + o_cfl);
  a->d_leaves = reinterpret_cast<int*>(base + o_leaves);
  a->d_vblocks = reinterpret_cast<AmrVBlock*>(base + o_vblocks);
  a->d_xptr = reinterpret_cast<int*>(base + o_xptr);
  a->d_contribs = listed ? reinterpret_cast<AmrContrib*>(base + o_contribs) : nullptr;
  a->d_ghosts = reinterpret_cast<AmrGhost*>(base + o_ghosts);
  a->d_walls = reinterpret_cast<AmrWalls*>(base + o_walls);
  a->d_wall_dims = reinterpret_cast<int*>(base + o_wall_dims);
  a->d_clock = reinterpret_cast<AmrClock*>(base + o_clock);
  a->d_clock_next = reinterpret_cast<AmrClock*>(base + o_next);
  a->list.recs = reinterpret_cast<SegRec*>(base + o_recs);
  a->list.scn = 0;  // the plan has its own clock
  a->d_tasks = reinterpret_cast<Task*>(base + o_tasks);
  a->d_desc = reinterpret_cast<SegDesc*>(base + o_desc);
  a->d_cptr = reinterpret_cast<int*>(base + o_cptr);
  a->d_cpairs = reinterpret_cast<int*>(base + o_cpairs);
  a->d_pairs = reinterpret_cast<AmrRestrict*>(base + o_pairs);
  a->h_desc = std::move(desc);
  a->h_vblocks = std::move(vblocks);
  a->h_ghosts = std::move(gh);
  int rc = gmap_bytes && hipMemsetAsync(a->d_gmap, 0xff, gmap_bytes, p->stream) != hipSuccess
               ? fail(PC_E_HIP, "ghost map")
               : PC_OK;
  if (rc == PC_OK && a->nghosts > 0)
    hipLaunchKernelGGL(k_amr_ghost_map, dim3((a->nghosts + 3) / 4), dim3(256), 0, p->stream,
                       a->d_ghosts, reinterpret_cast<int*>(base + o_ghost_task), a->nghosts,
                       a->max_cells, a->d_gmap);
  if (rc == PC_OK) rc = amr_device_tables(a, true);
  if (rc != PC_OK) {
    amr_free(a);
    delete a;
    return rc;
  }
  *out = a;
  return PC_OK;
}

}  // extern "C"

namespace {

AmrPlanDev amr_plan(const pc_amr* a) {
  return AmrPlanDev{a->list,   a->max_waves, a->max_cells, a->d_blocks,
                    a->d_gmap, a->d_ghosts,  a->d_walls,   a->d_wall_dims};
}

// Pinned host memory of at least n doubles for a call's results, and its
// device address; the call waits for the GPU before it reads them.
int amr_host_buffer(pc_pool* p, size_t n) {
  if (n <= p->amr_host_cap) return PC_OK;
  if (p->h_amr) HIPCHK(hipHostFree(p->h_amr));
  p->h_amr = nullptr;
  p->amr_host_cap = 0;
  const size_t cap = std::max<size_t>(2 * n, 4096);
  HIPCHK(hipHostMalloc(reinterpret_cast<void**>(&p->h_amr), cap * sizeof(double),
                       hipHostMallocMapped | hipHostMallocCoherent));
  HIPCHK(hipHostGetDevicePointer(reinterpret_cast<void**>(&p->d_amr_host), p->h_amr, 0));
  p->amr_host_cap = cap;
  return PC_OK;
}

// The end time of the steps to come, on the device (it stays from call to
// call).
int amr_set_end(pc_amr* a, double end_time) {
  if (std::memcmp(&a->h_clock.end_time, &end_time, sizeof(double)) == 0) return PC_OK;
  HIPCHK(hipMemcpyAsync(&a->d_clock->end_time, &end_time, sizeof(double),
                        hipMemcpyHostToDevice, a->pool->stream));
  a->h_clock.end_time = end_time;
  return PC_OK;
}

template <int R, int SOLVER, bool LTS>
void amr_launch_segments(pc_amr* a, Fields F, int cur, AmrClock* host) {
  pc_pool* p = a->pool;
  const AmrPlanDev A = amr_plan(a);
  const dim3 b(64 * a->max_waves);
  if (LTS && a->max_waves <= 8) {
    hipLaunchKernelGGL((k_lts_leaves<R, SOLVER>), dim3(a->nblocks), b, 0, p->stream, A, F, cur,
                       a->d_clock, a->lts);
    return;
  }
  if (!LTS && a->max_waves <= 8)
    hipLaunchKernelGGL((k_amr_fill<R, SOLVER, false, 512>), dim3(a->nblocks), b, 0, p->stream, A,
                       F, cur, a->d_clock, a->d_cfl, a->lts);
  else
    hipLaunchKernelGGL((k_amr_fill<R, SOLVER, LTS, 1024>), dim3(a->nblocks), b, 0, p->stream, A,
                       F, cur, a->d_clock, a->d_cfl, a->lts);
  const double* cfl = a->d_cfl;
  int ncfl = a->nblocks;
  if (!LTS && ncfl > kCflFold) {
    hipLaunchKernelGGL(k_cfl_fold, dim3(1), dim3(1024), 0, p->stream, a->d_cfl, ncfl,
                       a->d_cfl + a->nblocks);
    cfl = a->d_cfl + a->nblocks;
    ncfl = 1;
  }
  hipLaunchKernelGGL((k_amr_update<R, SOLVER, LTS>), dim3(a->nsegs / kSegWaves + 1),
                     dim3(64 * kSegWaves), 0, p->stream, A, F, cur, a->d_clock, a->d_clock_next,
                     host, cfl, ncfl, a->lts);
}

template <bool LTS>
void amr_launch_leaves(pc_amr* a, Fields F, int cur, AmrClock* host = nullptr) {
  if (a->pool->solver) {
    if (a->seg_rows == 2)
      amr_launch_segments<2, 1, LTS>(a, F, cur, host);
    else
      amr_launch_segments<4, 1, LTS>(a, F, cur, host);
  } else {
    if (a->seg_rows == 2)
      amr_launch_segments<2, 0, LTS>(a, F, cur, host);
    else
      amr_launch_segments<4, 0, LTS>(a, F, cur, host);
  }
}

template <bool LTS>
void amr_launch_restrict(pc_amr* a, Fields F, int cur) {
  pc_pool* p = a->pool;
  if (a->nvblocks == 0) return;
  if (a->d_contribs)
    hipLaunchKernelGGL(k_amr_restrict<LTS>, dim3(a->nvblocks), dim3(256), 0, p->stream,
                       a->d_vblocks, a->d_xptr, a->d_contribs, a->d_leaves, F, cur, a->d_clock,
                       a->lts);
  else
    hipLaunchKernelGGL(k_amr_restrict_pairs<LTS>, dim3(a->nvblocks), dim3(256), 0, p->stream,
                       a->d_vblocks, a->d_cptr, a->d_cpairs, a->d_pairs, p->d_pd, F, cur,
                       a->d_clock, a->lts);
}

int amr_launch_step(pc_amr* a, Fields F, int cur, AmrClock* host) {
  pc_pool* p = a->pool;
  amr_launch_restrict<false>(a, F, cur);
  amr_launch_leaves<false>(a, F, cur, host);
  HIPCHK(hipGetLastError());
  std::swap(a->d_clock, a->d_clock_next);
  return PC_OK;
}

// One grid iteration with local time stepping: advance flags from the
// clocks at its start; restriction of every leaf on its own interval; the
// ghost faces of the advancing leaves (every neighbour read before any leaf
// changes); their uNew -> uOld, walls, speeds and steps; update and clocks.
int amr_launch_lts(pc_amr* a, Fields F, int cur) {
  pc_pool* p = a->pool;
  const int nl = (int)a->leaves.size();
  const AmrLts& L = a->lts;
  const int nv = (int)a->vleaves.size();
  if (a->d_neighbours) {
    hipLaunchKernelGGL(k_lts_flags_block, dim3((nl + 255) / 256), dim3(256),
                       std::max(nv, 1) * sizeof(double), p->stream, a->d_leaves, nl,
                       a->d_neighbours, a->d_vleaf, a->d_vowner, a->npairs, nv, a->d_rptr,
                       a->d_rsrc, a->d_clock, L);
  } else {
    if (nv > 0)
      hipLaunchKernelGGL(k_lts_virtual_ends, dim3((nv + 3) / 4), dim3(256), 0, p->stream,
                         a->d_vptr, a->d_vleaf, nv, L, a->d_vend);
    hipLaunchKernelGGL(k_lts_flags, dim3((nl + 255) / 256), dim3(256), 0, p->stream,
                       a->d_leaves, nl, a->d_nptr, a->d_nbr, a->d_vend, a->d_vidx, a->d_rptr,
                       a->d_rsrc, a->d_clock, L);
  }
  amr_launch_restrict<true>(a, F, cur);
  const int ncells = a->nblocks * a->max_cells;
  if (ncells > 0)
    hipLaunchKernelGGL(k_lts_ghosts, dim3((ncells + 255) / 256), dim3(256), 0, p->stream,
                       a->d_gmap, a->max_cells, ncells, a->d_ghosts, F, cur, a->d_clock, L);
  amr_launch_leaves<true>(a, F, cur);
  HIPCHK(hipGetLastError());
  return PC_OK;
}

}  // namespace

extern "C" {

int pc_amr_lts_init(pc_amr* a, const int32_t* nptr, const int32_t* nbr) {
  if (!a || !nptr || (nptr[a->leaves.size()] > 0 && !nbr))
    return fail(PC_E_INVALID, "invalid argument");
  pc_pool* p = a->pool;
  hipSetDevice(p->device);
  CHK(prepare(p));
  CHK(amr_follow_slots(a));
  const int nl = (int)a->leaves.size();
  std::vector<char> role(p->slots.size(), 0);
  for (int s : a->leaves) role[s] = 1;
  for (int s : a->virtuals) role[s] = 2;
  std::vector<int> np(nptr, nptr + nl + 1), nb;
  if (np[0] != 0) return fail(PC_E_INVALID, "neighbour lists must start at 0");
  for (int k = 0; k < nl; ++k) {
    if (np[k + 1] < np[k]) return fail(PC_E_INVALID, "neighbour list offsets must not decrease");
    for (int j = np[k]; j < np[k + 1]; ++j) {
      const int q = nbr[j];
      if (q < 0 || q >= (int)role.size() || !role[q])
        return fail(PC_E_INVALID, "a neighbour is not a patch of the plan");
      nb.push_back(role[q] == 1 ? q : -1 - q);
    }
  }
  std::vector<int> vptr{0}, vleaf;
  for (const auto& v : a->vleaves) {
    vleaf.insert(vleaf.end(), v.begin(), v.end());
    vptr.push_back((int)vleaf.size());
  }
  const size_t ns = p->slots.size();
  std::vector<double> t(ns, 0.0), dt(ns, 0.0);
  for (int s : a->leaves) slot_clock(p, s, &t[s], &dt[s]);
  void* old[] = {a->lts.t,   a->lts.dt,   a->lts.adv, a->lts.stepdt, a->lts.iter, a->lts.steps,
                 a->lts.itn, a->lts.need, a->d_vidx,  a->d_vptr,     a->d_vleaf,  a->d_nptr,
                 a->d_nbr,   a->d_rptr,   a->d_rsrc, a->d_vowner, a->d_neighbours, a->d_vend};
  for (void* q : old) hipFree(q);
  a->lts = AmrLts{};
  a->d_vidx = a->d_vptr = a->d_vleaf = a->d_nptr = a->d_nbr = nullptr;
  a->d_rptr = a->d_rsrc = a->d_vowner = a->d_neighbours = nullptr;
  a->d_vend = nullptr;
  CHK(amr_upload(&a->lts.t, t));
  CHK(amr_upload(&a->lts.dt, dt));
  CHK(amr_upload(&a->lts.adv, std::vector<int>(ns, 0)));
  CHK(amr_upload(&a->lts.stepdt, std::vector<double>(ns, 0.0)));
  CHK(amr_upload(&a->lts.iter, std::vector<int>(1, 0)));
  CHK(amr_upload(&a->lts.steps, std::vector<unsigned long long>(1, 0)));
  std::vector<int> vidx(ns, -1);
  for (size_t v = 0; v < a->virtuals.size(); ++v) vidx[a->virtuals[v]] = (int)v;
  // per leaf the virtual patches its ghost faces read
  std::vector<int> lidx(ns, -1), rptr{0}, rsrc;
  for (int k = 0; k < nl; ++k) lidx[a->leaves[k]] = k;
  std::vector<std::vector<int>> reads(nl);
  for (const AmrGhost& g : a->h_ghosts)
    if (g.kind == kAmrTransferVirtual) reads[lidx[g.dst]].push_back(g.src);
  for (int k = 0; k < nl; ++k) {
    rsrc.insert(rsrc.end(), reads[k].begin(), reads[k].end());
    rptr.push_back((int)rsrc.size());
  }
  CHK(amr_upload(&a->d_rptr, rptr));
  CHK(amr_upload(&a->d_rsrc, rsrc));
  CHK(amr_upload(&a->lts.itn, std::vector<int>(1, 1)));
  CHK(amr_upload(&a->lts.need, std::vector<int>(ns, 0)));
  CHK(amr_upload(&a->d_vleaf, vleaf));
  a->npairs = (int)vleaf.size();
  int most = 0;
  for (int k = 0; k < nl; ++k) most = std::max(most, np[k + 1] - np[k]);
  if (most <= kLtsNeighbours && a->virtuals.size() <= kLtsBlockVirtuals &&
      a->npairs <= kLtsBlockPairs) {
    // what k_lts_flags_block reads
    std::vector<int> vowner(vleaf.size());
    for (size_t v = 0; v + 1 < vptr.size(); ++v)
      std::fill(vowner.begin() + vptr[v], vowner.begin() + vptr[v + 1], (int)v);
    CHK(amr_upload(&a->d_vowner, vowner));
    std::vector<int> t8((size_t)nl * kLtsNeighbours);
    for (int k = 0; k < nl; ++k)
      for (int j = 0; j < kLtsNeighbours; ++j) {
        const int e = np[k] + j < np[k + 1] ? nb[np[k] + j] : a->leaves[k];
        t8[(size_t)k * kLtsNeighbours + j] = e >= 0 ? e : -1 - vidx[-1 - e];
      }
    CHK(amr_upload(&a->d_neighbours, t8));
  } else {
    // what k_lts_virtual_ends and k_lts_flags read
    CHK(amr_upload(&a->d_vidx, vidx));
    CHK(amr_upload(&a->d_vptr, vptr));
    CHK(amr_upload(&a->d_nptr, np));
    CHK(amr_upload(&a->d_nbr, nb));
    CHK(amr_upload(&a->d_vend, std::vector<double>(a->virtuals.size(), 0.0)));
  }
  a->lts_ready = true;
  return PC_OK;
}

int pc_amr_lts_step(pc_amr* a, int k, double end_time, long long* leaf_steps) {
  if (!a || k < 0) return fail(PC_E_INVALID, "invalid argument");
  if (!a->lts_ready) return fail(PC_E_INVALID, "pc_amr_lts_init has not been called");
  pc_pool* p = a->pool;
  hipSetDevice(p->device);
  CHK(prepare(p));
  CHK(amr_follow_slots(a));
  int cur;
  CHK(amr_cur(a, &cur));
  mark_state_changed(p);
  a->shared_clock = false;
  Fields F = fields_of(p);
  const int nl = (int)a->leaves.size();
  CHK(amr_host_buffer(p, 2 * (size_t)nl + 1));
  CHK(amr_set_end(a, end_time));
  for (int it = 0; it < k; ++it) CHK(amr_launch_lts(a, F, cur));
  hipLaunchKernelGGL(k_lts_report, dim3((nl + 255) / 256), dim3(256), 0, p->stream, a->d_leaves,
                     nl, a->lts, p->d_amr_host);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(p->stream));
  // the leaves' descriptors follow their device clocks
  for (int i = 0; i < nl; ++i) {
    Slot& s = p->slots[a->leaves[i]];
    s.desc.time = p->h_amr[2 * i + 1];
    s.desc.timestep_size = p->h_amr[2 * i + 2];
    s.clock_from_scenario = false;
  }
  unsigned long long n;
  std::memcpy(&n, p->h_amr, sizeof(n));
  if (leaf_steps) *leaf_steps = (long long)n;
  return PC_OK;
}

int pc_amr_step(pc_amr* a, int k, double end_time, double* last_dt) {
  if (!a || k < 0) return fail(PC_E_INVALID, "invalid argument");
  if (!a->shared_clock)
    return fail(PC_E_INVALID, "global steps need every leaf of the plan on one clock");
  pc_pool* p = a->pool;
  hipSetDevice(p->device);
  CHK(prepare(p));
  CHK(amr_follow_slots(a));
  int cur;
  CHK(amr_cur(a, &cur));
  mark_state_changed(p);
  Fields F = fields_of(p);
  CHK(amr_host_buffer(p, sizeof(AmrClock) / sizeof(double)));
  CHK(amr_set_end(a, end_time));
  for (int it = 0; it < k; ++it)
    CHK(amr_launch_step(a, F, cur,
                        it == k - 1 ? reinterpret_cast<AmrClock*>(p->d_amr_host) : nullptr));
  HIPCHK(hipStreamSynchronize(p->stream));
  if (k > 0) std::memcpy(&a->h_clock, p->h_amr, sizeof(AmrClock));
  const AmrClock& c = a->h_clock;
  // the leaves' descriptors follow the device clock (as pc_solve_timestep
  // would have left them)
  for (int s : a->leaves) {
    p->slots[s].desc.time = c.time;
    p->slots[s].desc.timestep_size = c.dt;
    p->slots[s].clock_from_scenario = false;
  }
  a->last_dt = (k > 0 && c.advance) ? c.bound : 0.0;
  if (last_dt) *last_dt = a->last_dt;
  return PC_OK;
}

int pc_amr_clock(pc_amr* a, double* time, double* timestep_size, long long* steps) {
  if (!a) return fail(PC_E_INVALID, "invalid argument");
  const AmrClock& c = a->h_clock;  // every step call has brought it back
  if (time) *time = c.time;
  if (timestep_size) *timestep_size = c.dt;
  if (steps) *steps = c.steps;
  return PC_OK;
}

// Face, corner and wall entries of every leaf of a tree of patches with
// refinement factor 3 (host only, no device work): the rows pc_amr_create
// takes.  Patch k has level[k] >= 1 and index (ij[2k], ij[2k+1]) on its
// level; level 1 is a px x py grid.  For each leaf in `leaves` order
// (indices into the patch arrays): its four faces x-, x+, y-, y+ (a face
// outside the domain is a wall), then its four corners (-,-), (-,+), (+,-),
// (+,+) (skipped outside the domain); a face or corner is a transfer from
// the patch of the leaf's level there, else an interpolation from the
// nearest coarser patch covering it (the compositor's choice,
// GhostLayerCompositor.cpp:280-320, GhostlayerCompositorFunctors.cpp:87-141);
// then its walls in the order left, top, right, bottom
// (SolveTimestep.cpp:94-131).  Entries name patches by handle[k].
int pc_amr_face_plan(int px, int py, int n, int npatch, const int32_t* level,
                     const int32_t* ij, const int32_t* handle, const int32_t* leaves,
                     int nleaves, pc_amr_ghost* ghosts, int cap_ghosts, int* nghosts,
                     pc_amr_wall* walls, int cap_walls, int* nwalls) {
  if (px < 1 || py < 1 || n < 1 || npatch < 0 || nleaves < 0 || !nghosts || !nwalls ||
      (npatch && (!level || !ij || !handle)) || (nleaves && !leaves))
    return fail(PC_E_INVALID, "invalid argument");
  // index grid of every level: px 3^(l-1) x py 3^(l-1) patches
  constexpr int kMaxLevel = 12;
  long long gw[kMaxLevel + 1][2];
  for (int l = 1; l <= kMaxLevel; ++l) {
    gw[l][0] = l == 1 ? px : 3 * gw[l - 1][0];
    gw[l][1] = l == 1 ? py : 3 * gw[l - 1][1];
  }
  // patch lookup per level: a dense table where the level's grid is small
  // against the patch count, else a hash map (25 bits per index in its key)
  auto key = [](long long l, long long i, long long j) { return (l << 50) | (i << 25) | j; };
  std::unordered_map<long long, int> at;
  std::vector<int> dense[kMaxLevel + 1];
  int nat = 0;
  for (int k = 0; k < npatch; ++k) {
    const int l = level[k];
    if (l < 1 || l > kMaxLevel || ij[2 * k] < 0 || ij[2 * k + 1] < 0 ||
        ij[2 * k] >= gw[l][0] || ij[2 * k + 1] >= gw[l][1] || ij[2 * k] >= (1 << 25) ||
        ij[2 * k + 1] >= (1 << 25))
      return fail(PC_E_INVALID, "invalid patch level or index");
  }
  const long long dense_cap = 16LL * npatch + 65536;
  for (int k = 0; k < npatch; ++k) {
    const int l = level[k];
    if (dense[l].empty() && gw[l][0] <= dense_cap / gw[l][1])
      dense[l].assign(gw[l][0] * gw[l][1], -1);
    if (!dense[l].empty())
      dense[l][ij[2 * k] * gw[l][1] + ij[2 * k + 1]] = k;
    else
      ++nat;
  }
  if (nat) {
    at.reserve((size_t)nat * 2);
    for (int k = 0; k < npatch; ++k)
      if (dense[level[k]].empty()) at[key(level[k], ij[2 * k], ij[2 * k + 1])] = k;
  }
  auto find = [&](int lev, long long i, long long j) {
    if (!dense[lev].empty()) return dense[lev][i * gw[lev][1] + j];
    if (!nat) return -1;
    auto it = at.find(key(lev, i, j));
    return it != at.end() ? it->second : -1;
  };
  // the patch at (lev, i, j), else the nearest coarser one covering it;
  // -1 outside the domain or where nothing covers it
  auto covering = [&](int lev, long long i, long long j) {
    if (i < 0 || j < 0 || i >= gw[lev][0] || j >= gw[lev][1]) return -1;
    for (; lev >= 1; --lev, i /= 3, j /= 3) {
      const int k = find(lev, i, j);
      if (k >= 0) return k;
    }
    return -1;
  };
  const int steps[4][2] = {{-1, 0}, {1, 0}, {0, -1}, {0, 1}};  // x-, x+, y-, y+
  const int geom[4][6] = {  // size, source offset, destination offset per face
      {1, n, n - 1, 0, -1, 0}, {1, n, 0, 0, n, 0}, {n, 1, 0, n - 1, 0, -1}, {n, 1, 0, 0, 0, n}};
  const int corners[4][2] = {{-1, -1}, {-1, 1}, {1, -1}, {1, 1}};
  const int wall_face[4] = {0, 3, 1, 2};  // left, top, right, bottom as face indices
  int ng = 0, nw = 0;
  for (int li = 0; li < nleaves; ++li) {
    const int p = leaves[li];
    if (p < 0 || p >= npatch) return fail(PC_E_INVALID, "invalid leaf index");
    const int lev = level[p];
    const long long i = ij[2 * p], j = ij[2 * p + 1];
    const long long wx = gw[lev][0], wy = gw[lev][1];
    bool wall[4];
    auto emit = [&](int src, int sx, int sy, int sox, int soy, int dox, int doy) {
      if (ghosts && ng < cap_ghosts) {
        pc_amr_ghost& g = ghosts[ng];
        g.kind = level[src] == lev ? 0 : 1;
        g.src = handle[src];
        g.dst = handle[p];
        g.size[0] = sx;
        g.size[1] = sy;
        g.src_offset[0] = sox;
        g.src_offset[1] = soy;
        g.dst_offset[0] = dox;
        g.dst_offset[1] = doy;
      }
      ++ng;
    };
    for (int f = 0; f < 4; ++f) {
      const long long qi = i + steps[f][0], qj = j + steps[f][1];
      wall[f] = qi < 0 || qj < 0 || qi >= wx || qj >= wy;
      if (wall[f]) continue;
      const int src = covering(lev, qi, qj);
      if (src < 0) return fail(PC_E_INVALID, "face region not covered");
      const int* g = geom[f];
      emit(src, g[0], g[1], g[2], g[3], g[4], g[5]);
    }
    for (const auto& c : corners) {
      const int src = covering(lev, i + c[0], j + c[1]);
      if (src < 0) continue;  // outside the domain: the walls fill it
      emit(src, 1, 1, c[0] == -1 ? n - 1 : 0, c[1] == -1 ? n - 1 : 0, c[0] == -1 ? -1 : n,
           c[1] == -1 ? -1 : n);
    }
    for (int w = 0; w < 4; ++w) {
      const int f = wall_face[w];
      if (!wall[f]) continue;
      if (walls && nw < cap_walls) {
        walls[nw].slot = handle[p];
        walls[nw].dimension = f / 2;
        walls[nw].upper = f % 2;
      }
      ++nw;
    }
  }
  *nghosts = ng;
  *nwalls = nw;
  if ((ghosts && ng > cap_ghosts) || (walls && nw > cap_walls))
    return fail(PC_E_INVALID, "output capacity too small");
  return PC_OK;
}

int pc_amr_destroy(pc_amr* a) {
  if (!a) return fail(PC_E_INVALID, "invalid argument");
  hipSetDevice(a->pool->device);
  hipStreamSynchronize(a->pool->stream);
  amr_free(a);
  delete a;
  return PC_OK;
}

}  // extern "C"
