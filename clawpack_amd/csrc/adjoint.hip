// Adjoint of the fused 2D unsplit shallow-water step (FP64, dt fixed) for gfx950, and its C ABI.
//
// lam_out = (d q^{n+1} / d q^n)^T lam_in, with q^{n+1} the step of claw2d_step from q^n.  The
// step is a sum of per-interface contributions (see adjoint.hpp), so its transpose is a sum of
// per-interface reverses, scattered onto the four cells each interface reads.  Kernels:
//   adj_sweeps    both sweep directions in one launch (they are independent).  x part: one
//                 wavefront per (row line, segment of 58 columns); lane = column = the x-interface
//                 on its left.  Each lane computes its interface's Roe split once; the limiter
//                 partners' data and, in reverse, their adjoints travel one lane left or right by
//                 DPP wavefront rotations; the cell adjoint of column c is the sum of the shares of
//                 interfaces c and c+1.  It writes lam_in plus the x-sweep share of every extended
//                 cell (interior + 2 ghost layers) to the workspace's first three (my+4) x (mx+4)
//                 planes.  y part: the same along columns (lane = row position), from tiles of
//                 8 columns in LDS, into the next three planes.
//                 Bound by FP64 issue at 2 wavefronts per SIMD and, from 2048^2 up, by the six
//                 workspace planes.  A wavefront of plain interfaces (adjoint.hpp) takes the short
//                 reverse, about 580 vector instructions where the general one has 820: a reverse
//                 step at 512^2 36.7 -> 30.3 us with it, -> 27.1 with the columns' tiles, -> 26.8
//                 with lambda added here and not in the fold (1024^2 115 -> 77 us, 2048^2 478 -> 351).
//   adj_fold      lam_out = both planes' sum (interior) + the ghost-cell shares folded back to
//                 the interior cells they were copied from (extrap / periodic / wall, with the
//                 wall's sign), in a fixed order (deterministic, no atomics).
// Branches (entropy fix, limiter cases, upwind side, transverse speed signs) are taken as the
// forward took them at q^n.  No counterpart upstream: PyClaw has no adjoint.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <string>

#include "../../include/clawpack_amd.h"
#include "adjoint.hpp"

namespace claw {
int set_error(int code, const char* msg);
int set_hip_error(hipError_t e, const char* where);

namespace adj {

constexpr int kOwnA = 58;  // owned positions per wavefront (3 halo lanes left, 3 right)
constexpr int kWPBA = 4;   // wavefronts per workgroup

// One-lane exchanges as DPP wavefront rotations (VALU moves, no LDS round trip): rotl gives lane i
// the value of lane i-1 and lane 0 that of lane 63; rotr gives lane i the value of lane i+1 and
// lane 63 that of lane 0.  At the sweep kernel's 2 wavefronts per SIMD the crossbar's latency sat
// on the dependency chain: a reverse step ran 3% faster with these than with ds_bpermute.  Every
// call site is in wave-uniform control flow (all 64 lanes active).
template <int CTRL> __device__ __forceinline__ double dpp_rot(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = (int)(b & 0xffffffffLL), hi = (int)(b >> 32);
  const int rlo = __builtin_amdgcn_update_dpp(lo, lo, CTRL, 0xF, 0xF, false);
  const int rhi = __builtin_amdgcn_update_dpp(hi, hi, CTRL, 0xF, 0xF, false);
  return __longlong_as_double(((long long)rhi << 32) | (unsigned int)rlo);
}
constexpr int kDppWaveRor1 = 0x13C, kDppWaveRol1 = 0x134;
__device__ __forceinline__ double rotl(double v) { return dpp_rot<kDppWaveRor1>(v); }
__device__ __forceinline__ double rotr(double v) { return dpp_rot<kDppWaveRol1>(v); }
__device__ __forceinline__ LimD rotl(const LimD& d) {
  LimD o;
  o.a1 = rotl(d.a1); o.a2 = rotl(d.a2); o.a3 = rotl(d.a3);
  o.s1 = rotl(d.s1); o.s3 = rotl(d.s3); o.v = rotl(d.v);
  return o;
}
__device__ __forceinline__ LimD rotr(const LimD& d) {
  LimD o;
  o.a1 = rotr(d.a1); o.a2 = rotr(d.a2); o.a3 = rotr(d.a3);
  o.s1 = rotr(d.s1); o.s3 = rotr(d.s3); o.v = rotr(d.v);
  return o;
}

struct AdjArgs {
  const double* q;
  const double* lam;
  double* ext;
  double* lam_out;
  int mx, my;
  double dtdx, dtdy;
  Method M;
  double sqgm;  // sqrt(g), reduced (plain_lanes)
  int bxl, bxh, byl, byh, rfx, rfy;
  int nseg_x, nseg_y;
};

// state at (x, y) of the extended grid, ghost cells by index mapping, as frame (h, hn, ht)
template <int DIR>
__device__ __forceinline__ void load_q(const AdjArgs& a, int x, int y, double o[3]) {
  bool fx, fy;
  const int ix = bc_src(x, a.mx, a.bxl, a.bxh, fx);
  const int iy = bc_src(y, a.my, a.byl, a.byh, fy);
  const size_t plane = (size_t)a.mx * (size_t)a.my;
  const size_t off = (size_t)iy * (size_t)a.mx + (size_t)ix;
  double c[3];
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    const double v = a.q[(size_t)m * plane + off];
    c[m] = ((fx && m == a.rfx) != (fy && m == a.rfy)) ? -v : v;
  }
  o[0] = c[0];
  o[1] = DIR == 0 ? c[1] : c[2];
  o[2] = DIR == 0 ? c[2] : c[1];
}

// lambda at (x, y) as frame; zero outside the interior (ghost cells receive no update)
template <int DIR>
__device__ __forceinline__ void load_lam(const AdjArgs& a, int x, int y, double o[3]) {
  if (x < 0 || x >= a.mx || y < 0 || y >= a.my) {
    o[0] = o[1] = o[2] = 0.0;
    return;
  }
  const size_t plane = (size_t)a.mx * (size_t)a.my;
  const size_t off = (size_t)y * (size_t)a.mx + (size_t)x;
  const double c0 = a.lam[off], c1 = a.lam[plane + off], c2 = a.lam[2 * plane + off];
  o[0] = c0;
  o[1] = DIR == 0 ? c1 : c2;
  o[2] = DIR == 0 ? c2 : c1;
}

// The reverse of one x- or y-interface per lane: interface p between the cells cL = p-1 (the lane to
// the left) and cR = p, from lambda at (line, p), (line-1, p) and (line+1, p).  o: the adjoint of
// cell p (frame), valid on lanes 3..60.  PL: every interface of lanes 2..62 is plain.
template <int LIM, bool PL>
__device__ __forceinline__ void reverse_iface(const AdjArgs& a, const CellF& cL, const CellF& cR, const WaveF& w,
                                              const double r0[3], const double rm[3], const double rp[3], double r,
                                              double rt, double o[3]) {
  // adjoints of the six output cells: (p-1 | p) x (line-1, line, line+1)
  double bLX[3], bLG1[3], bLG2[3], bRX[3], bRG1[3], bRG2[3];
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    bRX[m] = r0[m];
    bRG1[m] = r0[m] - rm[m];
    bRG2[m] = rp[m] - r0[m];
    bLX[m] = rotl(bRX[m]);
    bLG1[m] = rotl(bRG1[m]);
    bLG2[m] = rotl(bRG2[m]);
  }
  // Interface p is the right limiter partner of interface p-1 and the left one of p+1.
  WaveB Wb;
  CellB Lb, Rb;
  zero(Lb);
  zero(Rb);
  if constexpr (PL) {
    LimD nl, nr, NLb, NRb;
    nl.a2 = rotl(w.a2); nl.a3 = rotl(w.a3); nl.s3 = rotl(w.s3); nl.v = rotl(w.v);
    nr.a1 = rotr(w.a1); nr.a2 = rotr(w.a2); nr.s1 = rotr(w.s1); nr.v = rotr(w.v);
    iface_plain<LIM>(w, nl, nr, bLX, bLG1, bLG2, bRX, bRG1, bRG2, r, rt, Wb, NLb, NRb);
    Wb.a1 += rotl(NRb.a1);
    Wb.a2 += rotl(NRb.a2) + rotr(NLb.a2);
    Wb.a3 += rotr(NLb.a3);
    Wb.s1 += rotl(NRb.s1);
    Wb.s3 += rotr(NLb.s3);
    Wb.v += rotl(NRb.v) + rotr(NLb.v);
  } else {
    // (the method at run time here too: folded into iface_core it made the kernel spill 68 registers)
    const Method& M = a.M;
    const FixF fx = fix_fwd(cL, cR, w, M.g, M.sqg);
    const LimD me = lim_of(w);
    const LimD nl = rotl(me), nr = rotr(me);
    LimD NLb, NRb;
    zero(Wb);
    zero(NLb);
    zero(NRb);
    iface_core(cL, cR, w, fx, nl, nr, bLX, bLG1, bLG2, bRX, bRG1, bRG2, r, rt, M, Wb, NLb, NRb, Lb, Rb);
    add_lim(Wb, rotl(NRb));
    add_lim(Wb, rotr(NLb));
  }
  wave_rev(cL, cR, w, a.M.g, Wb, Lb, Rb);
  // cell p: right cell of interface p, left cell of interface p+1
  CellB tot = Rb;
  tot.h += rotr(Lb.h);
  tot.hn += rotr(Lb.hn);
  tot.ht += rotr(Lb.ht);
  tot.s += rotr(Lb.s);
  tot.P += rotr(Lb.P);
  tot.Q += rotr(Lb.Q);
  if constexpr (!PL) tot.r += rotr(Lb.r);  // only the entropy fix reads 1/sqrt(h)
  cell_rev(cR, tot, o);
}

// The forward Roe split of a lane's interface from its cell's state, then its reverse; `lam` gives the
// three lambda vectors.
template <int LIM, class LAM>
__device__ __forceinline__ void reverse_line(const AdjArgs& a, const double qo[3], double r, double rt, LAM lam,
                                             double o[3]) {
  const CellF cR = cell_fwd(qo[0], qo[1], qo[2]);
  CellF cL;
  cL.h = rotl(cR.h); cL.hn = rotl(cR.hn); cL.ht = rotl(cR.ht); cL.r = rotl(cR.r);
  cL.s = cL.h * cL.r; cL.P = cL.hn * cL.r; cL.Q = cL.ht * cL.r;
  const WaveF w = wave_fwd(cL, cR, a.M.g);
  // lanes whose interface reaches an owned cell (3..60): 3..61, and their partners 2 and 62
  constexpr unsigned long long kNeed = 0x7ffffffffffffffcull;
  double r0[3], rm[3], rp[3];
  if constexpr (LIM > 0) {
    if ((~plain_lanes(cL, cR, w, a.sqgm) & kNeed) == 0ull) {
      lam(r0, rm, rp);
      reverse_iface<LIM, true>(a, cL, cR, w, r0, rm, rp, r, rt, o);
      return;
    }
  }
  lam(r0, rm, rp);
  reverse_iface<LIM, false>(a, cL, cR, w, r0, rm, rp, r, rt, o);
}

// x part: one wavefront per (row line, segment of 58 columns); block `blk` of this part.  The waves
// of a workgroup take adjacent rows of one segment, whose lambda rows they share in the CU's cache.
// It writes lambda plus its share of every extended cell to the workspace's first three planes.  LIM 1 or 4: minmod
// or MC for every wave at order 2 with transverse_waves 2, known at compile time; a wavefront whose
// interfaces are all plain then takes iface_plain.  LIM 0: the method from a.M.
template <int LIM> __device__ __forceinline__ void sweep_rows(const AdjArgs& a, const int blk) {
  const int lane = threadIdx.x & 63;
  const int grp = blk / a.nseg_x, seg = blk - grp * a.nseg_x;
  const int li = grp * kWPBA + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (li >= a.my + 4) return;
  const int line = li - 2;                 // -2 .. my + 1
  const int p = seg * kOwnA - 5 + lane;    // column: lanes 3..60 own
  const bool own = lane >= 3 && lane < 3 + kOwnA && p <= a.mx + 1;
  const int ew = a.mx + 4;
  const size_t eplane = (size_t)ew * (size_t)(a.my + 4);
  double* const ext = a.ext + (size_t)li * ew;
  double o[3] = {0.0, 0.0, 0.0};
  // the forward sweeps rows -1 .. my only
  if (line >= -1 && line <= a.my) {
    double qo[3];
    load_q<0>(a, p, line, qo);
    double lam0[3];
    reverse_line<LIM>(a, qo, a.dtdx, a.dtdy, [&](double* r0, double* rm, double* rp) {
      load_lam<0>(a, p, line, r0);
      load_lam<0>(a, p, line - 1, rm);
      load_lam<0>(a, p, line + 1, rp);
#pragma unroll
      for (int m = 0; m < 3; ++m) lam0[m] = r0[m];
    }, o);
    // the interior's own lambda goes in with this share (load_lam gives 0 outside)
#pragma unroll
    for (int m = 0; m < 3; ++m) o[m] += lam0[m];
  }
  if (own) {
#pragma unroll
    for (int m = 0; m < 3; ++m) ext[(size_t)m * eplane + (size_t)(p + 2)] = o[m];
  }
}

// y part: a workgroup takes COLS adjacent columns of one segment of 58 rows.  Lanes walk a
// column, so the state and lambda of the 64 rows are read row by row (whole pieces of a cache line,
// not one element of 64 lines) into LDS, each wave reverses its columns from there, and the shares
// go back through LDS.  The row stride of both tiles is odd in doubles (no bank conflicts down a
// column).  Workgroups are dealt to the 8 XCDs in turn; each XCD gets consecutive column groups of a
// segment, which share cache lines in its L2.  It writes the workspace's other three planes.
template <int COLS> struct ColTiles {
  static constexpr int kQStride = COLS + 1, kLStride = COLS + 3;
  double q[3][64 * kQStride];    // state in the y frame (h, hv, hu); then the shares
  double lam[3][64 * kLStride];  // columns -1 .. COLS of the group
};
template <int LIM, int COLS>
__device__ __forceinline__ void sweep_cols(const AdjArgs& a, const int blk, const int nblk, ColTiles<COLS>& t) {
  constexpr int kColsY = COLS, kQStride = ColTiles<COLS>::kQStride, kLStride = ColTiles<COLS>::kLStride;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int q8 = nblk >> 3, r8 = nblk & 7, x = blk & 7, i = blk >> 3;
  const int bb = x < r8 ? x * (q8 + 1) + i : r8 * (q8 + 1) + (x - r8) * q8 + i;  // a bijection of [0, nblk)
  const int ngrp = (a.mx + 4 + kColsY - 1) / kColsY;
  const int seg = bb / ngrp, c0 = (bb - seg * ngrp) * kColsY - 2;  // first column of the group
  const int p0 = seg * kOwnA - 5;                                  // row of lane 0
  for (int k = threadIdx.x; k < 64 * kColsY; k += 64 * kWPBA) {
    const int row = k / kColsY, col = k % kColsY;
    double v[3];
    load_q<1>(a, c0 + col, p0 + row, v);
#pragma unroll
    for (int m = 0; m < 3; ++m) t.q[m][row * kQStride + col] = v[m];
  }
  for (int k = threadIdx.x; k < 64 * (kColsY + 2); k += 64 * kWPBA) {
    const int row = k / (kColsY + 2), col = k % (kColsY + 2);
    double v[3];
    load_lam<1>(a, c0 + col - 1, p0 + row, v);
#pragma unroll
    for (int m = 0; m < 3; ++m) t.lam[m][row * kLStride + col] = v[m];
  }
  __syncthreads();
#pragma unroll 1
  for (int k = 0; k < kColsY / kWPBA; ++k) {
    const int col = wv * (kColsY / kWPBA) + k, line = c0 + col;
    double o[3] = {0.0, 0.0, 0.0};
    // the forward sweeps columns -1 .. mx only
    if (line >= -1 && line <= a.mx) {
      double qo[3];
#pragma unroll
      for (int m = 0; m < 3; ++m) qo[m] = t.q[m][lane * kQStride + col];
      reverse_line<LIM>(a, qo, a.dtdy, a.dtdx, [&](double* r0, double* rm, double* rp) {
#pragma unroll
        for (int m = 0; m < 3; ++m) {
          const double* row = t.lam[m] + lane * kLStride + col;
          rm[m] = row[0]; r0[m] = row[1]; rp[m] = row[2];
        }
      }, o);
    }
#pragma unroll
    for (int m = 0; m < 3; ++m) t.q[m][lane * kQStride + col] = o[m];  // this wave's own column
  }
  __syncthreads();
  const int ew = a.mx + 4;
  const size_t eplane = (size_t)ew * (size_t)(a.my + 4);
  double* const ext = a.ext + 3 * eplane;
  for (int k = threadIdx.x; k < kOwnA * kColsY; k += 64 * kWPBA) {
    const int row = 3 + k / kColsY, col = k % kColsY;
    if (p0 + row > a.my + 1 || c0 + col > a.mx + 1) continue;
    const size_t e = (size_t)(p0 + row + 2) * ew + (size_t)(c0 + col + 2);
    ext[e] = t.q[0][row * kQStride + col];
    ext[eplane + e] = t.q[2][row * kQStride + col];  // frame (h, hv, hu) -> (h, hu, hv)
    ext[2 * eplane + e] = t.q[1][row * kQStride + col];
  }
}

// Both sweep directions in one launch: blocks [0, nbx) take the x-sweep lines, the rest the
// y-sweep columns.  The two are independent (each writes its own planes), so they overlap on the
// device instead of running as two dependent launches.
// The reverse steps of a backward pass form one dependent chain, which sets the pass's time; the
// forward recompute of the next checkpoint segment runs beside it on another stream and has slack.
// Both reverse kernels therefore issue at the highest wavefront priority, so that where their
// wavefronts share a SIMD with the recompute's, theirs are picked first (backward -4% on a
// 512 x 512 grid; neither result changes).
template <int LIM, int COLS>
__global__ void __launch_bounds__(64 * kWPBA) __attribute__((amdgpu_waves_per_eu(2))) adj_sweeps(AdjArgs a, int nby) {
  __builtin_amdgcn_s_setprio(3);
  __shared__ ColTiles<COLS> tiles;
  const int b = (int)blockIdx.x;
  if (b < nby) sweep_cols<LIM, COLS>(a, b, nby, tiles);
  else sweep_rows<LIM>(a, b - nby);
}

// extended index k (0..4 = i, -2, -1, n, n+1) along one axis: does its value come from cell i, and
// with the wall's sign flip?  (k = 0 is cell i itself.)
__device__ __forceinline__ bool source_k(int k, int i, int n, int lo, int hi, int& e, bool& fl) {
  e = k == 0 ? i : (k == 1 ? -2 : (k == 2 ? -1 : (k == 3 ? n : n + 1)));
  fl = false;
  if (k == 0) return true;
  return bc_src(e, n, lo, hi, fl) == i;
}

__global__ void __launch_bounds__(256) adj_fold(AdjArgs a) {
  __builtin_amdgcn_s_setprio(3);  // on the backward's critical chain, like adj_sweeps
  // one row per grid line y (no division by mx, which cost more than the sums)
  const int j = (int)blockIdx.y, i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (i >= a.mx) return;
  const size_t cells = (size_t)a.mx * (size_t)a.my, t = (size_t)j * (size_t)a.mx + (size_t)i;
  const int ew = a.mx + 4;
  const size_t eplane = (size_t)ew * (size_t)(a.my + 4);
  const size_t plane = (size_t)cells;
  double acc[3];
#pragma unroll
  for (int m = 0; m < 3; ++m) acc[m] = 0.0;
  const double* const ey_ = a.ext + 3 * eplane;  // the y-sweep's planes
  if (i >= 2 && i < a.mx - 2 && j >= 2 && j < a.my - 2) {
    const size_t eo = (size_t)(j + 2) * ew + (size_t)(i + 2);
#pragma unroll
    for (int m = 0; m < 3; ++m) acc[m] += a.ext[(size_t)m * eplane + eo] + ey_[(size_t)m * eplane + eo];
  } else {
    // fixed order: y candidate outer, x candidate inner
#pragma unroll
    for (int b = 0; b < 5; ++b) {
      int ey;
      bool fy;
      if (!source_k(b, j, a.my, a.byl, a.byh, ey, fy)) continue;
#pragma unroll
      for (int c = 0; c < 5; ++c) {
        int ex;
        bool fx;
        if (!source_k(c, i, a.mx, a.bxl, a.bxh, ex, fx)) continue;
        const size_t eo = (size_t)(ey + 2) * ew + (size_t)(ex + 2);
#pragma unroll
        for (int m = 0; m < 3; ++m) {
          const double v = a.ext[(size_t)m * eplane + eo] + ey_[(size_t)m * eplane + eo];
          acc[m] += ((fx && m == a.rfx) != (fy && m == a.rfy)) ? -v : v;
        }
      }
    }
  }
#pragma unroll
  for (int m = 0; m < 3; ++m) a.lam_out[(size_t)m * plane + t] = acc[m];
}

}  // namespace adj
}  // namespace claw

using namespace claw;
using namespace claw::adj;

static int check_adjoint_desc(const claw2d_desc* d) {
  const int rc = claw2d_validate(d);
  if (rc != 0) return rc;
  if (d->solver != CLAW_SOLVER_SHALLOW_ROE_EFIX)
    return set_error(-20, "the adjoint step is implemented for shallow water (shallow_roe_with_efix) only");
  if (d->dtype != CLAW_FP64) return set_error(-21, "the adjoint step runs in FP64 only");
  if (d->num_aux != 0) return set_error(-23, "the adjoint step takes no aux arrays (no capacity function)");
  return 0;
}

extern "C" {

size_t claw2d_adjoint_workspace_bytes(const claw2d_desc* d) {
  if (check_adjoint_desc(d) != 0) return 0;
  return (size_t)6 * (size_t)(d->mx + 4) * (size_t)(d->my + 4) * sizeof(double);
}

int claw2d_adjoint_step(const claw2d_desc* d, const void* q, const void* lam_in, void* lam_out, void* workspace,
                        double dt, void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  const int rc = check_adjoint_desc(d);
  if (rc != 0) return rc;
  if (!q || !lam_in || !lam_out || !workspace) return set_error(-1, "null device pointer");
  if (!(dt > 0.0)) return set_error(-22, "dt must be positive");
  AdjArgs a;
  a.q = (const double*)q;
  a.lam = (const double*)lam_in;
  a.ext = (double*)workspace;
  a.lam_out = (double*)lam_out;
  a.mx = d->mx;
  a.my = d->my;
  a.dtdx = dt / d->dx;
  a.dtdy = dt / d->dy;
  a.M.g = d->grav;
  a.M.sqg = sqrt(d->grav);
  a.sqgm = sqrt(d->grav) * (1.0 - 1e-12);
  a.M.order = d->order;
  a.M.tw = d->transverse_waves;
  for (int p = 0; p < 3; ++p) a.M.mthlim[p] = d->mthlim[p];
  a.bxl = d->bc_lower[0];
  a.bxh = d->bc_upper[0];
  a.byl = d->bc_lower[1];
  a.byh = d->bc_upper[1];
  a.rfx = d->reflect_index[0];
  a.rfy = d->reflect_index[1];
  a.nseg_x = (d->mx + 4 + kOwnA - 1) / kOwnA;
  a.nseg_y = (d->my + 4 + kOwnA - 1) / kOwnA;
  const long long nbx = (long long)((d->my + 4 + kWPBA - 1) / kWPBA) * a.nseg_x;
  // Columns of a y workgroup: 8 (each wave two, one after the other), or 4 where all the launch's
  // workgroups then start at once (512 at 2 wavefronts per SIMD), which halves the longest
  // (128^2: 10.4 -> 8.7 us; from 401 x 214 up 8 is as fast or faster, 512^2 28.0 -> 27.1 us).
  long long nby = (long long)((d->mx + 4 + 3) / 4) * a.nseg_y;
  const bool narrow = nbx + nby <= 512;
  if (!narrow) nby = (long long)((d->mx + 4 + 7) / 8) * a.nseg_y;
  if (nbx > (1LL << 28) || nby > (1LL << 28)) return set_error(-23, "grid too large for the adjoint launch");
  const bool same = d->mthlim[0] == d->mthlim[1] && d->mthlim[0] == d->mthlim[2];
  const int lim = same && d->order == 2 && d->transverse_waves == 2 ? d->mthlim[0] : 0;
  const dim3 grid((unsigned)(nbx + nby)), block(64 * kWPBA);
  const void* kern = lim == 4   ? (narrow ? (const void*)adj_sweeps<4, 4> : (const void*)adj_sweeps<4, 8>)
                     : lim == 1 ? (narrow ? (const void*)adj_sweeps<1, 4> : (const void*)adj_sweeps<1, 8>)
                                : (narrow ? (const void*)adj_sweeps<0, 4> : (const void*)adj_sweeps<0, 8>);
  int nb = (int)nby;
  void* args[] = {&a, &nb};
  const hipError_t es = hipLaunchKernel(kern, grid, block, args, 0, stream);
  if (es != hipSuccess) return set_hip_error(es, "adjoint launch");
  hipLaunchKernelGGL(adj_fold, dim3((unsigned)((d->mx + 255) / 256), (unsigned)d->my), dim3(256), 0, stream, a);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_hip_error(e, "adjoint launch");
  return 0;
}

}  // extern "C"
