// One kernel for the boundary of a stage: the ghost layers (k_ghost) and the records' increments (k_bcrec), one thread
// per record that has either to do.
//
// The increments of viscous connection and symmetry records read ghost cells of other faces (the transverse neighbours
// of a cell on a block edge), which made the two kernels a chain.  Here such a neighbour is read from the interior cell
// that its own record copies (BcNbr holds the rows), or, behind mirror and cubic ghosts, formed again with that record's
// statements (ghost1).  No record then reads a ghost that another stores, and they need no order: along its normal a
// planned record that reads its cell's neighbour (connections, symmetry, walls, far field) has a block of two cells or
// more, so that the neighbour is an interior cell (plan_boundary).
// A record's own layers stay in registers between the ghost store and the flux.
//
// The Euler increment (with the ghosts) and the viscous one of a record are two threads of different workgroups: the
// two share little but loads, and at small sizes a launch lasts as long as one thread's chain.
//
// What bounds it: the chain of one record (loads, the flux) at the sizes where launches count, the HBM lines of the
// strided planes at the large ones.  The records are planned once per case (BcPlan): rows and offsets ready, records of
// one kind and direction together, so that a wavefront runs one closure with the direction known at compile time (with
// the direction a run-time value the gradient arrays lived in scratch memory), and none for the faces whose ghosts
// nothing reads (bc_dead).  A stage's boundary took 204 us and takes 146 on the 256^3 Taylor-Green case, 27 -> 11.6 at 48^3,
// 139 -> 8.2 on a 1023^2 Riemann problem, 9.8 -> 5.4 on a shock tube of 1000 cells; three one-thread launches a step go
// with it (StepBegin).
#pragma once

#include "mose_kernels.hpp"

namespace mose {

struct BcPlan {
  int c, src, fg, pos;       // the cell's row, the donor's row, the face in fm<dir>, the place in the increment planes
  int e, meta, b, bs;        // the record, the bits below, its block and the donor's
};
// meta: type (4 bits), direction 0..2 (2), odd face (1), zero-gradient ghosts (1), cubic ghosts (1), then which
// transverse neighbours ghost1 forms: the cell's -b, +b, -c, +c (4) and the donor's (4); then the donor's inward axis
// (2) and its sign (1)
enum : int { BCP_DIR = 4, BCP_ODD = 6, BCP_ZG = 7, BCP_CUB = 8, BCP_EDGE = 9, BCP_DEDGE = 13, BCP_IN = 17 };
// viscous records: the rows of the transverse neighbours in the order of the edge bits; where ghost1 forms one, its
// boundary face as -(place in the increment planes) - 1
struct BcNbr {
  int r[8];
};

// The geometry of a record in plan order, value q of record t at [q n + t]: the face's normal and area, the four lengths of
// the face's stencil (both ghosts, the cell, its interior neighbour) and, for viscous connections, the metric averaged
// over the face's two cells, 0.5 (m(cell) + m(ghost)), entry (a, b) at BCG_M + a + 3 b.  Read from the geometry arrays,
// every value of an i-face record is a cache line of its own (26 lines a record).
enum : int { BCG_N = 0, BCG_AREA = 3, BCG_DL = 4, BCG_M = 8, BCG_INVISCID = 8, BCG_VISCOUS = 17 };

__device__ __forceinline__ int64_t bcp_in(const CaseDev& C, const BcPlan& p) {   // row step to the interior neighbour
  const int d = (p.meta >> BCP_DIR) & 3;
  const mose_blk B = C.blk[p.b];
  const int64_t st = d == 0 ? 1 : (d == 1 ? (int64_t)B.pi : (int64_t)B.pi * B.pj);
  return ((p.meta >> BCP_ODD) & 1) ? st : -st;
}

// once per case: the geometry of the plan's records
static __global__ void __launch_bounds__(64) k_bc_geometry(CaseDev C, const BcPlan* plan, int n, double* geo) {
  const int t = blockIdx.x * 64 + threadIdx.x;
  if (t >= n) return;
  const BcPlan p = plan[t];
  const int d = (p.meta >> BCP_DIR) & 3;
  const double* fm = d == 0 ? C.fm1 : (d == 1 ? C.fm2 : C.fm3);
  const int64_t N = n, c = p.c, in = bcp_in(C, p);
  for (int q = 0; q < 4; ++q) geo[q * N + t] = fm[4 * (int64_t)p.fg + q];
  const double* dlp = C.dl + (int64_t)d * C.NC;
  geo[BCG_DL * N + t] = dlp[c - 2 * in];
  geo[(BCG_DL + 1) * N + t] = dlp[c - in];
  geo[(BCG_DL + 2) * N + t] = dlp[c];
  geo[(BCG_DL + 3) * N + t] = dlp[c + in];
  if (!C.visc) return;
  for (int q = 0; q < 9; ++q) geo[(BCG_M + q) * N + t] = 0.5 * (C.m[9 * c + q] + C.m[9 * (c - in) + q]);
}

// The part of a step's start that the first stage's boundary kernel does (one thread): dt and its history from the
// minimum that the last stage of the step before left, and the slot made ready for this step's.
struct StepBegin {
  unsigned long long* dtnext;   // null: not a step's first stage
  double *dt, *hist;
  int *pos, cap;
};

__device__ __forceinline__ int64_t bc_stride(const mose_blk& B, int code) {   // axis and sign bits of meta
  const int64_t st = (code & 3) == 0 ? 1 : ((code & 3) == 1 ? (int64_t)B.pi : (int64_t)B.pi * B.pj);
  return (code & 4) ? -st : st;
}

// The first ghost layer behind the boundary face at `pos` of the increment planes, where its record mirrors or
// extrapolates: the values that the record stores
template <int NS, int NR>
__device__ __forceinline__ void ghost1(const CaseDev& C, const int* recof, int pos, double* q) {
  using V = Vars<NS, NR>;
  const mose_bc_record& r = C.rec[recof[pos]];
  const mose_blk B = C.blk[r.b];
  const double* P = C.Pin;
  const int64_t NC = C.NC, c = row(B, r.i, r.j, r.k);
  if (r.typ == MOSE_BC_SYMMETRY) {
    double nx, ny, nz, area;
    rec_face(C, B, r, nx, ny, nz, area);
#pragma unroll
    for (int s = 0; s < V::nprim; ++s) q[s] = P[s * NC + c];
    const double udn = q[V::nu] * nx + q[V::nv] * ny + q[V::nw] * nz;
    q[V::nu] = q[V::nu] - 2.0 * udn * nx;
    q[V::nv] = q[V::nv] - 2.0 * udn * ny;
    q[V::nw] = q[V::nw] - 2.0 * udn * nz;
    return;
  }
  const int dir = (r.f + 1) / 2 - 1;
  const int64_t st = dir == 0 ? 1 : (dir == 1 ? (int64_t)B.pi : (int64_t)B.pi * B.pj), in = (r.f & 1) ? st : -st;
#pragma unroll
  for (int s = 0; s < V::nprim; ++s) q[s] = 3.0 * P[s * NC + c] - 3.0 * P[s * NC + c + in] + P[s * NC + c + 2 * in];
}

// Both neighbours of a cell along one transverse direction
template <int NS, int NR>
__device__ __forceinline__ void bc_pair(const CaseDev& C, const int* recof, int rm, int rp, unsigned edge, double* qm,
                                        double* qp) {
  using V = Vars<NS, NR>;
  const int64_t NC = C.NC;
#pragma unroll
  for (int s = 0; s < V::nprim; ++s) {
    qm[s] = C.Pin[s * NC + (rm < 0 ? 0 : rm)];
    qp[s] = C.Pin[s * NC + (rp < 0 ? 0 : rp)];
  }
  if (edge & 1u) ghost1<NS, NR>(C, recof, -rm - 1, qm);
  if (edge & 2u) ghost1<NS, NR>(C, recof, -rp - 1, qp);
}

// the values that the record gradients difference: Y, u, v, w, T and nu~ per unit density
template <int NS, int NR>
__device__ __forceinline__ void bc_vals(const mose_dtab& T, const double* q, double* w) {
  using V = Vars<NS, NR>;
  const double rho = rho_sum<NS>(q), rg = f_Rtot<NS>(T, q);
#pragma unroll
  for (int s = 0; s < NS; ++s) w[s] = q[s] / rho;
#pragma unroll
  for (int s = V::nu; s <= V::nw; ++s) w[s] = q[s];
  w[V::np] = q[V::np] / (rho * rg);
#pragma unroll
  for (int s = V::nt; s < V::nprim; ++s) w[s] = q[s] / rho;
}

// The ghosts and the Euler increment of one record of direction D
template <int NS, int NR, int D>
__device__ __forceinline__ void bc_euler(const CaseDev& C, const BcPlan& p, const double* geo, int64_t N) {
  using V = Vars<NS, NR>;
  constexpr int NP = V::nprim;
  const mose_dtab& T = *C.tab;
  const double* P = C.Pin;
  double* Pg = C.Pg;
  const int64_t NC = C.NC, c = p.c;
  const int typ = p.meta & 15, modfm = (p.meta >> BCP_ODD) & 1, gstep = 2 * modfm - 1, modfm2 = 1 - 2 * modfm;
  const mose_blk B = C.blk[p.b];
  const int64_t st = D == 0 ? 1 : (D == 1 ? (int64_t)B.pi : (int64_t)B.pi * B.pj);
  const int64_t in = gstep * st;       // to the interior neighbour; ghost g lies at c - g in
  double e1[NP];
#pragma unroll
  for (int s = 0; s < NP; ++s) e1[s] = 0.0;

  if (typ == MOSE_BC_CONNECTION) {
    const mose_blk S = C.blk[p.bs];
    const int64_t src = p.src, src2 = src + bc_stride(S, p.meta >> BCP_IN);
    double q1[NP], q2[NP], qc[NP], qi[NP];    // ghost layers 1 and 2, the cell, its interior neighbour
#pragma unroll
    for (int s = 0; s < NP; ++s) {
      q1[s] = P[s * NC + src];
      q2[s] = P[s * NC + src2];
      qc[s] = P[s * NC + c];
      qi[s] = P[s * NC + c + in];
    }
    const double nx = geo[0], ny = geo[N], nz = geo[2 * N], area = geo[BCG_AREA * N];
    // lengths in the face's order (r1, r2 | r3, r4): the ghosts are on the left of an odd face
    const double* dlp = geo + BCG_DL * N;
    const double g2 = dlp[0], g1 = dlp[N], cc = dlp[2 * N], ci = dlp[3 * N];
    const double Dl1 = (modfm ? g2 : ci) * 0.5, Dl2 = (modfm ? g1 : cc) * 0.5, Dl3 = (modfm ? cc : g1) * 0.5,
                 Dl4 = (modfm ? ci : g2) * 0.5;
#pragma unroll
    for (int s = 0; s < NP; ++s) {
      Pg[s * NC + c - in] = q1[s];
      Pg[s * NC + c - 2 * in] = q2[s];
    }
    const double D12 = Dl1 + Dl2, D23 = Dl2 + Dl3, D34 = Dl3 + Dl4;
    double L[NP], R[NP];
    with_limiter(C.lim, [&](auto lim) {
#pragma unroll
      for (int s = 0; s < NP; ++s) {
        const double a1 = modfm ? q2[s] : qi[s], a2 = modfm ? q1[s] : qc[s], a3 = modfm ? qc[s] : q1[s],
                     a4 = modfm ? qi[s] : q2[s];
        const double d21 = (a2 - a1) / D12, d32 = (a3 - a2) / D23, d43 = (a4 - a3) / D34;
        L[s] = a2 + 1.0 * limiter(lim.id, d32, d21) * Dl2;
        R[s] = a3 - 1.0 * limiter(lim.id, d43, d32) * Dl3;
      }
    });
    const double rL = rho_sum<NS>(L), RL = f_Rtot<NS>(T, L), rR = rho_sum<NS>(R), RR = f_Rtot<NS>(T, R);
    const double aL = f_ss<NS>(T, L, L[V::np], rL, RL), aR = f_ss<NS>(T, R, R[V::np], rR, RR);
    const F5 F = riemann<NS>(T, C.rs, C.mco, false, L, L[V::nu], L[V::nv], L[V::nw], L[V::np], aL, rL, R, R[V::nu],
                             R[V::nv], R[V::nw], R[V::np], aR, rR, nx, ny, nz, RL, RR);
    const double su = copysign(0.5, F.r), sL = 0.5 + su, sR = su - 0.5, Fms = F.r * area, m2 = (double)modfm2;
#pragma unroll
    for (int s = 0; s < NS; ++s) e1[s] = m2 * Fms * (sL * L[s] / rL - sR * R[s] / rR);
    e1[V::nu] = m2 * F.u * area; e1[V::nv] = m2 * F.v * area; e1[V::nw] = m2 * F.w * area; e1[V::np] = m2 * F.e * area;
#pragma unroll
    for (int s = V::np + 1; s < NP; ++s) e1[s] = m2 * Fms * (sL * L[s] / rL - sR * R[s] / rR);
  } else {
    double q[NP];
#pragma unroll
    for (int s = 0; s < NP; ++s) q[s] = P[s * NC + c];
    if (typ == MOSE_BC_SYMMETRY) {
      const double nx = geo[0], ny = geo[N], nz = geo[2 * N], area = geo[BCG_AREA * N];
      // Ghost_Symmetry (Lib_Extrapolation.f90:558-587): the first layer only
      const double udn = q[V::nu] * nx + q[V::nv] * ny + q[V::nw] * nz;
      double g[NP];
#pragma unroll
      for (int s = 0; s < NP; ++s) g[s] = q[s];
      g[V::nu] = q[V::nu] - 2.0 * udn * nx;
      g[V::nv] = q[V::nv] - 2.0 * udn * ny;
      g[V::nw] = q[V::nw] - 2.0 * udn * nz;
#pragma unroll
      for (int s = 0; s < NP; ++s) Pg[s * NC + c - in] = g[s];
      const RecCells rc{c, c + in, D + 1, modfm};
      bc_symmetry<NS, NR>(T, P, NC, C.dl, C.lim, C.rs, C.mco, rc, nx, ny, nz, area, e1);
    } else {
      // zero gradient (Ghost_ZG_Extrapolate :590-607), then the cubic of layers g-1, g-2, g-3 (Ghost_Extrapolate :616-640)
      if ((p.meta >> BCP_CUB) & 1) {
        double qa[NP], qb[NP];
#pragma unroll
        for (int s = 0; s < NP; ++s) { qa[s] = P[s * NC + c + in]; qb[s] = P[s * NC + c + 2 * in]; }
#pragma unroll
        for (int s = 0; s < NP; ++s) {
          const double l1 = 3.0 * q[s] - 3.0 * qa[s] + qb[s];
          Pg[s * NC + c - in] = l1;
          Pg[s * NC + c - 2 * in] = 3.0 * l1 - 3.0 * q[s] + qa[s];
        }
      } else if ((p.meta >> BCP_ZG) & 1) {
#pragma unroll
        for (int s = 0; s < NP; ++s) { Pg[s * NC + c - in] = q[s]; Pg[s * NC + c - 2 * in] = q[s]; }
      }
      if (typ == MOSE_BC_NONE) return;   // no flux: its plane entries stay at the zeros of the case's creation
      const double nx = geo[0], ny = geo[N], nz = geo[2 * N], area = geo[BCG_AREA * N];
      if (typ == MOSE_BC_EXTRAPOLATION) {
        // BC_Extrapolation (Lib_BC.f90:1119-1163): the physical flux of the boundary cell
        double Fl[NP];
        double Un = q[V::nu] * nx + q[V::nv] * ny + q[V::nw] * nz, Fm_ = 0.0;
#pragma unroll
        for (int s = 0; s < NS; ++s) { Fl[s] = q[s] * Un * area; Fm_ = Fm_ + Fl[s]; }
        Fl[V::nu] = Fm_ * q[V::nu] + q[V::np] * area * nx;
        Fl[V::nv] = Fm_ * q[V::nv] + q[V::np] * area * ny;
        Fl[V::nw] = Fm_ * q[V::nw] + q[V::np] * area * nz;
        double vmag = sqrt(q[V::nu] * q[V::nu] + q[V::nv] * q[V::nv] + q[V::nw] * q[V::nw]);
        Fl[V::np] = Fm_ * H0<NS>(T, q[V::np], q, vmag);
#pragma unroll
        for (int s = V::np + 1; s < NP; ++s) Fl[s] = q[s] * Un * area;
        double sg = (double)(1 - 2 * modfm);
#pragma unroll
        for (int s = 0; s < NP; ++s) e1[s] = sg * Fl[s];
      } else {
        const mose_bc_record& r = C.rec[p.e];
        const RecCells rc{c, c + in, D + 1, modfm};
        bool closed = false;
        if (typ == MOSE_BC_FARFIELD) {
          const double tv[3] = {r.tvec[0], r.tvec[1], r.tvec[2]};
          closed = !bc_farfield<NS, NR>(T, P, NC, C.lim, C.rs, C.mco, C.ff[r.ff], tv, rc, nx, ny, nz, area, e1);
        }
        if (typ != MOSE_BC_FARFIELD || closed)
          bc_symmetry<NS, NR>(T, P, NC, C.dl, C.lim, C.rs, C.mco, rc, nx, ny, nz, area, e1);
      }
    }
  }
#pragma unroll
  for (int s = 0; s < NP; ++s) C.binc[(int64_t)s * C.NBP + p.pos] = e1[s];
}

// The viscous increment of a connection, symmetry or wall record of direction D
template <int NS, int NR, int D>
__device__ __forceinline__ void bc_viscous(const CaseDev& C, const int* recof, const BcPlan& p, const BcNbr* nbr,
                                           const double* geo, int64_t N) {
  using V = Vars<NS, NR>;
  constexpr int NP = V::nprim;
  constexpr int ib = D == 0 ? 1 : 0, ic = D == 2 ? 1 : 2;
  const mose_dtab& T = *C.tab;
  const double* P = C.Pin;
  const int64_t NC = C.NC, c = p.c;
  const int typ = p.meta & 15, modfm = (p.meta >> BCP_ODD) & 1, gstep = 2 * modfm - 1, modfm2 = 1 - 2 * modfm;
  if (typ != MOSE_BC_CONNECTION && typ != MOSE_BC_SYMMETRY && typ != MOSE_BC_WALL_ADIABATIC &&
      typ != MOSE_BC_WALL_ISOTHERMAL)
    return;                            // no viscous part: zeros since the case's creation
  const mose_blk B = C.blk[p.b];
  const int64_t st = D == 0 ? 1 : (D == 1 ? (int64_t)B.pi : (int64_t)B.pi * B.pj), in = gstep * st;
  const double nx = geo[0], ny = geo[N], nz = geo[2 * N], area = geo[BCG_AREA * N];
  const RecCells rc{c, c + in, D + 1, modfm};
  double e2[NP];
#pragma unroll
  for (int s = 0; s < NP; ++s) e2[s] = 0.0;
  if (typ == MOSE_BC_CONNECTION) {
    // BC_Connection_Visc_lean (Lib_BC.f90:2113-2201): the face gradient on the receiver's and on the donor's side,
    // the two record fluxes averaged
    const BcNbr n = *nbr;
    const unsigned edge = (unsigned)p.meta >> BCP_EDGE & 15u, dedge = (unsigned)p.meta >> BCP_DEDGE & 15u;
    double qc[NP], q1[NP], w0[NP], w1[NP], Pa[NP], Gl[NP][3], Gg[NP][3], qm[NP], qp[NP], wm[NP], wp[NP];
#pragma unroll
    for (int s = 0; s < NP; ++s) { qc[s] = P[s * NC + c]; q1[s] = P[s * NC + p.src]; }
    bc_vals<NS, NR>(T, qc, w0);
    bc_vals<NS, NR>(T, q1, w1);
#pragma unroll
    for (int s = 0; s < NP; ++s) {
      Pa[s] = 0.5 * (qc[s] + q1[s]);
      Gl[s][D] = (w1[s] - w0[s]) * (double)modfm2;
      Gg[s][D] = (w0[s] - w1[s]) * (double)(-modfm2);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      bc_pair<NS, NR>(C, recof, n.r[2 * t], n.r[2 * t + 1], edge >> (2 * t), qm, qp);
      bc_vals<NS, NR>(T, qm, wm);
      bc_vals<NS, NR>(T, qp, wp);
#pragma unroll
      for (int s = 0; s < NP; ++s) Gl[s][t ? ic : ib] = (wp[s] - wm[s]) * 0.5;
      bc_pair<NS, NR>(C, recof, n.r[4 + 2 * t], n.r[5 + 2 * t], dedge >> (2 * t), qm, qp);
      bc_vals<NS, NR>(T, qm, wm);
      bc_vals<NS, NR>(T, qp, wp);
#pragma unroll
      for (int s = 0; s < NP; ++s) Gg[s][t ? ic : ib] = (wp[s] - wm[s]) * 0.5;
    }
    double Mm[3][3];
#pragma unroll
    for (int b = 0; b < 3; ++b)
#pragma unroll
      for (int a = 0; a < 3; ++a)
        Mm[a][b] = geo[(BCG_M + a + 3 * b) * N];
#pragma unroll
    for (int s = 0; s < NP; ++s) {
      const double l0 = Gl[s][0], l1 = Gl[s][1], l2 = Gl[s][2], g0 = Gg[s][0], h1 = Gg[s][1], h2 = Gg[s][2];
#pragma unroll
      for (int kk = 0; kk < 3; ++kk) {
        Gl[s][kk] = l0 * Mm[0][kk] + l1 * Mm[1][kk] + l2 * Mm[2][kk];
        Gg[s][kk] = g0 * Mm[0][kk] + h1 * Mm[1][kk] + h2 * Mm[2][kk];
      }
    }
    const FaceThermo ft = face_thermo<NS>(T, Pa, Pa[V::np], C.vc.prl);
    double Fl[NP], Fg[NP];
    diff_flux_st<NS, NR>(T, C.vc, Gl, Pa, ft, nx, ny, nz, area, Fl);
    diff_flux_st<NS, NR>(T, C.vc, Gg, Pa, ft, nx, ny, nz, area, Fg);
#pragma unroll
    for (int s = 0; s < NP; ++s) e2[s] = -(0.5 * (double)modfm2 * (Fl[s] + Fg[s]));
  } else if (typ == MOSE_BC_SYMMETRY) {
    const BcNbr n = *nbr;
    const unsigned edge = (unsigned)p.meta >> BCP_EDGE & 15u;
    double vn[4][3], qm[NP], qp[NP];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      bc_pair<NS, NR>(C, recof, n.r[2 * t], n.r[2 * t + 1], edge >> (2 * t), qm, qp);
#pragma unroll
      for (int a = 0; a < 3; ++a) { vn[2 * t][a] = qm[V::nu + a]; vn[2 * t + 1][a] = qp[V::nu + a]; }
    }
    bc_sym_visc_n<NS, NR>(T, P, NC, C.m, rc, vn, nx, ny, nz, area, e2);
  } else {
    bc_wall_visc<NS, NR>(T, P, NC, C.m, C.vc.prl, typ, C.rec[p.e].tw, rc, nx, ny, nz, area, e2);
  }
#pragma unroll
  for (int s = 0; s < NP; ++s) C.binc[(int64_t)(NP + s) * C.NBP + p.pos] = e2[s];
}

// 64 records per workgroup; in viscous cases the second half of the grid, a multiple of 8 workgroups after the first (so on
// the same XCD's L2), forms the viscous increments
template <int NS, int NR>
__global__ void __launch_bounds__(64) k_bc(CaseDev C, const BcPlan* plan, const BcNbr* nbr, int n, const int* recof,
                                           const double* geo, int64_t N, StepBegin B) {
  const unsigned half = C.visc ? gridDim.x / 2 : gridDim.x;
  const bool viscous = blockIdx.x >= half;
  const int t = (int)((viscous ? blockIdx.x - half : blockIdx.x) * 64 + threadIdx.x);
  if (B.dtnext && blockIdx.x == 0 && threadIdx.x == 0) {
    const double v = __longlong_as_double((long long)*B.dtnext);
    *B.dt = v;
    const int at = *B.pos;
    if (at < B.cap) B.hist[at] = v;
    *B.pos = at + 1;
    *B.dtnext = (unsigned long long)__double_as_longlong(1e5);   // dtglobal = 1d5 before Compute_dt
  }
  if (t >= n) return;
  const BcPlan p = plan[t];
  const int d = (p.meta >> BCP_DIR) & 3;
  if (viscous) {
    if (d == 0) bc_viscous<NS, NR, 0>(C, recof, p, nbr + t, geo + t, N);
    else if (d == 1) bc_viscous<NS, NR, 1>(C, recof, p, nbr + t, geo + t, N);
    else bc_viscous<NS, NR, 2>(C, recof, p, nbr + t, geo + t, N);
  } else {
    if (d == 0) bc_euler<NS, NR, 0>(C, p, geo + t, N);
    else if (d == 1) bc_euler<NS, NR, 1>(C, p, geo + t, N);
    else bc_euler<NS, NR, 2>(C, p, geo + t, N);
  }
}

}  // namespace mose
