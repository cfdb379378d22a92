// The stage of inviscid one-species cases whose blocks are one cell thick in k (the shock tube, the 2D Riemann problems),
// for both fused paths: FAST with the formulas of mose_stage_fast.hpp, otherwise those of mose_stage.hpp to the bit.
//
// One face per thread, all of a tile's faces at once.  With N = TI TJ cells, threads 0 .. N-1 take the lower i-faces of the
// cells, N .. 2N-1 their lower j-faces (absent in one dimension), the rest the TJ + TI faces on the tile's upper sides:
//   load    the cells and two rim cells along each direction into LDS; the cell's step base and volume into registers
//   faces   the two limited half-slopes from the LDS stencil, the flux into LDS
//   update  threads 0 .. N-1: the face sums, boundary increments, stage update, next dt
//
// The tiles of the general kernels treat the one-cell direction like the others: a three-layer box, two slabs and two
// faces per cell in k, none of which an inviscid plane reads.  Without them a 16 x 8 tile needs 21 KB of LDS in place of
// 51 KB, and the faces take one pass.  A small case is bound by the length of one thread's chain of loads and operations
// (load, face, update), a large one by the FP64 units.
// Stage times, general kernel -> this one (boundary kernel included): shock tube of 1000 cells 22 -> 16 us, Riemann problems of
// 64^2 20 -> 16 us, 1023^2 285 -> 135 us (65 us of it FP64 issue; 180 us with a thread per face there).
#pragma once

#include "mose_stage_fast.hpp"

namespace mose {

template <bool FAST, int RS, bool WIDE>
__global__ void __launch_bounds__(WIDE ? FLAT_THREADS : 256, (!FAST && RS == MOSE_RS_LMROE) ? 3 : 4) k_flat(CaseDev C, StageArgs A, int two) {
  using V = Vars<1, 0>;
  constexpr int NP = V::nprim;
  const int tidx = xcd_tile(blockIdx.x, A.ntiles);
  if (tidx < 0) return;
  extern __shared__ double sm[];
  const int tid = threadIdx.x;
  const Tile tl = A.tiles[tidx];
  const mose_blk B = C.blk[tl.b];
  const mose_dtab& T = *C.tab;
  const int64_t NC = C.NC, sj = B.pi;
  const double* P = C.Pin;
  const int TI = A.TI, TJ = A.TJ, N = TI * TJ, lt = 31 - __clz(TI);     // the tile's sides are powers of two
  const int NX = N + 4 * TJ + (two ? 4 * TI : 0), NI = (TI + 1) * TJ, NF = NI + (two ? TI * (TJ + 1) : 0);
  double* Pl = sm;              // [NP][NX]: the cells a + TI b, then the rims -2, -1, TI, TI + 1 of each row, then of each column
  double* Fb = sm + NP * NX;    // [NP][NF]: the i-faces a + (TI + 1) b, then the j-faces a + TI b

  // ---------------- load ----------------
  const int ca = tid & (TI - 1), cb = tid >> lt;
  const int ci = tl.i0 + ca, cj = tl.j0 + cb;
  const bool mine = tid < N && ci <= B.n1 && cj <= B.n2;
  const int64_t c0 = mine ? row(B, ci, cj, 1) : 0;
  double po[NP], vol = 1.0;
#pragma unroll
  for (int s = 0; s < NP; ++s) po[s] = 0.0;
  if (mine) {
#pragma unroll
    for (int s = 0; s < NP; ++s) po[s] = C.PO[s * NC + c0];
    vol = C.vol[c0];
  }
  for (int q = tid; q < NX; q += blockDim.x) {
    int a, b;
    if (q < N) { a = q & (TI - 1); b = q >> lt; }
    else if (q < N + 4 * TJ) { const int h = q - N, e = h & 3; b = h >> 2; a = e < 2 ? e - 2 : TI + e - 2; }
    else { const int h = q - N - 4 * TJ, e = h >> lt; a = h & (TI - 1); b = e < 2 ? e - 2 : TJ + e - 2; }
    const int i = tl.i0 + a, j = tl.j0 + b;
    if (i > B.n1 + GC || j > B.n2 + GC) continue;
    const int64_t r = row(B, i, j, 1);
    double y[NP];
#pragma unroll
    for (int s = 0; s < NP; ++s) y[s] = P[s * NC + r];
#pragma unroll
    for (int s = 0; s < NP; ++s) Pl[s * NX + q] = y[s];
  }

  // ---------------- faces: the face between the cells a - 1 and a (d = 0) or b - 1 and b (d = 1) ----------------
  const int nface = two ? 2 * N + TJ + TI : N + TJ;
  for (int r0 = 0; r0 < (WIDE ? 1 : nface); r0 += blockDim.x) {
    const int r = r0 + tid;
    int d, a = r & (TI - 1), b = r >> lt;
    if (r < N) d = 0;
    else if (two && r < 2 * N) { d = 1; b -= TJ; }
    else {
      const int e = r - (two ? 2 : 1) * N;
      if (e < TJ) { d = 0; a = TI; b = e; }
      else { d = 1; a = e - TJ; b = TJ; }
    }
    const int i = tl.i0 + a, j = tl.j0 + b;                // the face's upper cell
    const bool face = r < nface && i <= B.n1 && j <= B.n2 && (d == 0 ? i : j) >= 2;
    double dLL = 1.0, dL = 1.0, dR = 1.0, dRR = 1.0, nx = 0.0, ny = 0.0, nz = 0.0, area = 0.0;
    if (face) {
      const double* dlp = C.dl + d * NC + row(B, i, j, 1);
      const int64_t st = d ? sj : 1;
      dLL = dlp[-2 * st]; dL = dlp[-st]; dR = dlp[0]; dRR = dlp[st];
      const double* fm = d ? C.fm2 + 4 * (B.f2off + (i - 1) + (int64_t)B.n1 * (j - 1))
                           : C.fm1 + 4 * (B.f1off + (i - 1) + (int64_t)(B.n1 + 1) * (j - 1));
      nx = fm[0]; ny = fm[1]; nz = fm[2]; area = fm[3];
    }
    if (r0 == 0) __syncthreads();             // the LDS stencil, with the first face's geometry in flight
    if (face) {
      // the stencil's slots: a rim cell e (0, 1 below the tile, 2, 3 above) of the face's row or column, or a tile cell
      const int x = d ? b : a, n = d ? TJ : TI;
      const int c = a + TI * b, st = d ? TI : 1, rim = d ? N + 4 * TJ + a : N + 4 * b, rs = d ? TI : 1;
      const int kLL = x >= 2 ? c - 2 * st : rim + rs * x, kL = x >= 1 ? c - st : rim + rs,
                kR = x < n ? c : rim + 2 * rs, kRR = x < n - 1 ? c + st : rim + rs * (x - n + 3);
      double L[NP], R[NP], res[NP];
      if constexpr (FAST) {
        const double i0 = rcp_nr(0.5 * (dLL + dL)), i1 = rcp_nr(0.5 * (dL + dR)), i2 = rcp_nr(0.5 * (dR + dRR));
        const double hL = 0.5 * dL, hR = 0.5 * dR;
        with_limiter(C.lim, [&](auto lim) {
#pragma unroll
          for (int s = 0; s < NP; ++s) {
            const double* q = Pl + s * NX;
            const double qLL = q[kLL], qL = q[kL], qR = q[kR], qRR = q[kRR];
            L[s] = qL + limiter_nr(lim.id, (qR - qL) * i1, (qL - qLL) * i0) * hL;
            R[s] = qR - limiter_nr(lim.id, (qRR - qR) * i2, (qR - qL) * i1) * hR;
          }
        });
        conv_face_fast<1, 0, RS>(T, C.rs, C.mco, L, R, nx, ny, nz, area, res);
      } else {
        const double i0 = 1.0 / (0.5 * (dLL + dL)), i1 = 1.0 / (0.5 * (dL + dR)), i2 = 1.0 / (0.5 * (dR + dRR));
        const double hL = 0.5 * dL, hR = 0.5 * dR;
        with_limiter(C.lim, [&](auto lim) {
#pragma unroll
          for (int s = 0; s < NP; ++s) {
            const double* q = Pl + s * NX;
            const double qLL = q[kLL], qL = q[kL], qR = q[kR], qRR = q[kRR];
            L[s] = qL + half_slope(lim.id, qLL, qL, qR, i0, i1, hL);
            R[s] = qR - half_slope(lim.id, qL, qR, qRR, i1, i2, hR);
          }
        });
        conv_face_lr<1, 0, RS>(T, C.rs, C.mco, L, R, nx, ny, nz, area, res);
      }
      const int f = d ? NI + a + TI * b : a + (TI + 1) * b;
#pragma unroll
      for (int s = 0; s < NP; ++s) Fb[s * NF + f] = res[s];
    }
  }
  __syncthreads();

  // ---------------- update ----------------
  double dtl = 1e300, dres[NP];
#pragma unroll
  for (int s = 0; s < NP; ++s) dres[s] = 0.0;
  if (mine) {
    const int fi = ca + (TI + 1) * cb, fj = NI + ca + TI * cb;
    double p[NP], tmp[NP], out[NP];
#pragma unroll
    for (int s = 0; s < NP; ++s) {
      p[s] = Pl[s * NX + tid];
      double t = 0.0;
      if (ci < B.n1) t = t + Fb[s * NF + fi + 1];
      if (ci > 1) t = t - Fb[s * NF + fi];
      if (cj < B.n2) t = t + Fb[s * NF + fj + TI];
      if (cj > 1) t = t - Fb[s * NF + fj];
      tmp[s] = t;
    }
    const bool on[6] = {ci == 1, ci == B.n1, cj == 1, cj == B.n2, true, true};
#pragma unroll
    for (int f = 1; f <= 6; ++f) {
      if (!on[f - 1]) continue;
      const int64_t pos = B.bpoff[f - 1] + plane_pos(B, f, ci, cj, 1);
#pragma unroll
      for (int s = 0; s < NP; ++s) {
        tmp[s] = tmp[s] + C.binc[(int64_t)s * C.NBP + pos];
        tmp[s] = tmp[s] + C.binc[(int64_t)(NP + s) * C.NBP + pos];
      }
    }
    const double rho = rho_sum<1>(p), Rg = f_Rtot<1>(T, p);
    const double Tseed = p[V::np] / (rho * Rg);
    if (C.prim) update_cell_prim<1, 0>(T, p, po, tmp, vol, *C.dt, C.strang, A.rkc, out);
    else if constexpr (FAST) update_cell_nr<1, 0>(T, p, po, tmp, *C.dt * C.strang * rcp_nr(vol), A.rkc, Tseed, out);
    else update_cell<1, 0>(T, p, po, tmp, vol, *C.dt, C.strang, A.rkc, Tseed, out);
    bool good = out[V::np] >= 0.0;
#pragma unroll
    for (int s = 0; s < NP; ++s) good = good && isfinite(out[s]);
    if (!good) flag_bad(C, tl.b, ci, cj, 1, 0);
#pragma unroll
    for (int s = 0; s < NP; ++s) C.Pout[s * NC + c0] = out[s];
    if (A.last) {
      dtl = cell_dt<1, 0>(C, c0, out);
      step_change<1, 0>(out, po, dres);
    }
  }
  if (A.last) {
    block_sum_store<NP>(dres, A.rpart + (int64_t)tidx * NP);
    block_min_atomic(dtl, A.dtnext);
  }
}

// `two`: some block has more than one cell in j; `threads`: flat_threads
template <bool FAST, bool WIDE>
inline void launch_flat_rs(const CaseDev& D, const StageArgs& A, int rs, bool two, int threads, unsigned grid,
                           hipStream_t s) {
  const size_t lds = flat_lds_doubles(A.TI, A.TJ, two) * sizeof(double);
  if (rs == MOSE_RS_LMROE) k_flat<FAST, MOSE_RS_LMROE, WIDE><<<grid, threads, lds, s>>>(D, A, two);
  else if (rs == MOSE_RS_AUSMP) k_flat<FAST, MOSE_RS_AUSMP, WIDE><<<grid, threads, lds, s>>>(D, A, two);
  else if (rs == MOSE_RS_HLLE) k_flat<FAST, MOSE_RS_HLLE, WIDE><<<grid, threads, lds, s>>>(D, A, two);
  else {
    if constexpr (!FAST) {
      if (rs == MOSE_RS_SLAU) { k_flat<FAST, MOSE_RS_SLAU, WIDE><<<grid, threads, lds, s>>>(D, A, two); return; }
    }
    k_flat<FAST, MOSE_RS_HLLC, WIDE><<<grid, threads, lds, s>>>(D, A, two);
  }
}
template <bool FAST>
inline void launch_flat(const CaseDev& D, const StageArgs& A, int rs, bool two, int threads, unsigned grid,
                        hipStream_t s) {
  if (threads > A.TI * A.TJ) launch_flat_rs<FAST, true>(D, A, rs, two, threads, grid, s);
  else launch_flat_rs<FAST, false>(D, A, rs, two, threads, grid, s);
}

}  // namespace mose
