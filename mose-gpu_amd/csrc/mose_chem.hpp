// Per-cell stiff chemistry on the device: FLINT's general law-of-mass-action source, the constant-volume ODE of
// rhs_native, and the RODAS integrator with the numerical Jacobian of the host path (wrap_rodas -> hairerRodas.f),
// one team of NS + 1 lanes per cell.
//
//   net_rate    general()                 lib/FLINT/src/lib/Lib_Chemistry_wdot.f90:163-288 (+ falloff :12-80)
//   team_rhs    rhs_native                lib/FLINT/src/lib/Lib_Chemistry_rhs.f90:29-81
//   team_dec_lds / team_sol_lds  DEC / SOL  lib/FLINT/src/lib/Lib_Radau5_dev.f90:950-1035
//   chem_cells  ROSCOR (METH = 1, IJAC = 0, autonomous) hairerRodas.f:540-880 inside Chemistry_Newstate_blk
//               (src/lib/physics/Lib_Chemistry.f90:33-76)
//
// A team of NS + 1 lanes integrates one cell (row r of every matrix and component r of every vector on lane r).
// Work distribution: a persistent grid; each team takes its next cell from an atomic queue when its cell is done
// (uneven stiffness -> uneven step counts), and every iteration of the team loop does one step attempt.
#pragma once

#include <hip/hip_runtime.h>

#include "mose_internal.h"
#include "mose_libm.h"

namespace mose {

struct ChemDev {
  int ns, na, nt, nl, tmin, rows;
  double wm[MOSE_MAX_SPECIES], Ri[MOSE_MAX_SPECIES];
  const double *cp, *h, *ni1, *ni2, *eps, *kf, *kb, *troe, *lind;
  // The tables of a two-round mechanism (chem_two_rounds) as its lanes read them, one row of `lcol` doubles per Kelvin:
  // pairs (kf, kb), or (k_inf, k_0) of a falloff reaction, of the reaction of lane r in round n at 2 (n (ns + 1) + r),
  // then (K_c, F_cent) of lane r's falloff reaction at 2 (2 (ns + 1) + r), then (h, cp) of species s at
  // 2 (3 (ns + 1) + s).  One temperature of a cell then touches six cache lines; in the tables by reaction every pair
  // was a line of its own.
  const double* lanes;
  int lcol;
  int two_rounds;
};

// Where the reactions run: round n of lane r takes reaction ord[n (ns + 1) + r]; falloff reactions first, then the
// other third-body ones, then the rest, each in reaction order (the rates go to their own places, so the order of
// evaluation does not enter).  nr entries.
inline void chem_order(int ns, int na, int nr, const double* ni1, int* ord) {
  int at = 0;
  for (int rank = 0; rank < 3; ++rank)
    for (int q = 0; q < nr; ++q) {
      const int mine = q >= na ? 0 : (ni1[(size_t)q * (ns + 1) + ns] > 0.0 ? 1 : 2);
      if (mine == rank) ord[at++] = q;
    }
}
// The mechanisms whose rates the kernels form in two straight-line rounds: at most 2 (ns + 1) reactions, at most ns + 1
// of them falloff or third body (all in the first round), and on each side of a reaction whole orders that sum to at
// most 2 (the product is then c_a, c_a c_a or c_a c_b).  Others run the general loops.
inline bool chem_two_rounds(int ns, int na, int nr, const double* ni1, const double* ni2) {
  if (nr > 2 * (ns + 1)) return false;
  int first = 0;
  for (int q = 0; q < nr; ++q) {
    const double *a = ni1 + (size_t)q * (ns + 1), *b = ni2 + (size_t)q * (ns + 1);
    if (q >= na || a[ns] > 0.0) ++first;
    for (const double* n : {a, b}) {
      double sum = 0.0;
      for (int s = 0; s < ns; ++s) {
        if (!(n[s] == 0.0 || n[s] == 1.0 || n[s] == 2.0)) return false;
        sum += n[s];
      }
      if (sum > 2.0) return false;
    }
  }
  return first <= ns + 1;
}

struct ChemArgs {
  double* state;            // rows of `stride` doubles: species densities in rows 0..NS-1, p in row prow
  const long long* rows;    // the column of cell c in state (a flow case's interior rows), or null: column c
  int prow;                 // the row of p: NS for a batch, NS + 3 on a flow case's arena
  const double* dtp;        // the case's dt on the device (a Strang step reacts over the step's dt), or null: dt
  double* hr;               // [ncell]
  int* idid;                // [ncell]
  int* nstep;               // [ncell]
  unsigned long long* queue;   // [0] next cell
  unsigned long long* stats;   // [0] steps, [1] rejected, [2] rhs calls, [3] failed, [4] max steps,
                               // [5] ~0 - (first failed cell), 0 if none
  int tpw;                  // teams per wavefront that take cells (chem_teams)
  long long ncell;
  long long stride;          // row stride of state (>= ncell)
  double dt;
  double rtol[MOSE_MAX_SPECIES + 1], atol[MOSE_MAX_SPECIES + 1];   // RADAU5: the transformed tolerances
  double rk[12];             // RADAU5: c1, c2, c1 - 1, c2 - 1, c1 - c2, dd1, dd2, dd3, 1/u1, alph, beta, FNEWT
};

// Teams per wavefront for a batch: few cells are spread over all the SIMDs (one wavefront of each first), so that the
// teams of a wavefront, which step together, wait for fewer others.
inline int chem_teams(long long ncell, int cus, int per_wave) {
  const long long t = (ncell + 4LL * cus - 1) / (4LL * cus);
  return t < 1 ? 1 : (t > per_wave ? per_wave : (int)t);
}

// one persistent launch of RADAU5 or RODAS over the cells of A, in the form that the mechanism takes (mose_chem.hip)
void launch_chem(const ChemDev& M, ChemArgs A, bool radau5, int cus, hipStream_t s);

__device__ __forceinline__ double ctab(const ChemDev& M, const double* t, int T1, double Td) {
  int r1 = T1 - M.tmin, r2 = r1 + 1;
  r1 = r1 < 0 ? 0 : (r1 > M.rows - 1 ? M.rows - 1 : r1);
  r2 = r2 < 0 ? 0 : (r2 > M.rows - 1 ? M.rows - 1 : r2);
  double a = t[r1], b = t[r2];
  return a + (b - a) * Td;
}

// Fortran x**n for a small non-negative integer n (repeated squaring, as the run-time integer power)
__device__ __forceinline__ double chem_ipow(double x, int n) {
  double r = 1.0;
  bool first = true;
  while (n > 0) {
    if (n & 1) { r = first ? x : r * x; first = false; }
    n >>= 1;
    if (n) x = x * x;
  }
  return first ? 1.0 : r;
}


// b / e from r = 1 / e (rounded to nearest), with the bits of the division: two corrections of b r by exact
// remainders; the second makes the quotient the rounded one (Markstein's theorem: a quotient within one ulp, corrected
// by its exact remainder and the rounded reciprocal).  r is NaN where |e| is outside [1e-100, 1e100] (rcp_of), and a
// numerator outside [1e-150, 1e150] (zero apart) divides too.  Five operations where the division takes eleven.
__device__ __forceinline__ double rcp_of(double e) {
  const double a = fabs(e);
  const double r = 1.0 / e;
  return (a >= 1e-100 && a <= 1e100) ? r : __builtin_nan("");
}
__device__ __forceinline__ double div_rcp(double b, double e, double r) {
  const double q0 = b * r;
  const double q1 = fma(fma(-e, q0, b), r, q0);
  double q = fma(fma(-e, q1, b), r, q1);
  const double ab = fabs(b);
  if (b == 0.0 && r == r) q = q0;     // the signed zero of b r
  else if (!(ab >= 1e-150 && ab <= 1e150 && r == r)) q = b / e;
  return q;
}
// the same for a divisor known to be positive and in rcp_of's range and a numerator that is not a negative zero
__device__ __forceinline__ double div_pos(double b, double e, double r) {
  const double q0 = b * r;
  const double q1 = fma(fma(-e, q0, b), r, q0);
  double q = fma(fma(-e, q1, b), r, q1);
  const double ab = fabs(b);
  if (!((ab >= 1e-150 && ab <= 1e150) || b == 0.0)) q = b / e;
  return q;
}

/* Deterministic natural log for the Troe broadening factor's log10, the statements of the host side: x = m 2^e with
 * m in [sqrt(1/2), sqrt(2)), log m = 2 atanh(s), s = (m-1)/(m+1), odd series to s^23.  Within a few ulp of the true
 * value for the arguments met here (Fcent in (0, 1], Pr > 0). */
__device__ __forceinline__ double dm_log(double x) {
  int e;
  double m = frexp(x, &e);            /* x = m 2^e, m in [0.5, 1) */
  if (m < 0.70710678118654752440) { m = m * 2.0; e = e - 1; }
  double s = (m - 1.0) / (m + 1.0), s2 = s * s, t = 0.0;
  for (int k = 23; k >= 3; k -= 2) t = (t + 1.0 / (double)k) * s2;
  double lm = 2.0 * s * (1.0 + t);
  return (double)e * 0.69314718055994528623 + ((double)e * 2.3190468138462996154e-17 + lm);
}

constexpr double DM_LN10 = 2.30258509299404568402;

// f_F (Lib_Chemistry_falloff.f90:63-80) from lF = log10 Fcent; log10 through dm_log, 10** through mose_pow (glibc's
// pow, as the reference)
__device__ __forceinline__ double troe_F(double Pr, double lF) {
  double lP = div_pos(dm_log(Pr), DM_LN10, 1.0 / DM_LN10);
  double cc = -0.4 - 0.67 * lF, nn = 0.75 - 1.27 * lF;
  double f1 = (lP + cc) / (nn - 0.14 * (lP + cc));
  return mose_pow(10.0, lF / (1.0 + f1 * f1));
}

// c**nu of the falloff classes: integer power for integral nu, pow otherwise
__device__ __forceinline__ double rpow(double c, double nu) {
  double r = rint(nu);
  return (r == nu && r >= 0.0 && r <= 8.0) ? chem_ipow(c, (int)r) : mose_pow(c, nu);
}

// ---------------------------------------------------------------------------------------------------------------
// A team of NS + 1 lanes integrates one cell: lane r of the team owns row r of the Jacobian and of the LU factors and
// component r of every vector.  Reactions are spread over the lanes; every sum the sequential statements form (species
// production over the reactions, the energy sums, the pivot search, the error norm) is gathered into each lane
// through the team's LDS area and added in the same order, so the team reproduces the sequential statements bit for
// bit.
// ---------------------------------------------------------------------------------------------------------------
constexpr int SLOT = 16;    // component slots of the Jacobian in LDS (ns + 1 <= 16)
constexpr int CSL = 12;     // species slots of the workgroup's LDS tables (ns <= 12)
constexpr int NRMAX = 32;   // reactions per mechanism in these kernels

// A team is NS + 1 lanes (one per ODE component); a wavefront holds 64 / (NS + 1) teams and its remaining lanes idle.
template <int NS>
struct TeamShape {
  static constexpr int size = NS + 1;
  static constexpr int per_wave = 64 / size;
  static constexpr int per_wg = 4 * per_wave;   // 256-lane workgroups
};

__device__ __forceinline__ double tsh(double v, int src) { return __shfl(v, src, 64); }
__device__ __forceinline__ int tshi(int v, int src) { return __shfl(v, src, 64); }

// Compact form of the mechanism's reactions, built once per workgroup in LDS: the orders nu'(q, s) and nu''(q, s)
// as 4-bit fields when every one is an integer in [0, 8] (the powers of both rate classes are then integer powers:
// nint(nu) for the Arrhenius class, the integral branch of rpow for the falloff classes), the third-body flag
// (nu'(q, ns+1) > 0) and the third-body efficiencies.  Reactions run in rounds of one per lane: ord lists them with
// the falloff reactions first, then the other third-body ones, so that the rounds after the first skip both (the
// rates go to their own places, the order of evaluation does not enter).
struct RxnLds {
  unsigned long long o1[NRMAX], o2[NRMAX];
  unsigned int c1[NRMAX], c2[NRMAX];   // the nonzero orders of each side as bytes (species << 4 | order), ascending;
                                       // empty places name the concentration slot that holds 1 (order 1)
  int flags[NRMAX];          // bit 0: third body; bit 1: the orders are packed in o1 / o2; bit 2: and in c1 / c2
  int ord[NRMAX];            // the reaction of lane r in round n at [n (ns + 1) + r]
  int kmax;                  // the most nonzero orders on one side of a reaction listed in c1 / c2, if no order is
                             // above 2; else 8 (the general powers)
  double eps[NRMAX * CSL];   // eps(q, s) at [q * CSL + s]
};

template <int NS>
__device__ __forceinline__ void rxn_build(const ChemDev& M, RxnLds& X) {
  constexpr int W = NS + 1;
  constexpr unsigned ONE = (unsigned)(NS + 1) << 4 | 1u;
  static_assert(NS + 1 < 16, "the slot of the constant 1 is named in 4 bits");
  const int nr = M.na + M.nt + M.nl;
  if (threadIdx.x == 0) X.kmax = 0;
  __syncthreads();
  for (int q = threadIdx.x; q < NRMAX; q += blockDim.x) {
    int fl = 0;
    unsigned long long o1 = 0ull, o2 = 0ull;
    unsigned int c1 = 0u, c2 = 0u;
    if (q < nr) {
      const double* n1 = M.ni1 + (size_t)q * W;
      const double* n2 = M.ni2 + (size_t)q * W;
      if (n1[NS] > 0.0) fl |= 1;
      bool packed = true;
      for (int s = 0; s < NS; ++s) {
        const double a = n1[s], b = n2[s];
        if (a == rint(a) && a >= 0.0 && a <= 8.0 && b == rint(b) && b >= 0.0 && b <= 8.0) {
          o1 |= (unsigned long long)(int)a << (4 * s);
          o2 |= (unsigned long long)(int)b << (4 * s);
        } else {
          packed = false;
        }
      }
      if (packed) fl |= 2;
      // at most four species with a nonzero order on each side: the byte lists (SLOT = 16 species fit 4 bits)
      int k1 = 0, k2 = 0, top = 0;
      for (int s = 0; packed && s < NS; ++s) {
        const int a = (int)((o1 >> (4 * s)) & 15ull), b = (int)((o2 >> (4 * s)) & 15ull);
        if (a != 0) { if (k1 < 4) c1 |= (unsigned)(s << 4 | a) << (8 * k1); ++k1; }
        if (b != 0) { if (k2 < 4) c2 |= (unsigned)(s << 4 | b) << (8 * k2); ++k2; }
        top = top > a ? top : a;
        top = top > b ? top : b;
      }
      if (packed && k1 <= 4 && k2 <= 4) {
        fl |= 4;
        for (int e = k1; e < 4; ++e) c1 |= ONE << (8 * e);
        for (int e = k2; e < 4; ++e) c2 |= ONE << (8 * e);
        atomicMax(&X.kmax, top > 2 ? 8 : (k1 > k2 ? k1 : k2));
      }
      // the place in the rounds: falloff, third body, the rest, each in reaction order
      auto rank = [&](int p) { return p >= M.na ? 0 : (M.ni1[(size_t)p * W + NS] > 0.0 ? 1 : 2); };
      const int mine = rank(q);
      int at = 0;
      for (int p = 0; p < nr; ++p) at += (rank(p) < mine || (rank(p) == mine && p < q)) ? 1 : 0;
      X.ord[at] = q;
    }
    X.o1[q] = o1;
    X.o2[q] = o2;
    X.c1[q] = c1;
    X.c2[q] = c2;
    X.flags[q] = fl;
  }
  for (int i = threadIdx.x; i < NRMAX * CSL; i += blockDim.x) {
    const int q = i / CSL, s = i % CSL;
    X.eps[i] = (q < nr && s < NS) ? M.eps[(size_t)q * W + s] : 0.0;
  }
}

// The exchange area of one team in LDS.  A team's lanes are in one wavefront, so a write by one lane is seen by the
// others after a wavefront-scope fence (no workgroup barrier).
template <int NS, bool TWO>
struct TeamLds {
  static constexpr int SL = NS + 3;
  static constexpr int NR = TWO ? 2 * (NS + 1) : NRMAX;
  double c[SL];            // the concentrations max(Z_s, 0) / W_s; c[NS + 1] = 1
  double net[NR];          // rates of progress, reaction q at [q]; 0 past the last reaction
  double ka[TWO ? 1 : NR]; // general mechanisms: the rate constants at the last temperature: kf, or k_inf of a falloff
  double kb[TWO ? 1 : NR]; // reaction; kb, or k_0
  double ei[SL];           // per-species terms of the energy sums; pivot rows
  double rc[SL];           // and the imaginary parts of DECC's
  double q[SL];            // columns and vectors of DEC / DECC, squared errors
  double d[SL], rd[SL];    // the increments of the Jacobian columns and their reciprocals; DECC's imaginary columns (d)
};

// What the rhs takes from the tables at one temperature, kept on the lanes while the temperature stays the same (f(y)
// and all but the last column of the Jacobian, 10 of a RODAS step's 16 evaluations).  The values are those that the
// loads would give again.
struct RateAt {
  double T;                // NaN: none yet
  double ka0, kb0, ka1, kb1;   // two-round mechanisms: the rate constants of this lane's two reactions
  double kc, lF, Fc;       // K_c, log10 F_cent and F_cent of the falloff reaction of this lane in the first round
  double rki, rkc;         // 1 / k_inf, 1 / K_c (rcp_of)
  double hR, cR;           // h - R T and cp - R of this lane's species
};

__device__ __forceinline__ void wsync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The rate constants of reaction q at (Ti, Td) into L.ka / L.kb, and K_c, log10 F_cent for a falloff reaction
template <int NS>
__device__ __forceinline__ void rate_load(const ChemDev& M, int q, int Ti, double Td, TeamLds<NS, false>& L, double& kc,
                                          double& lF) {
  if (q < M.na) {
    L.ka[q] = ctab(M, M.kf + (size_t)q * M.rows, Ti, Td);
    L.kb[q] = ctab(M, M.kb + (size_t)q * M.rows, Ti, Td);
  } else {
    const bool troe = q < M.na + M.nt;
    const double* tb = troe ? M.troe + (size_t)(q - M.na) * 4 * M.rows : M.lind + (size_t)(q - M.na - M.nt) * 3 * M.rows;
    L.ka[q] = ctab(M, tb, Ti, Td);
    L.kb[q] = ctab(M, tb + M.rows, Ti, Td);
    kc = ctab(M, tb + 2 * M.rows, Ti, Td);
    if (troe) lF = dm_log(ctab(M, tb + 3 * M.rows, Ti, Td)) / DM_LN10;
  }
}

// rate of progress of reaction q (the body of the loops of general(), Lib_Chemistry_wdot.f90:185-285) from the
// concentrations L.c and the rate constants of rate_load
template <int NS>
__device__ __forceinline__ double net_rate(const ChemDev& M, const RxnLds& X, int q, const TeamLds<NS, false>& L,
                                           double kc, double lF) {
  constexpr int W = NS + 1;
  const double* coi = L.c;
  const bool falloff = q >= M.na;
  const int fl = X.flags[q];
  double coM = 1.0;
  if (fl & 1) {
    coM = 0.0;
#pragma unroll
    for (int s = 0; s < NS; ++s) coM = coM + coi[s] * X.eps[q * CSL + s];
  }
  double pf = 1.0, pr = 1.0, rf, rr;
  if (fl & 4) {
    // the products over the nonzero orders, in species order; X.kmax is the same for every lane
    const unsigned c1 = X.c1[q], c2 = X.c2[q];
    const int kmax = X.kmax;
    if (kmax <= 4) {
      // orders 1 and 2 only; the empty places multiply by 1
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (e < kmax) {
          const unsigned v = (c1 >> (8 * e)) & 255u, w = (c2 >> (8 * e)) & 255u;
          const double a = coi[v >> 4], b = coi[w >> 4];
          pf = pf * ((v & 15u) == 2u ? a * a : a);
          pr = pr * ((w & 15u) == 2u ? b * b : b);
        }
      }
    } else {
#pragma unroll 1
      for (int e = 0; e < 4; ++e) {
        const unsigned v = (c1 >> (8 * e)) & 255u, w = (c2 >> (8 * e)) & 255u;
        pf = pf * chem_ipow(coi[v >> 4], (int)(v & 15u));
        pr = pr * chem_ipow(coi[w >> 4], (int)(w & 15u));
      }
    }
  } else if (fl & 2) {
    const unsigned long long o1 = X.o1[q], o2 = X.o2[q];
#pragma unroll 1
    for (int s = 0; s < NS; ++s) {
      const int a = (int)((o1 >> (4 * s)) & 15ull), b = (int)((o2 >> (4 * s)) & 15ull);
      if (a != 0) pf = pf * chem_ipow(coi[s], a);
      if (b != 0) pr = pr * chem_ipow(coi[s], b);
    }
  } else {
    const double* n1 = M.ni1 + (size_t)q * W;
    const double* n2 = M.ni2 + (size_t)q * W;
#pragma unroll 1
    for (int s = 0; s < NS; ++s) {
      const double a = n1[s], b = n2[s];
      if (!falloff) {
        if (a != 0) pf = pf * chem_ipow(coi[s], (int)round(a));
        if (b != 0) pr = pr * chem_ipow(coi[s], (int)round(b));
      } else {
        if (a != 0) pf = pf * rpow(coi[s], a);
        if (b != 0) pr = pr * rpow(coi[s], b);
      }
    }
  }
  if (!falloff) {
    rf = L.ka[q] * pf * coM;
    rr = L.kb[q] * pr * coM;
  } else {
    const double kinf = L.ka[q], k0 = L.kb[q];
    const double Pr = k0 * coM / kinf;
    double k1 = kinf * (Pr / (1.0 + Pr));
    if (q < M.na + M.nt) k1 = k1 * troe_F(Pr, lF);
    const double k2 = k1 / kc;
    rf = k1 * pf;
    rr = k2 * pr;
  }
  return rf - rr;
}

// What a lane keeps of the mechanism for the whole kernel
template <int NS, bool TWO>
struct LaneChem {
  double wm, rwm;          // the molecular weight of its species and 1 / wm
  double Ri;
  int q0, q1;              // two rounds: its reactions (-1: none)
  unsigned i0, i1;         // the LDS places (bytes) in TeamLds::c of the factors of both sides: f1 | f2 | r1 | r2
  int kind;                // of q0: bit 0 third body, bit 1 falloff, bit 2 Troe
};

template <int NS, bool TWO>
__device__ __forceinline__ void lane_setup(const ChemDev& M, const RxnLds& X, TeamLds<NS, TWO>& L, int r,
                                           LaneChem<NS, TWO>& K, RateAt& C) {
  constexpr int NZ = NS + 1;
  K.wm = M.wm[r < NS ? r : 0];
  K.rwm = 1.0 / K.wm;
  K.Ri = M.Ri[r < NS ? r : 0];
  K.q0 = K.q1 = -1;
  K.i0 = K.i1 = 0u;
  K.kind = 0;
  if (r == 0) L.c[NS + 1] = 1.0;
  if constexpr (TWO) {
    const int nr = M.na + M.nt + M.nl;
    L.net[r] = 0.0;
    L.net[NZ + r] = 0.0;
    // the factors of a side of order at most 2: the species of its list, one of order 2 twice, 1 for what is missing
    auto places = [&](unsigned c) -> unsigned {
      const unsigned a = (c & 255u) >> 4, na = c & 15u, b = na == 2u ? a : (c >> 8 & 255u) >> 4;
      return a * 8u | b * 8u << 8;
    };
    if (r < nr) K.q0 = X.ord[r];
    if (NZ + r < nr) K.q1 = X.ord[NZ + r];
    if (K.q0 >= 0) {
      K.i0 = places(X.c1[K.q0]) | places(X.c2[K.q0]) << 16;
      K.kind = (X.flags[K.q0] & 1) | (K.q0 >= M.na ? 2 : 0) | (K.q0 >= M.na && K.q0 < M.na + M.nt ? 4 : 0);
    }
    if (K.q1 >= 0) K.i1 = places(X.c1[K.q1]) | places(X.c2[K.q1]) << 16;
  }
  C.T = __builtin_nan("");
  C.ka0 = C.kb0 = C.ka1 = C.kb1 = C.kc = C.lF = C.rki = C.rkc = C.hR = C.cR = 0.0;
  C.Fc = __builtin_nan("");
}

// rhs_native (Lib_Chemistry_rhs.f90:29-81) for the team: z = this lane's component of Z, returns this lane's F.
// cw[q * CSL + s] = wm(s) * (nu''(q, s) - nu'(q, s)), the first product of the production statement of general()
// (Lib_Chemistry_wdot.f90:280-284), so that omega_s = sum over q in order of cw * net_q rounds as that statement.
// K = this lane's part of the mechanism, C = the values of the last temperature.
//
// The evaluation is one chain of short dependent pieces (a lone wavefront took 9,200 cycles for it), so what bounds it
// is latency: the two-round form reads each batch of LDS values at once, keeps the lane's reaction and rate constants in
// registers, and sums the production over a fixed number of reactions (zeros past the last) instead of branching at
// each one.
template <int NS, bool TWO>
__device__ __forceinline__ double team_rhs(const ChemDev& M, const RxnLds& X, const double* cw, TeamLds<NS, TWO>& L, int r,
                                           int base, const LaneChem<NS, TWO>& K, double z, RateAt& C) {
  constexpr int NZ = NS + 1;
  const int rs = r < NS ? r : 0;
  const double zp = z > 0.0 ? z : 0.0;
  const double T = tsh(z, base + NS);
  L.c[r] = div_pos(zp, K.wm, K.rwm);   // coi(s) on lane s
  wsync();
  if (T < (double)M.tmin || T >= (double)(M.tmin + M.rows - 1) || T != T) return -1.0;
  const int nr = M.na + M.nt + M.nl;
  if constexpr (TWO) {
    if (T != C.T) {
      const int Ti = static_cast<int>(T);
      const double Tf = T - (double)Ti;
      C.T = T;
      const double2* a = reinterpret_cast<const double2*>(M.lanes + (size_t)(Ti - M.tmin) * M.lcol) + r;
      const double2* b = a + M.lcol / 2;
      const double2 a0 = a[0], b0 = b[0], a1 = a[NZ], b1 = b[NZ], ah = a[3 * NZ], bh = b[3 * NZ];
      double2 af = a0, bf = b0;
      if (K.kind & 2) { af = a[2 * NZ]; bf = b[2 * NZ]; }
      C.ka0 = a0.x + (b0.x - a0.x) * Tf;
      C.kb0 = a0.y + (b0.y - a0.y) * Tf;
      C.ka1 = a1.x + (b1.x - a1.x) * Tf;
      C.kb1 = a1.y + (b1.y - a1.y) * Tf;
      C.hR = (ah.x + Tf * (bh.x - ah.x)) - K.Ri * T;
      C.cR = (ah.y + Tf * (bh.y - ah.y)) - K.Ri;
      if (K.kind & 2) {
        C.kc = af.x + (bf.x - af.x) * Tf;
        C.rki = rcp_of(C.ka0);
        C.rkc = rcp_of(C.kc);
        if (K.kind & 4) {
          const double Fc = af.y + (bf.y - af.y) * Tf;
          if (Fc != C.Fc) { C.Fc = Fc; C.lF = dm_log(Fc) / DM_LN10; }
        }
      }
    }
    const char* cb = reinterpret_cast<const char*>(L.c);
    auto at = [&](unsigned w, int n) { return *reinterpret_cast<const double*>(cb + (w >> (8 * n) & 255u)); };
    const double f0 = at(K.i0, 0) * at(K.i0, 1), r0 = at(K.i0, 2) * at(K.i0, 3);
    const double f1 = at(K.i1, 0) * at(K.i1, 1), r1 = at(K.i1, 2) * at(K.i1, 3);
    double coM = 0.0;
    const double* ep = X.eps + (K.q0 < 0 ? 0 : K.q0) * CSL;
#pragma unroll
    for (int s = 0; s < NS; ++s) coM = coM + L.c[s] * ep[s];
    coM = (K.kind & 1) ? coM : 1.0;
    if (K.q1 >= 0) L.net[K.q1] = C.ka1 * f1 - C.kb1 * r1;
    double n0 = C.ka0 * f0 * coM - C.kb0 * r0 * coM;
    if (K.kind & 2) {
      const double Pr = div_rcp(C.kb0 * coM, C.ka0, C.rki);
      double k1 = C.ka0 * (Pr / (1.0 + Pr));
      if (K.kind & 4) k1 = k1 * troe_F(Pr, C.lF);
      n0 = k1 * f0 - div_rcp(k1, C.kc, C.rkc) * r0;
    }
    if (K.q0 >= 0) L.net[K.q0] = n0;
  } else {
    // falloff reactions past the first round have no lane registers: their tables are read again
    if (T != C.T || M.nt + M.nl > NZ) {
      const int Ti = static_cast<int>(T);
      const double Tf = T - (double)Ti;
      C.T = T;
#pragma unroll 1
      for (int q0 = 0; q0 < nr; q0 += NZ)
        if (q0 + r < nr) {
          double kc = 0.0, lF = 0.0;
          const int q = X.ord[q0 + r];
          rate_load<NS>(M, q, Ti, Tf, L, kc, lF);
          if (q0 == 0) { C.kc = kc; C.lF = lF; }
          else if (q >= M.na) L.net[q] = net_rate<NS>(M, X, q, L, kc, lF);
        }
      const int row = Ti - M.tmin;
      const double* ht = M.h + (size_t)rs * M.rows;
      const double* ct = M.cp + (size_t)rs * M.rows;
      const double h0 = ht[row], h1 = ht[row + 1], c0 = ct[row], c1 = ct[row + 1];
      C.hR = (h0 + Tf * (h1 - h0)) - K.Ri * T;
      C.cR = (c0 + Tf * (c1 - c0)) - K.Ri;
    }
#pragma unroll 1
    for (int q0 = 0; q0 < nr; q0 += NZ)
      if (q0 + r < nr) {
        const int q = X.ord[q0 + r];
        if (q0 == 0 || q < M.na) L.net[q] = net_rate<NS>(M, X, q, L, C.kc, C.lF);
      }
  }
  wsync();
  // omega_s on lane s: production summed over the reactions in order
  double om = 0.0;
  if constexpr (TWO) {
#pragma unroll
    for (int q = 0; q < 2 * NZ; ++q) om = om + cw[q * CSL + rs] * L.net[q];
  } else {
#pragma unroll 4
    for (int q = 0; q < nr; ++q) om = om + cw[q * CSL + rs] * L.net[q];
  }
  // the energy sums over the species, in order, on the lane of the T equation
  L.ei[r] = C.hR * om;
  L.rc[r] = zp * C.cR;   // roi(s) (cv - R_s) on lane s
  wsync();
  double ei = 0.0, rcv = 0.0;
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    ei = ei + L.ei[s];
    rcv = rcv + L.rc[s];
  }
  return r == NS ? -ei / rcv : om;
}

// The places of a team's rows after DEC's exchanges: this lane's row stands at pos; lane(k) is the lane (in the wave) of
// the row at place k, from nibbles.
struct RowMap {
  int pos;
  unsigned lo, hi;         // nibble k of hi:lo = the team's lane of the row at place k
  double rd;               // 1 / the pivot of this lane's row (rcp_of); DECC: 1 / |pivot|^2
  __device__ __forceinline__ int lane(int base, int k) const { return base + (int)((k < 8 ? lo >> (4 * k) : hi >> (4 * (k - 8))) & 15u); }
  __device__ __forceinline__ void init(int r) { pos = r; lo = 0x76543210u; hi = 0xfedcba98u; }
  // rows at places k and m change places (k is a compile-time index)
  __device__ __forceinline__ void swap(int k, int m) {
    const int sm = 4 * (m & 7);
    const unsigned a = (k < 8 ? lo >> (4 * k) : hi >> (4 * (k - 8))) & 15u, b = ((m < 8 ? lo : hi) >> sm) & 15u;
    const unsigned x = a ^ b;
    if (k < 8) lo ^= x << (4 * k);
    else hi ^= x << (4 * (k - 8));
    if (m < 8) lo ^= x << sm;
    else hi ^= x << sm;
    pos = pos == m ? k : (pos == k ? m : pos);
  }
};

// DEC (Moler, ACM 423; Lib_Radau5_dev.f90:950-997) with one row of the matrix per lane, e[j] = a(row, j).  Returns
// ier (0: regular).  Rows are not exchanged: the pivot search reads the column in the exchanged order (L.q[pos]) and
// so picks the row that DEC picks, and only the pivot row passes through LDS (L.ei).  Every row sees the operations
// that DEC does on it wherever it stands.
template <int N, class TL>
__device__ __forceinline__ int team_dec_lds(double (&e)[N], RowMap& W, TL& L, int r) {
  W.init(r);
#pragma unroll
  for (int k = 0; k < N - 1; ++k) {
    L.q[W.pos] = e[k];
    wsync();
    int m = k;
    double t = L.q[k];
    double am = fabs(t);
#pragma unroll
    for (int i = k + 1; i < N; ++i) {
      const double c = L.q[i], v = fabs(c);
      const bool up = v > am;
      m = up ? i : m;
      am = up ? v : am;
      t = up ? c : t;
    }
    if (m != k) W.swap(k, m);
    if (W.pos == k) {
#pragma unroll
      for (int j = k + 1; j < N; ++j) L.ei[j] = e[j];
    }
    wsync();
    if (t == 0.0) return k + 1;
    const double ti = 1.0 / t;
    const bool below = W.pos > k;
    W.rd = W.pos == k ? ((am >= 1e-100 && am <= 1e100) ? ti : __builtin_nan("")) : W.rd;
    e[k] = below ? -e[k] * ti : e[k];
#pragma unroll
    for (int j = k + 1; j < N; ++j) {
      const double amj = L.ei[j];
      const double v = e[j] + e[k] * amj;
      e[j] = (amj != 0.0 && below) ? v : e[j];
    }
  }
  if (W.pos == N - 1) { L.q[N - 1] = e[N - 1]; W.rd = rcp_of(e[N - 1]); }
  wsync();
  if (L.q[N - 1] == 0.0) return N;
  return 0;
}

// SOL (Lib_Radau5_dev.f90:1003-1035) on the team: b = the component of this lane's row, returns component r of the
// solution.  A step's chain is the broadcast of one component to the team; through a permute from the lane of its row it
// is one LDS-unit access long, through a write and a read of LDS two.
template <int N>
__device__ __forceinline__ double team_sol_lds(const double (&e)[N], const RowMap& W, double b, int base, int r) {
#pragma unroll
  for (int k = 0; k < N - 1; ++k) {
    const double t = tsh(b, W.lane(base, k));
    const double v = b + e[k] * t;
    b = W.pos > k ? v : b;
  }
#pragma unroll
  for (int kb = 1; kb <= N - 1; ++kb) {
    const int k = N - kb;
    if (W.pos == k) b = div_rcp(b, e[k], W.rd);
    const double t = -tsh(b, W.lane(base, k));
    const double v = b + e[k] * t;
    b = W.pos < k ? v : b;
  }
  if (W.pos == 0) b = div_rcp(b, e[0], W.rd);
  return tsh(b, base + (int)((r < 8 ? W.lo >> (4 * r) : W.hi >> (4 * (r - 8))) & 15u));
}

// RODAS4 (METH = 1) coefficients (ROCOE; the values of rodas_dev, Lib_Radau5_dev.f90:710-737)
struct RodasC {
  static constexpr double GAMMA = 0.25;
  static constexpr double A21 = 0.1544000000000000e+01, A31 = 0.9466785280815826e+00, A32 = 0.2557011698983284e+00;
  static constexpr double A41 = 0.3314825187068521e+01, A42 = 0.2896124015972201e+01, A43 = 0.9986419139977817e+00;
  static constexpr double A51 = 0.1221224509226641e+01, A52 = 0.6019134481288629e+01, A53 = 0.1253708332932087e+02;
  static constexpr double A54 = -0.6878860361058950e+00;
  static constexpr double C21 = -0.5668800000000000e+01, C31 = -0.2430093356833875e+01, C32 = -0.2063599157091915e+00;
  static constexpr double C41 = -0.1073529058151375e+00, C42 = -0.9594562251023355e+01, C43 = -0.2047028614809616e+02;
  static constexpr double C51 = 0.7496443313967647e+01, C52 = -0.1024680431464352e+02, C53 = -0.3399990352819905e+02;
  static constexpr double C54 = 0.1170890893206160e+02;
  static constexpr double C61 = 0.8083246795921522e+01, C62 = -0.7981132988064893e+01, C63 = -0.3152159432874371e+02;
  static constexpr double C64 = 0.1631930543123136e+02, C65 = -0.6058818238834054e+01;
};

// The workgroup's LDS copies of the mechanism: the compact reactions and cw (see team_rhs)
template <int NS>
__device__ __forceinline__ void chem_setup(const ChemDev& M, double* cw, RxnLds& X) {
  rxn_build<NS>(M, X);
  const int nr = M.na + M.nt + M.nl;
  for (int i = threadIdx.x; i < NRMAX * CSL; i += blockDim.x) {
    const int q = i / CSL, s = i % CSL;
    double v = 0.0;
    if (q < nr && s < NS) {
      double dn = M.ni2[(size_t)q * (NS + 1) + s] - M.ni1[(size_t)q * (NS + 1) + s];
      v = M.wm[s] * dn;
    }
    cw[i] = v;
  }
  __syncthreads();
}

// Chemistry_Newstate_blk, entry (src/lib/physics/Lib_Chemistry.f90:55-60): Z = (rho_i, T = p / (rho R)); returns
// this lane's component, rho and T of the cell in rho0 / Tb
template <int NS>
__device__ __forceinline__ double cell_load(const ChemDev& M, const ChemArgs& A, int cell, int base, int r, int rc,
                                            double& rho0, double& Tb) {
  const long long col = A.rows ? A.rows[cell] : (long long)cell;
  const double q = A.state[(long long)(rc < NS ? rc : A.prow) * A.stride + col];
  const double p = A.state[(long long)A.prow * A.stride + col];
  double rho = 0.0, Rm = 0.0;
#pragma unroll
  for (int s = 0; s < NS; ++s) rho = rho + tsh(q, base + s);
#pragma unroll
  for (int s = 0; s < NS; ++s) Rm = Rm + M.Ri[s] * tsh(q, base + s) / rho;
  const double T = p / (rho * Rm);
  rho0 = rho;
  Tb = T;
  return r < NS ? q : T;
}

// Chemistry_Newstate_blk, exit (:62-70): floors, p = T rho R, hr; and the batch statistics
template <int NS>
__device__ __forceinline__ void cell_store(const ChemDev& M, const ChemArgs& A, int cell, int base, int r, double y,
                                           double rho0, double Tb, int idid, int nst, int nrej, int nfcn) {
  const double yf = (r < NS && y <= 1e-20) ? 1e-20 : y;
  double rs = 0.0, R2 = 0.0;
  const double T = tsh(y, base + NS);
#pragma unroll
  for (int s = 0; s < NS; ++s) rs = rs + tsh(yf, base + s);
#pragma unroll
  for (int s = 0; s < NS; ++s) R2 = R2 + M.Ri[s] * tsh(yf, base + s) / rs;
  const long long col = A.rows ? A.rows[cell] : (long long)cell;
  if (r < NS) A.state[(long long)r * A.stride + col] = yf;
  if (r == NS) {
    A.state[(long long)A.prow * A.stride + col] = T * rho0 * R2;
    A.hr[cell] = fabs(T - Tb) / Tb;
    A.idid[cell] = idid;
    A.nstep[cell] = nst;
  }
  if (r == 0) {
    atomicAdd(&A.stats[0], (unsigned long long)nst);
    atomicAdd(&A.stats[1], (unsigned long long)nrej);
    atomicAdd(&A.stats[2], (unsigned long long)nfcn);
    if (idid < 0) {
      atomicAdd(&A.stats[3], 1ull);
      atomicMax(&A.stats[5], ~0ull - (unsigned long long)cell);   // the lowest failed cell gives the largest value
    }
    atomicMax(&A.stats[4], (unsigned long long)nst);
  }
}

// One team of NS + 1 lanes per cell, persistent over the cell queue; one iteration of the team loop is one step
// attempt, and the teams of a wavefront make it together, evaluation by evaluation:
//   s = 0        f(y) at the start of a step
//   s = 1..NZ    f(y + delta e_i), column i = s - 1 of the numerical Jacobian
//   then DEC and the first SOL, and s = NZ + 1..NZ + 5: f at the input of stage k = 2..6 with its SOL
// (one rhs call site).  A team whose last attempt was rejected keeps its f(y) and Jacobian and sits out the first
// NZ + 1 evaluations.  Teams that ran through these phases each on its own had the wavefront execute DEC, SOL and the
// stage of every team in every evaluation (3,000 VALU instructions per evaluation); in step, an attempt executes each
// once.  Measured on hydrogen-air cells over 1e-6 s (41 % of the attempts rejected): 24,576 cells 1,333 -> 566 ms, 16,384
// cells 1,142 -> 398 ms, 300 cells (the longest cell's chain alone) 879 -> 342 ms.
template <int NS, bool TWO>
__device__ __forceinline__ void chem_cells(const ChemDev& M, const ChemArgs& A) {
  constexpr int NZ = NS + 1;
  static_assert(NZ <= SLOT && NS <= CSL, "one lane per ODE component");
  using TSh = TeamShape<NS>;
  using R = RodasC;
  const double uround = 1.1e-19, safe = 0.9, fac1 = 5.0, fac2 = 1.0 / 6.0;
  const int nmax = 100000;
  const double dtend = A.dtp ? *A.dtp : A.dt;   // XEND of every cell

  __shared__ double cw[NRMAX * CSL];
  __shared__ TeamLds<NS, TWO> tl[TSh::per_wg];
  __shared__ RxnLds X;
  chem_setup<NS>(M, cw, X);

  const int wl = threadIdx.x & 63;
  const int tw = wl / NZ;                // the team within the wavefront
  if (tw >= A.tpw) return;               // the lanes past the last team at work (no barrier follows)
  const int base = tw * NZ;              // lane (in the wave) of the team's row 0
  const int r = wl - base;               // this lane's row / component
  const int rc = r;
  TeamLds<NS, TWO>& L = tl[(threadIdx.x >> 6) * TSh::per_wave + tw];
  LaneChem<NS, TWO> K;
  RateAt C;
  lane_setup<NS, TWO>(M, X, L, r, K, C);

  int cell = -1;
  bool reject = false, last = false, fresh = false;   // fresh: this attempt starts with f(y) and the Jacobian
  int nsing = 0, nst = 0, nacc = 0, nrej = 0, nfcn = 0, idid = 0;
  double x = 0.0, h = 0.0, hopt = 0.0, hacc = 0.0, erracc = 1e-2, hmaxn = 0.0, posneg = 1.0;
  double rho0 = 0.0, Tb = 0.0;
  double y = 0.0, dy1 = 0.0, yn = 0.0, zin = 0.0, yd = 0.0, rh = 0.0;
  double ak1 = 0.0, ak2 = 0.0, ak3 = 0.0, ak4 = 0.0, ak5 = 0.0;
  double fjr[NZ];                         // row r of the Jacobian (kept for rejected steps)
  double e[NZ];                           // a row of the LU factors
  RowMap W;
  W.init(r);
  W.rd = 0.0;
#pragma unroll
  for (int j = 0; j < NZ; ++j) { fjr[j] = 0.0; e[j] = 0.0; }

  // label 1 of ROSCOR: the checks at the start of a step; true when the integration ends here
  auto step_start = [&]() -> bool {
    if (nst > nmax) { idid = -2; return true; }
    if (0.1 * fabs(h) <= fabs(x) * uround) { idid = -3; return true; }
    if (last) { h = hopt; idid = 1; return true; }
    hopt = h;
    if ((x + h * 1.0001 - dtend) * posneg >= 0.0) { h = dtend - x; last = true; }
    zin = y;
    fresh = true;
    return false;
  };
  while (true) {
    if (cell < 0) {
      int c = 0;
      if (r == 0) c = (int)atomicAdd(A.queue, 1ull);
      c = tshi(c, base);
      if ((long long)c >= A.ncell) break;
      cell = c;
      y = cell_load<NS>(M, A, cell, base, r, rc, rho0, Tb);
      // ROSCOR initial preparations (x = 0, xend = dt, H = 0 -> 1e-6)
      x = 0.0;
      double hmax = dtend - x;
      posneg = copysign(1.0, dtend - x);
      hmaxn = fmin(fabs(hmax), fabs(dtend - x));
      h = 0.0;
      if (fabs(h) <= 10.0 * uround) h = 1.0e-6;
      h = fmin(fabs(h), hmaxn);
      h = copysign(h, posneg);
      reject = false; last = false; nsing = 0; nst = 0; nacc = 0; nrej = 0; nfcn = 0;
      hopt = h; hacc = 0.0; erracc = 1e-2;
      idid = 0;
      (void)step_start();   // a fresh cell always proceeds
    }

    bool fin = false;
    const int s0 = __ballot(fresh) != 0ull ? 0 : NZ + 1;
#pragma unroll 1
    for (int s = s0; s < NZ + 6; ++s) {
      if (s == NZ + 1) {
        // label 2: decompose E = 1/(h gamma) - J; a singular E halves h (at most 4 times)
        while (true) {
          const double fac = 1.0 / (h * R::GAMMA);
#pragma unroll
          for (int j = 0; j < NZ; ++j) e[j] = (j == r) ? -fjr[j] + fac : -fjr[j];
          if (team_dec_lds<NZ>(e, W, L, r) == 0) break;
          nsing++;
          if (nsing >= 5) { idid = -4; fin = true; break; }
          h = h * 0.5;
          reject = true;
          last = false;
        }
        rh = rcp_of(h);
        if (!fin) {
          ak1 = team_sol_lds<NZ>(e, W, dy1, base, r);
          yn = y + R::A21 * ak1;
          zin = yn;
        }
      }
      if (s <= NZ ? !fresh : fin) continue;

      const double f = team_rhs<NS, TWO>(M, X, cw, L, r, base, K, zin, C);

      if (s == 0) {
        dy1 = f;
        nfcn++;
        // the increments of the Jacobian columns: sqrt(uround max(1e-5, |y(i)|)) (IJAC = 0), column i's on lane i
        const double delt = sqrt(uround * fmax(1.0e-5, fabs(y)));
        yd = y + delt;
        L.d[r] = delt;
        L.rd[r] = rcp_of(delt);
        zin = r == 0 ? yd : y;
      } else if (s <= NZ) {
        const int i = s - 1;
        const double col = div_rcp(f - dy1, L.d[i], L.rd[i]);
#pragma unroll
        for (int j = 0; j < NZ; ++j) fjr[j] = (j == i) ? col : fjr[j];
        zin = r == i + 1 ? yd : y;
        if (i + 1 == NZ) nfcn += NZ;
      } else {
        const int k = s - NZ + 1;   // the stage whose rhs came back in f
        double b;
        if (k == 2) b = f + div_rcp(R::C21, h, rh) * ak1;
        else if (k == 3) b = f + (div_rcp(R::C31, h, rh) * ak1 + div_rcp(R::C32, h, rh) * ak2);
        else if (k == 4) b = f + (div_rcp(R::C41, h, rh) * ak1 + div_rcp(R::C42, h, rh) * ak2 + div_rcp(R::C43, h, rh) * ak3);
        else if (k == 5) b = f + (div_rcp(R::C52, h, rh) * ak2 + div_rcp(R::C54, h, rh) * ak4 + div_rcp(R::C51, h, rh) * ak1 +
                                  div_rcp(R::C53, h, rh) * ak3);
        else b = f + (div_rcp(R::C61, h, rh) * ak1 + div_rcp(R::C62, h, rh) * ak2 + div_rcp(R::C65, h, rh) * ak5 +
                      div_rcp(R::C64, h, rh) * ak4 + div_rcp(R::C63, h, rh) * ak3);
        const double ak = team_sol_lds<NZ>(e, W, b, base, r);
        if (k == 2) { ak2 = ak; yn = y + R::A31 * ak1 + R::A32 * ak2; }
        else if (k == 3) { ak3 = ak; yn = y + R::A41 * ak1 + R::A42 * ak2 + R::A43 * ak3; }
        else if (k == 4) { ak4 = ak; yn = y + R::A51 * ak1 + R::A52 * ak2 + R::A53 * ak3 + R::A54 * ak4; }
        else if (k == 5) { ak5 = ak; yn = yn + ak5; }
        else { ak1 = ak; yn = yn + ak; }   // ak6: the error estimate (ak1 is no longer needed)
        zin = yn;
      }
    }

    if (!fin) {
      // error estimation and step size control (ak6 = ak1)
      nfcn += 5;
      nst++;
      const double sk = A.atol[rc] + A.rtol[rc] * fmax(fabs(y), fabs(yn));
      const double ql = ak1 / sk;
      L.q[r] = ql * ql;
      wsync();
      double err = 0.0;
#pragma unroll
      for (int i = 0; i < NZ; ++i) err = err + L.q[i];
      err = sqrt(err / NZ);
      // err**0.25 and the predictor's (err err / erracc)**0.25 (libm pow) at once, on the even and the odd lanes
      const double pw = mose_pow((r & 1) ? err * err / erracc : err, 0.25);
      double fac = fmax(fac2, fmin(fac1, tsh(pw, base) / safe));
      const double pgus = tsh(pw, base + 1);
      double hnew = h / fac;
      if (err <= 1.0) {
        nacc++;
        if (nacc > 1) {
          double facgus = (hacc / h) * pgus / safe;
          facgus = fmax(fac2, fmin(fac1, facgus));
          fac = fmax(fac, facgus);
          hnew = h / fac;
        }
        hacc = h;
        erracc = fmax(1.0e-2, err);
        y = yn;
        x = x + h;
        if (fabs(hnew) > hmaxn) hnew = posneg * hmaxn;
        if (reject) hnew = posneg * fmin(fabs(hnew), fabs(h));
        reject = false;
        h = hnew;
        fin = step_start();
      } else {
        reject = true;
        last = false;
        h = hnew;
        if (nacc >= 1) nrej++;
        fresh = false;
      }
    }

    if (fin) {
      cell_store<NS>(M, A, cell, base, r, y, rho0, Tb, idid, nst, nrej, nfcn);
      cell = -1;
    }
  }
}

// The general form at four waves per SIMD (190 registers spill); the two-round form at two, where its 256 registers hold the
// lane's part of the step but for two spilled ones (at three waves 478 registers spilled and 24,576 cells took 1,151 ms; they
// take 566).
template <int NS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) k_chem(ChemDev M, ChemArgs A) {
  chem_cells<NS, false>(M, A);
}
template <int NS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) k_chem2(ChemDev M, ChemArgs A) {
  chem_cells<NS, true>(M, A);
}

}  // namespace mose
