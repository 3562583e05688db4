// vert_group.h -- the AUSM vertical step with a column's work split over the
// species: the mapping of the single-grid and batch steps.
//
// A column of L = nAlts+4 levels is advanced by a workgroup of NG groups of
// whole wavefronts.  Lane j of group g owns level k = j-1 and, of its group,
// SPW = 6/NG species (g*SPW ..): their densities, winds, face states, fluxes and RK4
// carries.  What a level has once (temperature, bulk winds, energy, the
// friction solve) is dealt out to the groups: group 0 takes Temp and Vel(up),
// the left face sums and the friction solve, group 1 Vel(east), LogRho and the
// right face sums, group 2 Vel(north) and the face densities' reciprocal.
//
// Why this split: one lane per level with all six species (vert_column.h)
// keeps 530 registers live through the flux phase, so a SIMD holds one
// wavefront, and a single wavefront leaves the FP64 pipe idle while it waits
// for LDS, barriers and its register spills (47 % of its cycles issue a
// vector instruction).  With two species a lane makes do with 128, a SIMD's
// registers hold four wavefronts and one's waits are another's work; at 100
// levels LDS admits two columns per CU, three wavefronts per SIMD.
//
// The stage's state lives in LDS (a level's 17 fields side by side), so every
// lane reads any level's field; what crosses levels or groups goes through
// the level's exchange slots, and the barriers between the phases of a stage
// (ten) are the only order there is.  Sums over the species are formed from
// the groups' partial sums.
//
// The reference is advance_vertical (src/advance_vertical.f90:45-219) with
// advance_vertical_1d_ausm (src/vertical_solver_ausm.f90:26-2117),
// set_vertical_bcs (src/set_vertical_bcs.Earth.f90:8-652) and
// calc_neutral_friction (src/calc_neutral_friction.f90:4-108).  The same
// source compiles for the host (GV_HOST_EMULATION).
#pragma once

#include "vert_column.h"

namespace gv {

constexpr int SPW = 2;         // species per lane
constexpr int NG = NSP / SPW;  // groups of a column
constexpr int IPW = NI / NG;   // ions per lane
static_assert(NG == 3 && IPW * NG == NI, "three groups share a level's work");

// A level's record (doubles): the state, the tables that neighbouring levels
// read, the gradient weights, the exchange slots, and with ions LogINS and a
// pad.  An odd length keeps 64-bit accesses of consecutive levels on
// different banks.
enum GroupRec {
  // the state: the fields the groups own (Temp, east, north; Vel(up), LogRho),
  // LogNS(6), VertVel(6)
  GU_T = 0, GU_VE, GU_VN, GU_VU, GU_LR, GU_LN, GU_W = GU_LN + NSP,
  GR_DF = GU_W + NSP, GR_IF, GR_DC, GR_CMF, GR_KP, GR_KU,
  GR_GLC,  // 5 weights of d ln(rho_s/rho)/dz
  // of the level alone (the lanes' registers are scarcer than LDS): areas and
  // inverse volume, 0.35 exp(-(z - z0)/45 km), 1/r, the eddy coefficient
  GR_AP = GR_GLC + 5, GR_AM, GR_IVOL, GR_HF, GR_INVR, GR_EDDY,
  GR_GT,                         // gradient of Temp
  GR_VEL, GR_VER, GR_VNL, GR_VNR,  // horizontal winds at face k|k+1
  GR_RL, GR_RR, GR_EPL, GR_EPR, GR_IRLR, GR_CSL, GR_CSR,  // bulk face values
  GR_LTK,                          // log(k Temp)
  GR_POOL,
  // pool slots, by the phase that writes them; a slot is written again only
  // after a barrier that follows its last readers
  //   gradients and hydrostatic factors
  GP_RF = GR_POOL, GP_LF = GP_RF + 3, GP_B = GP_LF + 3,
  GP_NT = GP_B + NSP, GP_IRF = GP_NT + NG, GP_ILF = GP_IRF + NI_ADVECT,
  GP_HNS = GP_ILF + NI_ADVECT,
  //   face states: log hydrostatic pressures, then the groups' sums
  //   (left and right side by side) and the hydrostatic flags
  GP_LH = GR_POOL, GP_RSUM = GP_LH + NSP, GP_PSUM = GP_RSUM + 2 * NG,
  GP_MSUM = GP_PSUM + 2 * NG,
  //   fluxes: the M12 side of face k|k+1, the numerical velocities' sums
  GP_FR = GR_POOL, GP_FM = GP_FR + NSP, GP_NP = GP_FM + NSP,
  GP_BP = GP_NP + NSP, GP_BM = GP_BP + NG,
  //   update: Temp**-DiffExp, the groups' densities (where the face sound
  //   speeds and log(k Temp) were), and what is set aside while the friction
  //   system is solved
  GP_PW = GP_BM + NG, GP_NRHO = GR_CSL, GP_SUB = GP_PW + NG,
  GP_KGLC = GR_POOL, GP_KNRS = GP_KGLC + NSP, GP_KLN = GP_KNRS + NSP,
  GP_KW = GP_KLN + NSP, GP_KL = GR_VNL,
  GR_LEN = GP_PW + 6
};
static_assert(GP_KW + NSP <= GP_PW && GP_KL + NSP <= GR_IRLR && GP_HNS + NSP <= GP_SUB &&
                  GP_MSUM + 2 * NG <= GP_PW, "pool slots");
GV_HD constexpr int group_rec_len(bool ions) { return GR_LEN + (ions ? NI + 1 : 0); }
static_assert(group_rec_len(false) % 2 == 1 && group_rec_len(true) % 2 == 1,
              "an odd record length keeps 64-bit LDS accesses conflict-free");

// The column's scalars.
enum GroupScalar {
  GS_CA = 0, GS_CB = 5, GS_CTA = 10, GS_CTB = 15,  // one-sided weights, as Scalar's
  GS_MG0 = 20, GS_MGT1, GS_MGT2, GS_MMM_M1, GS_MMM_0, GS_ALT0, GS_TEC,
  GS_MSIS,                      // msis_bcs: LogNS(0), Temp(0), winds
  GS_TIDE = GS_MSIS + 9,        // TidesTemp(0)
  GS_COR,                       // Coriolis
  GS_MN,                        // m n_s of ghost levels -1, 0, nAlts+1, nAlts+2
  GS_MNW = GS_MN + 4 * NSP,     // m n_s w_s of levels -1, 0
  GS_N = GS_MNW + 2 * NSP
};

// LDS of one column: the scalars, then nAlts+8 records (two guard levels on
// each side).  66 KiB at nAlts = 100 and 78 KiB at
// 120, two columns per CU; 36 KiB at 50, four.
GV_HD constexpr unsigned long group_lds_bytes(int n_alts, bool ions) {
  return ((unsigned long)group_rec_len(ions) * (unsigned long)(n_alts + 8) + GS_N) *
         sizeof(double);
}
// Whether a column's LDS fits a CU: every column without ions (157 KiB at
// nAlts = 252), up to nAlts = 226 with them.
GV_HD constexpr bool group_fits(int n_alts, bool ions) {
  return group_lds_bytes(n_alts, ions) + 256 <= 160 * 1024;  // 256: the barriers' own
}
// Threads of a column's workgroup: whole wavefronts per group, so that what
// only one group does is a branch that the others' wavefronts skip.  (Packed
// without gaps, 312 threads at nAlts = 100 against 384, a wavefront that holds
// lanes of two groups ran both groups' parts.)
GV_HD constexpr int group_stride(int n_alts) { return (n_alts + 4 + 63) / 64 * 64; }
GV_HD constexpr int group_threads(int n_alts) { return NG * group_stride(n_alts); }

// 1/d and a/d by Newton steps from the hardware's reciprocal seed, the quotient
// corrected by its remainder: the device's division without the scaling that
// guards exponents near the ends of the range (8 instructions in place of 11,
// none of them serialised through VCC).  For the positive temperatures,
// densities, sound speeds and pivots of the step, which lie far inside it.
GV_FN double recip(double d) {
#ifdef GV_HOST_EMULATION
  return 1.0 / d;
#else
  double r = rcp_seed(d);
  r = fma(fma(-d, r, 1.0), r, r);
  return fma(fma(-d, r, 1.0), r, r);
#endif
}
GV_FN double quot(double a, double d) {
#ifdef GV_HOST_EMULATION
  return a / d;
#else
  const double r = recip(d), q = a * r;
  return fma(fma(-d, q, a), r, q);
#endif
}

// What MPn's numerator (in Kp) and denominator (in the mean density) are
// multiplied by: the denominator of a species of 1e-283 per m^3 is then far from
// the end of the range, where recip overflows.  A power of two: the same bits.
constexpr double MP_SCALE = 0x1p100;

// The friction solve of one level (calc_neutral_friction.f90:47-106):
// (1 + dt sum_q C_iq) x_i - dt sum_q C_iq x_q = w_i with C_iq = k T n_q /
// (m_i N D_iq).  Row i times m_i n_i makes the system symmetric,
// A_iq = -dt k T n_i n_q / (N D_iq), and A_ii = m_i n_i - sum_q A_iq: positive
// definite and diagonally dominant, so the LDL^T factors need no pivoting and
// half the operations.  pw[u] = T**-DEXU[u], nt the sum of the n_i.  Returns the
// sum of the x_i: finite unless something in the system is not.
// The whole system is multiplied by a power of two, 2^110 over about nt: the
// m_i n_i of a minor species and the n_i n_q would leave the range (densities
// below 1e-282 or above 1e150 per m^3), and the solution does not change a bit.
GV_FN double friction_solve(const KParams &P, double dt, const double (&ns)[NSP], double nt,
                            double T, const double (&pw)[6], double (&w)[NSP]) {
  const double dkT = dt * ((FRIC_SCALE * KB) * T);
  int ex;
  frexp_mant(nt, ex);
  const double unit = ldexp(1.0, 64 - (ex < -900 ? -900 : ex));
  double a[NSP][NSP], e[6], nu[NSP];  // the upper triangle
#pragma unroll
  for (int u = 0; u < 6; u++) e[u] = dkT * pw[u];
#pragma unroll
  for (int i = 0; i < NSP; i++) {
    nu[i] = ns[i] * unit;
    a[i][i] = P.fmass[i] * nu[i];
  }
#pragma unroll
  for (int i = 0; i < NSP; i++) w[i] = a[i][i] * w[i];
#pragma unroll
  for (int i = 0; i < NSP; i++)
#pragma unroll
    for (int q = i + 1; q < NSP; q++) {
      const double g = 1.0e-19 / D0R[i][q];  // 1e-2 / Diff0, a constant
      const double c = (nu[i] * ns[q]) * (g * e[DEXI[i][q]]);
      a[i][q] = -c;
      a[i][i] = a[i][i] + c;
      a[q][q] = a[q][q] + c;
    }
  GV_ORDER();
  double rd[NSP];
#pragma unroll
  for (int p = 0; p < NSP; p++) {
    rd[p] = recip(a[p][p]);
#pragma unroll
    for (int i = p + 1; i < NSP; i++) {
      const double f = a[p][i] * rd[p];
#pragma unroll
      for (int q = i; q < NSP; q++) a[i][q] = a[i][q] - f * a[p][q];
      w[i] = w[i] - f * w[p];
    }
    GV_ORDER();
  }
  double sum = 0.0;
#pragma unroll
  for (int i = NSP - 1; i >= 0; i--) {
    double s = w[i];
#pragma unroll
    for (int q = i + 1; q < NSP; q++) s = s - a[i][q] * w[q];
    w[i] = s * rd[i];
    sum = sum + w[i];
  }
  return sum;
}

// Whether the reference's ludcmp would find a row of zeros or of NaN in the
// friction matrix (ludcmp.f:14-17): every entry is NaN unless 0 < T < inf; then
// row i has the nonzero entries C_iq of the nonzero n_q, q != i, and the
// diagonal 1 + dt sum C_iq, which only a NaN among the n_q makes NaN.
GV_FN bool friction_singular(const double *ns, double T) {
  int nonzero = 0, nans = 0;
  for (int q = 0; q < NSP; q++) {
    nonzero += fabs(ns[q]) > 0.0;
    nans += ns[q] != ns[q];
  }
  return !(T > 0.0 && T < __builtin_inf()) || (nonzero <= 1 && nans >= 1);
}

template <bool IONS, class Ctx>
struct GroupColumn {
  static constexpr int RS = group_rec_len(IONS);
  Ctx &cx;
  const KParams &kp;
  double *lds;
  const int nA, L;
  int t, g, j, k, s0;  // thread, group, lane of the level, level, first species
  const int col;                    // column number in error reports
  const double dt;
  // the level's constants
  double idC, eg, mgh, gm1;
  double gf[3] = {0.0, 0.0, 0.0};  // groups 0, 1: gamma factors of the face's own side
  // hydrostatic product: segment length, this level's segment, the segments
  int seg, gseg, nseg;
  // RK4 carries: LogNS, VertVel of the lane's species; the group's own fields
  double Yn[SPW], An[SPW], Yw[SPW], Aw[SPW], Yr[2], Ar[2];
  double Yi[IPW], Ai[IPW], ivu = 0.0;
  bool plasma = false;

  GV_MEM GroupColumn(Ctx &c, const KParams &p, double *l, int column, double step_dt, int n_alts)
      : cx(c), kp(p), lds(l), nA(n_alts), L(n_alts + 4), col(column), dt(step_dt) {
    locate();
  }
  // The lane's place in the column.  Called again where a stage and its
  // boundary conditions begin, from a thread number that the compiler cannot
  // know to be the same: otherwise every address and lane mask of the stage is
  // formed once, ahead of the loop, and kept in (spilled) registers.
  GV_MEM void locate() {
    t = cx.lane();
#ifndef GV_HOST_EMULATION
    asm volatile("" : "+v"(t));
#endif
    const int gs = group_stride(nA), w = cx.uniform(t);
    g = (w >= gs) + (w >= 2 * gs);
    j = t - g * gs;
    k = j - 1;
    s0 = g * SPW;
    oj = GS_N + (j + 2) * RS;
  }
  // whether the thread owns a level; the others take no part
  GV_MEM bool active() const { return j < L; }

  // The lane's addresses: its level's record, that of its group (one field
  // per group) and of its species (two).  Everything a lane reads at its own
  // or a neighbouring level is one of the three plus a constant, which is the
  // LDS instruction's offset.
  int oj;
  GV_MEM double &at(int slot, int d = 0) const { return (lds + oj)[slot + d * RS]; }
  GV_MEM double &own(int slot, int d = 0) const { return (lds + (oj + g))[slot + d * RS]; }
  GV_MEM double &spc(int slot, int q, int d = 0) const {
    return (lds + (oj + s0))[slot + q + d * RS];
  }
  // any level, any scalar
  GV_MEM double &x(int slot, int jj) const { return lds[GS_N + (jj + 2) * RS + slot]; }
  GV_MEM double &ion(int f, int jj) const { return x(GR_LEN + f, jj); }
  GV_MEM double &sc(int i) const { return lds[i]; }
  GV_MEM bool cell() const { return k >= 1 && k <= nA; }
  GV_MEM bool face() const { return k >= 0 && k <= nA; }
  GV_MEM void fail(int code, int level) { cx.report(error_key(col, code, level)); }

  // Geometry and per-level constants (advance_vertical.f90:84-151 and the
  // state-independent parts of the stage functions), as Column::setup.
  GV_MEM void setup(double alt, double grav, double invr, double dalt, double gam, double cmax,
                    double eddy, double mmm, double coslat) {
    const double centrifugal = (coslat * kp.omega) * (coslat * kp.omega);
    if (t == 0) sc(GS_COR) = 2 * coslat * kp.omega;
    eg = grav + centrifugal / invr;
    gm1 = gam - 1.0;
    const double rd = 1.0 / invr;
    idC = 1.0 / dalt;
    constexpr int ALT = GR_POOL, EG = ALT + 1, GAM = ALT + 2, CM = ALT + 3, RD = ALT + 4,
                  SL = ALT + 5;
    if (g == 0) {
      x(ALT, j) = alt;
      x(EG, j) = eg;
      x(GAM, j) = gam;
      x(CM, j) = cmax;
      x(RD, j) = rd;
      if (j == 0) sc(GS_MMM_M1) = mmm;
      if (j == 1) {
        sc(GS_MMM_0) = mmm;
        sc(GS_ALT0) = alt;
      }
    }
    cx.sync();
    const double dF = (j >= 1) ? alt - x(ALT, j - 1) : x(ALT, 1) - alt;
    mgh = (j >= 1) ? 0.5 * (eg + x(EG, j - 1)) : 0.0;
    if (g == 2) {  // spherical areas and volume, vertical_solver_ausm.f90:2029-2040
      const double LR = 0.5 * (rd + x(RD, j - 1)), RR = 0.5 * (rd + x(RD, j + 1));
      at(GR_AP) = RR * RR;
      at(GR_AM) = LR * LR;
      at(GR_IVOL) = 1.0 / ((1.0 / 3.0) * (RR * RR * RR - LR * LR * LR));
      at(GR_HF) = 0.35 * exp(-1.0 * (alt - sc(GS_ALT0)) / (45.0e+03));
    }
    if (g == 0) {
      at(GR_INVR) = invr;
      at(GR_EDDY) = eddy;
      x(GR_DF, j) = dF;
      x(GR_IF, j) = 1.0 / dF;
      x(GR_DC, j) = dalt;
      x(GR_CMF, j) = 0.5 * dmax(x(CM, j - 1), cmax);
      if (j == 1) sc(GS_MG0) = mgh;
      if (j == nA + 2) sc(GS_MGT1) = mgh;
      if (j == nA + 3) sc(GS_MGT2) = mgh;
    } else if (g == 1) {  // Kp/Ku blends, :1320-1352
      double vp = 0.0, vu = 0.0;
      if (cell()) {
        const double th = (1.0 + tanh((alt - 160.0e+03) / 15.0e+03));
        vp = MP_SCALE * exp(kp.log_min_kp + 0.5 * (kp.log_max_kp - kp.log_min_kp) * th);
        vu = exp(kp.log_min_ku + 0.5 * (kp.log_max_ku - kp.log_min_ku) * th);
      }
      x(GR_KP, j) = vp;
      x(GR_KU, j) = vu;
    }
    cx.sync();
    if (g == 0) {
      double dlg = 0.0;
      if (k >= 0 && k <= nA + 1)
        dlg = limiter_sel(kp.beta, (x(GAM, j + 1) - gam) * x(GR_IF, j + 1),
                          (gam - x(GAM, j - 1)) * x(GR_IF, j));
      x(SL, j) = dlg;
      if (j == 0) {
        bc_fwd_coefs(x(GR_DF, 3), x(GR_DF, 4), x(GR_DF, 5), x(GR_DF, 6), &sc(GS_CA));
        bc_fwd_coefs(x(GR_DF, 2), x(GR_DF, 3), x(GR_DF, 4), x(GR_DF, 5), &sc(GS_CB));
      }
      if (IONS && j == 1) {
        bc_bwd_coefs(x(GR_DF, nA + 1), x(GR_DF, nA), x(GR_DF, nA - 1), x(GR_DF, nA - 2),
                     &sc(GS_CTA));
        bc_bwd_coefs(x(GR_DF, nA + 2), x(GR_DF, nA + 1), x(GR_DF, nA), x(GR_DF, nA - 1),
                     &sc(GS_CTB));
      }
    } else if (g == 2) {  // 5-point gradient weights (:649-676)
      double w[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
      if (cell()) {
        const double h1 = x(GR_DF, j - 1), h2 = dF, h3 = x(GR_DF, j + 1), h4 = x(GR_DF, j + 2);
        const double m2 = h2 + h1, m3 = h3 + h2 + h1, m4 = h4 + h3 + h2 + h1;
        w[0] = (h2 * h3 * (h3 + h4)) / (h1 * m2 * m3 * m4);
        w[1] = -1.0 * (m2 * h3 * (h3 + h4)) / (h1 * h2 * (h2 + h3) * (h2 + h3 + h4));
        w[3] = m2 * h2 * (h4 + h3) / (m3 * (h2 + h3) * h3 * h4);
        w[4] = -1.0 * m2 * h2 * h3 / (m4 * (h2 + h3 + h4) * (h3 + h4) * h4);
        w[2] = (h2 * h3 * (h3 + h4) + m2 * h3 * (h3 + h4) - m2 * h2 * (h3 + h4) - m2 * h2 * h3) /
               (m2 * h2 * h3 * (h3 + h4));
      }
#pragma unroll
      for (int q = 0; q < 5; q++) x(GR_GLC + q, j) = w[q];
    }
    cx.sync();
    // gamma factors 1/(g-1), g/(g-1), 2(g-1)/(g+1) of face k|k+1 (:1535): its
    // left state in group 0, its right state in group 1
    if (g < 2 && face()) {
      const int jf = j + g;
      const double gs = x(GAM, jf) + (g == 0 ? 0.5 : -0.5) * x(SL, jf) * x(GR_DF, jf);
      gf[0] = 1.0 / (gs - 1.0);
      gf[1] = gs / (gs - 1.0);
      gf[2] = 2.0 * ((gs - 1.0) / (gs + 1.0));
    }
    nseg = (L / NSP) < 8 ? L / NSP : 8;  // >= 2: L >= 14 (nAlts >= 10)
    seg = (L - 2 + nseg - 1) / nseg;
    gseg = (j >= 2) ? (j - 2) / seg : 0;
    cx.sync();
  }

  // UseMSIS and tides set Temp(0) and the winds of level 0 before the
  // boundary conditions read them (set_vertical_bcs.Earth.f90:113-159; see
  // Column::bcs).  Before a barrier, on one lane.
  GV_MEM void bottom_values(bool first) {
    if (t != 1) return;
    double T0 = x(GU_T, 1);
    if (kp.msis || (kp.tides == 1 && !first)) T0 = sc(GS_MSIS + 6);
    if (kp.msis || kp.tides) {
      x(GU_VE, 1) = sc(GS_MSIS + 7);
      x(GU_VN, 1) = sc(GS_MSIS + 8);
    }
    if (kp.tides == 1) {
      T0 = sc(GS_TIDE) + T0;
      if (first && !kp.msis) sc(GS_MSIS + 6) = T0;
    } else if (kp.tides == 2) {
      T0 = sc(GS_TIDE);
    }
    x(GU_T, 1) = T0;
  }

  // set_vertical_bcs (set_vertical_bcs.Earth.f90:8-652, no BC perturbation):
  // the ghost levels of the state in LDS.  Exponentials and logarithms of
  // products of exponentials are taken in log space.  Ends in a barrier.
  GV_MEM void bcs() {
    locate();
    const int jn = nA + 1;
    // bottom on the first lanes of group 0, top on those of group 1: side by
    // side in different wavefronts
    const int top = group_stride(nA);
    if (t < NSP) {
      // bottom, one species per lane (:198-272, :277-344, :382-395)
      const int sp = t;
      const double *CA = &sc(GS_CA), *CB = &sc(GS_CB);
      const double dF1 = x(GR_DF, 2), dF0 = x(GR_DF, 1), dFm1 = x(GR_DF, 0);
      const double ln0 = x(GU_LN + sp, 1), ln1 = x(GU_LN + sp, 2), ln2 = x(GU_LN + sp, 3),
                   ln3 = x(GU_LN + sp, 4), ln4 = x(GU_LN + sp, 5), ln5 = x(GU_LN + sp, 6);
      double n0, nm1;
      if (photochemical(sp)) {
        double d = ln1 * CA[0] + ln2 * CA[1] + ln3 * CA[2] + ln4 * CA[3] + ln5 * CA[4];
        n0 = ln1 - dF1 * d;
        if (d <= 0.0) n0 = ln1;
        if (sp == S_NO && n0 < ln1 - 0.333) n0 = ln1 - 0.333;
        d = n0 * CB[0] + ln1 * CB[1] + ln2 * CB[2] + ln3 * CB[3] + ln4 * CB[4];
        nm1 = n0 - dF0 * d;
        if (d <= 0.0) nm1 = n0;
        if (sp == S_NO && nm1 < n0 - 0.333) nm1 = n0 - 0.333;
      } else {
        n0 = kp.msis ? sc(GS_MSIS + sp) : ln0;
        if (sp == S_O) {
          nm1 = n0;  // zero gradient below the boundary (:219-222)
        } else {
          // hydrostatic from the entry value, Temp(-1) = Temp(0)
          const double mm = 0.5 * (sc(GS_MMM_0) + sc(GS_MMM_M1));
          nm1 = ln0 + quot(-sc(GS_MG0) * mm, x(GU_T, 1) * KB) * dFm1;
        }
      }
      const double w1 = x(GU_W + sp, 2), w2 = x(GU_W + sp, 3), w3 = x(GU_W + sp, 4),
                   w4 = x(GU_W + sp, 5), w5 = x(GU_W + sp, 6);
      const double w0 =
          w1 - dF1 * (w1 * CA[0] + w2 * CA[1] + w3 * CA[2] + w4 * CA[3] + w5 * CA[4]);
      const double wm1 =
          w0 - dF0 * (w0 * CB[0] + w1 * CB[1] + w2 * CB[2] + w3 * CB[3] + w4 * CB[4]);
      const bool flip = photochemical(sp) && w1 > 0.0;
      x(GU_LN + sp, 1) = n0;
      x(GU_LN + sp, 0) = nm1;
      x(GU_W + sp, 1) = flip ? -1.0 * w1 : w0;
      x(GU_W + sp, 0) = flip ? -1.0 * w1 : wm1;
      const double m = kp.mass[sp];
      const double mm1 = m * exp(nm1), m0 = m * exp(n0);
      sc(GS_MN + sp) = mm1;
      sc(GS_MN + NSP + sp) = m0;
      sc(GS_MNW + sp) = mm1 * wm1;
      sc(GS_MNW + NSP + sp) = m0 * w0;
    } else if (t >= top && t < top + NSP) {
      // top, one species per lane (:429-441, :471-486)
      const int sp = t - top;
      const double tn = x(GU_T, jn), wn = x(GU_W + sp, jn), wnm1 = x(GU_W + sp, jn - 1);
      const bool flip = photochemical(sp) && wn < 0.0;
      const double m = kp.mass[sp];
      const double mkt = quot(m, tn * KB);
      const double l1 = x(GU_LN + sp, jn) + sc(GS_MGT1) * mkt * x(GR_DF, jn + 1);
      const double l2 = l1 + sc(GS_MGT2) * mkt * x(GR_DF, jn + 2);
      x(GU_LN + sp, jn + 1) = l1;
      x(GU_LN + sp, jn + 2) = l2;
      x(GU_W + sp, jn + 1) = flip ? -wn : wn;
      x(GU_W + sp, jn + 2) = flip ? -wnm1 : wn;
      sc(GS_MN + 2 * NSP + sp) = m * exp(l1);
      sc(GS_MN + 3 * NSP + sp) = m * exp(l2);
    }
    if (IONS) {
      if (j <= 1) {  // bottom: zero-gradient ions (:277-281)
#pragma unroll
        for (int q = 0; q < IPW; q++) own(GR_LEN + NG * q) = ion(g + NG * q, 2);
      }
      // TEC of the column in 1e16 m^-2 (:498-503), in the reference's order
      if (t == NSP + top && plasma) {
        double tec = 0.0;
        for (int jj = 2; jj <= nA + 1; jj++) {
          const double v = kp.improved_ions ? ion(0, jj) : exp(ion(0, jj));
          tec = tec + x(GR_DF, jj) * v;
        }
        sc(GS_TEC) = tec / 1e16;
      }
    }
    // the ghost lanes below are of the wavefronts of the species' lanes they read
    cx.wave_sync();
    if (t < 2 || (t >= top && t < top + 2)) {
      // ghost levels -1, 0, nAlts+1, nAlts+2: LogRho and bulk winds
      // (:346-375, :420-463, :598-604)
      const int q = t < 2 ? t : t - top + 2, jg = t < 2 ? t : nA + q;
      const double *mn = &sc(GS_MN + NSP * q);
      const double sr = ((mn[0] + mn[1]) + (mn[2] + mn[3])) + (mn[4] + mn[5]);
      x(GU_LR, jg) = ln(sr);
      if (t < 2) {
        const double *mw = &sc(GS_MNW + NSP * q);
        x(GU_VU, jg) = quot(((mw[0] + mw[1]) + (mw[2] + mw[3])) + (mw[4] + mw[5]), sr);
        if (!kp.msis) {
          if (!kp.tides) {  // :139-142
            x(GU_VE, jg) = 0.0;
            x(GU_VN, jg) = 0.0;
          } else if (t == 0) {  // the tides' level 0, Vel(-1) = Vel(0)
            x(GU_VE, 0) = x(GU_VE, 1);
            x(GU_VN, 0) = x(GU_VN, 1);
          }
        } else if (t == 0) {
          // Vel(-1) east and north extrapolated from levels 0..4 (:364-375)
          const double *CB = &sc(GS_CB);
          const double dF0 = x(GR_DF, 1);
          for (int d = 0; d < 2; d++) {
            const int f = GU_VE + d;
            const double v0 = x(f, 1);
            const double dv = v0 * CB[0] + x(f, 2) * CB[1] + x(f, 3) * CB[2] + x(f, 4) * CB[3] +
                              x(f, 5) * CB[4];
            x(f, 0) = v0 - dF0 * dv;
          }
        }
        if (t == 0) x(GU_T, 0) = x(GU_T, 1);
      } else {
        x(GU_VE, jg) = x(GU_VE, jn);
        x(GU_VN, jg) = x(GU_VN, jn);
        x(GU_VU, jg) = fabs(x(GU_VU, jn));
        x(GU_T, jg) = x(GU_T, jn);
      }
    }
    if (IONS && t >= top && t < top + NI) ion_top_bc(t - top);
    cx.sync();
  }

  // Top ghost levels of one ion (set_vertical_bcs.Earth.f90:505-649), as
  // Column::ion_top_bc.
  GV_MEM void ion_top_bc(int q) {
    const bool improved = kp.improved_ions != 0;
    const bool keep = plasma && sc(GS_TEC) < kp.min_tec;
    const double dFn = x(GR_DF, nA + 1);
    for (int u = 0; u < 2; u++) {
      const int jk = nA + 2 + u;  // level nAlts+1+u
      const double *C = &sc(u ? GS_CTB : GS_CTA);
      double n[6];
      if (improved) {
        double mn = ion(q, jk - 5);
        for (int jj = jk - 4; jj <= jk; jj++)
          if (ion(q, jj) < mn) mn = ion(q, jj);
        if (mn < 0.0) {  // check_for_negative_densities, :608-649
          if (ion(q, jk - 6) < 0.0) fail(GITM_VERT_ENEGION, jk - 1);
          for (int jj = jk - 5; jj <= jk - 1; jj++) {
            if (ion(q, jj) < 0.0) {
              if (ion(q, jj - 1) > 0.0 && ion(q, jj + 1) > 0.0)
                ion(q, jj) = (ion(q, jj - 1) + ion(q, jj + 1)) / 2.0;
              else
                ion(q, jj) = ion(q, jj - 1) * 0.95;
            }
          }
          if (ion(q, jk) < 0.0) ion(q, jk) = ion(q, jk - 1) * 0.95;
        }
      }
#pragma unroll
      for (int i = 0; i < 6; i++) n[i] = improved ? ln(ion(q, jk - i)) : ion(q, jk - i);
      double dn = C[0] * n[1] + C[1] * n[2] + C[2] * n[3] + C[3] * n[4] + C[4] * n[5];
      if (!keep) {
        if (dn > -0.001 * n[0] / dFn) dn = -0.001 * n[0] / dFn;
        const double n0 = n[1] + dn * x(GR_DF, jk);
        ion(q, jk) = improved ? exp(n0) : n0;
      }
    }
  }

  // One field of the RK4 driver (vertical_solver_ausm.f90:167-417): stage
  // input = Y + (New - U); the last stage gives (1/3)(-Y + S2 + 2 S3 + S4 +
  // (New - U)).
  GV_MEM double commit(int stg, double nv, double u, double y, double &a) const {
    const double d = nv - u;
    if (stg == 3) return (1.0 / 3.0) * (a + d);
    const double nxt = y + d;
    a = (stg == 0) ? -1.0 * y + nxt : a + (stg == 1 ? 2.0 * nxt : nxt);
    return nxt;
  }

  // Limited slope of a level's field (calc_rusanov_alts_*, :1007-1090) and
  // its states at the level's two faces.
  GV_MEM void rusanov_states(const double *v, double &right, double &left) const {
    const double vm2 = v[-2 * RS], vm1 = v[-RS], v0 = v[0], v1 = v[RS], v2 = v[2 * RS];
    const double iF0 = at(GR_IF), iF1 = at(GR_IF, 1);
    double up = (v1 - v0) * iF1, dn = (v0 - vm1) * iF0;
    if (cell()) {
      up = (iF1 * 2.0) * (FACT1 * (v1 - v0) - FACT2 * (v2 - vm1));
      dn = (iF0 * 2.0) * (FACT1 * (v0 - vm1) - FACT2 * (v1 - vm2));
    }
    const double dl = (k >= 0 && k <= nA + 1) ? limiter_sel(kp.beta, up, dn) : 0.0;
    right = v0 - 0.5 * dl * at(GR_DF);
    left = v0 + 0.5 * dl * at(GR_DF, 1);
  }
  // Gradient and dissipation from the states R0, L1 of the level's own faces
  // and the neighbours' (rslot, lslot of the group).
  GV_MEM void rusanov_diff(double R0, double L1, int rslot, int lslot, double &grad,
                           double &diff) const {
    const double L0 = own(lslot, -1), R1 = own(rslot, 1);
    grad = 0.5 * (L1 + R1 - L0 - R0) * idC;
    diff = (at(GR_CMF, 1) * (R1 - L1) - at(GR_CMF) * (R0 - L0)) * idC;
  }

  // States of face k|k+1 of a field with the values fm1, f0, f1, f2 on levels
  // k-1..k+2 (calc_kt_facevalues, :2073-2117).
  struct FaceGeo {
    double iF0, iF1, iF2, hF0, hF1;  // hF: half the distances below and above
  };
  GV_MEM void kt(const FaceGeo &q, double fm1, double f0, double f1, double f2, double &l,
                 double &r) const {
    const double mid = (f1 - f0) * q.iF1;
    const double d0 = limiter_sel(kp.beta, mid, (f0 - fm1) * q.iF0);
    const double d1 = limiter_sel(kp.beta, (f2 - f1) * q.iF2, mid);
    l = f0 + d0 * q.hF0;
    r = f1 - d1 * q.hF1;
  }

  // advance_vertical_1stage_ausm (vertical_solver_ausm.f90:436-999) with
  // calc_all_fluxes_hydro (:1093-2070) and the RK4 combination: the state in
  // LDS becomes the next stage's on cells.  The phases end in barriers; the
  // last one is the caller's.
  GV_MEM void stage(double dtin, double idt, int stg) {
    locate();
    // --- A: own densities, slopes, hydrostatic factors
    double rhos[SPW];
    {
      double ns2[SPW];
#pragma unroll
      for (int q = 0; q < SPW; q++) {
        ns2[q] = exp(spc(GU_LN, q));
        rhos[q] = kp.mass[s0 + q] * ns2[q];
        if (j == 1) spc(GP_HNS, q) = ns2[q];
        GV_HERE(rhos[q]);
      }
      own(GP_NT) = ns2[0] + ns2[1];
    }
    double rr, rl, ir = 0.0, il = 0.0;
    rusanov_states(&own(GU_T), rr, rl);
    own(GP_RF) = rr;
    own(GP_LF) = rl;
    if (IONS && g < NI_ADVECT) {
      rusanov_states(&own(GR_LEN), ir, il);
      own(GP_IRF) = ir;
      own(GP_ILF) = il;
    }
    {
      // factor of level k over k-1 (level -1: over level 0)
      const double T = at(GU_T), to = j == 0 ? at(GU_T, 1) : at(GU_T, -1), dF = at(GR_DF);
      const double ratio = quot(to, T), ikt = recip(KB * (0.5 * (T + to)));
      if (j != 1) {
        const double h = dF * (j == 0 ? sc(GS_MG0) : mgh) * ikt;
        const double mm = 0.5 * (sc(GS_MMM_M1) + sc(GS_MMM_0));
#pragma unroll
        for (int q = 0; q < SPW; q++)
          spc(GP_B, q) = ratio * exp(j == 0 ? -(mm * h) : kp.mass[s0 + q] * h);
      }
      if (g == 2) at(GR_LTK) = ln(T * KB);
    }
    cx.sync();
    // --- B: gradients; products of the hydrostatic factors within segments
    // kept: the total energy (group 0), the wind's dissipation (1, 2)
    double grad, kept;
    rusanov_diff(rr, rl, GP_RF, GP_LF, grad, kept);
    if (IONS && cell()) {
#pragma unroll
      for (int q = 0; q < IPW; q++) {
        double &u = own(GR_LEN + NG * q);
        double nv = u;
        if (q == 0 && g < NI_ADVECT) {
          double gi, di;
          rusanov_diff(ir, il, GP_IRF, GP_ILF, gi, di);
          nv = u - dtin * (ivu * gi) + dtin * di;
        }
        u = commit(stg, nv, u, Yi[q], Ai[q]);
      }
    }
    double rho = exp(at(GU_LR));
    GV_HERE(rho);
    if (g == 0) {
      at(GR_GT) = grad;
      const double nt = (at(GP_NT) + at(GP_NT + 1)) + at(GP_NT + 2);
      const double vu = at(GU_VU), vn = at(GU_VN), ve = at(GU_VE);
      kept = quot(nt * KB * at(GU_T), gm1) + 0.5 * rho * (vu * vu + vn * vn + ve * ve);
    }
    GV_HERE(kept);
    // (in group 2, which has the least to do here); the factors of eight levels
    // are read at once, so that the LDS latency is paid once
    if (g == 2 && j < nseg * NSP) {
      const int h = j / NSP, s = j - h * NSP;
      const int lo = 2 + h * seg, n = (lo + seg < L ? seg : L - lo);
      double p = (h == 0) ? x(GP_HNS + s, 1) : 1.0;
      double *r = &x(s, lo);
      for (int i0 = 0; i0 < n; i0 += 8, r += 8 * RS) {
        double f[8];
#pragma unroll
        for (int i = 0; i < 8; i++) f[i] = r[(i0 + i < n ? i : 0) * RS + GP_B];
#pragma unroll
        for (int i = 0; i < 8; i++) {
          p = p * f[i];
          if (i0 + i < n) r[i * RS + GP_HNS] = p;
        }
      }
    }
    cx.sync();
    // --- C: hydrostatic densities (:694-751) and the deviation from them
    double dev[SPW];
    int sub = 0;  // bit q: SubtractHydrostatic of species s0 + q
    int below = gseg;  // segments below the level's
    GV_HERE(below);
#pragma unroll
    for (int q = 0; q < SPW; q++) {
      double hns;
      if (j >= 2) {
        // the product up to the end of the segment below, times the level's own
        hns = spc(GP_HNS, q);
        double e[7];
#pragma unroll
        for (int h = 0; h < 7; h++)
          e[h] = x(GP_HNS + s0 + q, 1 + (h < below ? (h + 1) * seg : 0));
        double p = e[0];
#pragma unroll
        for (int h = 1; h < 7; h++) p = (h < below) ? p * e[h] : p;
        hns = (below > 0) ? p * hns : hns;
      } else {
        hns = x(GP_HNS + s0 + q, 1);
        if (j == 0) hns = hns * spc(GP_B, q);
      }
      spc(GP_LH, q) = ln(hns * KB * at(GU_T));
      const double hrhos = kp.mass[s0 + q] * hns;
      dev[q] = rhos[q] - hrhos;
      if (!(fabs(dev[q]) > rhos[q])) sub |= 1 << q;
      GV_HERE(dev[q]);
      GV_ORDER();
    }
    reinterpret_cast<int &>(own(GP_SUB)) = sub;
    cx.sync();
    // --- D: face states (:2073-2117) and the groups' sums over the species
    double RSL[SPW], RSR[SPW], PSL[SPW], PSR[SPW], HL[SPW], HR[SPW], VL[SPW], VR[SPW];
    const int subUp = reinterpret_cast<int &>(own(GP_SUB, 1));  // flags of cell k+1
    {
      const FaceGeo fg = {at(GR_IF), at(GR_IF, 1), at(GR_IF, 2), 0.5 * at(GR_DF),
                          0.5 * at(GR_DF, 1)};
      double mL = 0.0, mR = 0.0;
#pragma unroll
      for (int q = 0; q < SPW; q++) {
        double l, r;
        kt(fg, spc(GP_LH, q, -1), spc(GP_LH, q), spc(GP_LH, q, 1), spc(GP_LH, q, 2), l, r);
        HL[q] = exp(l);
        HR[q] = exp(r);
        GV_HERE(HL[q]);
        GV_HERE(HR[q]);
        GV_ORDER();
        kt(fg, spc(GU_W, q, -1), spc(GU_W, q), spc(GU_W, q, 1), spc(GU_W, q, 2), VL[q], VR[q]);
        const double nm1 = spc(GU_LN, q, -1), n0 = spc(GU_LN, q), n1 = spc(GU_LN, q, 1),
                     n2 = spc(GU_LN, q, 2);
        kt(fg, nm1 + at(GR_LTK, -1), n0 + at(GR_LTK), n1 + at(GR_LTK, 1), n2 + at(GR_LTK, 2),
           l, r);
        PSL[q] = exp(l);
        PSR[q] = exp(r);
        GV_HERE(PSL[q]);
        GV_HERE(PSR[q]);
        GV_HERE(VL[q]);
        GV_HERE(VR[q]);
        GV_ORDER();
        const double lm = kp.lmass[s0 + q];
        kt(fg, lm + nm1, lm + n0, lm + n1, lm + n2, l, r);
        RSL[q] = exp(l);
        RSR[q] = exp(r);
        GV_HERE(RSL[q]);
        GV_HERE(RSR[q]);
        mL = (q == 0) ? RSL[q] * VL[q] : mL + RSL[q] * VL[q];
        mR = (q == 0) ? RSR[q] * VR[q] : mR + RSR[q] * VR[q];
        GV_ORDER();
      }
      // (NG left sums, NG right ones, interleaved: slot 2 h + side of group h)
      spc(GP_RSUM, 0) = RSL[0] + RSL[1];
      spc(GP_RSUM, 1) = RSR[0] + RSR[1];
      spc(GP_PSUM, 0) = PSL[0] + PSL[1];
      spc(GP_PSUM, 1) = PSR[0] + PSR[1];
      spc(GP_MSUM, 0) = mL;
      spc(GP_MSUM, 1) = mR;
      if (g > 0) {
        double l, r;
        kt(fg, own(GU_T, -1), own(GU_T), own(GU_T, 1), own(GU_T, 2), l, r);
        spc(GR_VEL - 2, 0) = l;
        spc(GR_VEL - 2, 1) = r;
      }
    }
    cx.sync();
    // --- E: bulk face values (:1505-1655): the left state in group 0, the
    // right one in group 1; the friction's powers of Temp in group 2
    if (g < 2) {
      const double R = (own(GP_RSUM) + own(GP_RSUM + 2)) + own(GP_RSUM + 4);
      const double P = (own(GP_PSUM) + own(GP_PSUM + 2)) + own(GP_PSUM + 4);
      const double iR = recip(R);
      const double VU = ((own(GP_MSUM) + own(GP_MSUM + 2)) + own(GP_MSUM + 4)) * iR;
      const double VE = own(GR_VEL), VN = own(GR_VNL);
      const double k2 = VU * VU + VE * VE + VN * VN;
      const double Ht = 0.5 * k2 + (gf[1] * P) * iR;
      const double c = sqrt(gf[2] * Ht);
      own(GR_RL) = R;
      own(GR_EPL) = (gf[0] * P + 0.5 * R * k2) + P;
      own(GR_CSL) = quot(c * c, dmax(c, g == 0 ? VU : -VU));
    } else {
      at(GR_IRLR) = recip(((at(GP_RSUM) + at(GP_RSUM + 2)) + at(GP_RSUM + 4)) +
                          ((at(GP_RSUM + 1) + at(GP_RSUM + 3)) + at(GP_RSUM + 5)));
      double pw[6];
      cx.diff_powers(at(GU_T), -1.0, pw);
#pragma unroll
      for (int u = 0; u < 6; u++) at(GP_PW + u) = pw[u];
    }
    cx.sync();
    // --- F: AUSM+-up fluxes of face k|k+1 (:1659-1970).  The P12 side belongs
    // to cell k; the M12 side to cell k+1 (with its Kp, Ku, dAlt_C and flags),
    // whose lane reads it after the barrier.
    double FRp[SPW], FMp[SPW], NPp[SPW];
#pragma unroll
    for (int q = 0; q < SPW; q++) FRp[q] = FMp[q] = NPp[q] = 0.0;
    if (face()) {
      const double CS = dmin(at(GR_CSL), at(GR_CSR));
      const double icS = recip(CS);
      double bp = 0.0, bm = 0.0;
#pragma unroll
      for (int q = 0; q < SPW; q++) {
        const double MPS = 0.5 * (PSL[q] + PSR[q]), MHPS = 0.5 * (HL[q] + HR[q]);
        const double RS2 = RSL[q] + RSR[q], MRS = (0.5 * MP_SCALE) * RS2;
        const double ML = VL[q] * icS, MR = VR[q] * icS;  // :1689-1706
        const double M2 = 0.5 * (ML * ML + MR * MR);
        const double MZ = sqrt(dmin(1.0, dmax(M2, 1.0e-19)));
        const double FA = MZ * (2.0 - MZ);
        // :1789-1819 (16*LiouBeta = 2)
        const double m4p = 0.25 * ((ML + 1.0) * (ML + 1.0)) *
                           (1.0 - 2.0 * (-0.25 * ((ML - 1.0) * (ML - 1.0))));
        const double m4n = -0.25 * ((MR - 1.0) * (MR - 1.0)) *
                           (1.0 + 2.0 * (0.25 * ((MR + 1.0) * (MR + 1.0))));
        const double MF4P = fabs(ML) >= 1.0 ? 0.5 * (ML + fabs(ML)) : m4p;
        const double MF4N = fabs(MR) >= 1.0 ? 0.5 * (MR - fabs(MR)) : m4n;
        const double f1 = dmax((1.0 - M2), 0.0);
        const double pdh = (PSR[q] - HR[q]) - (PSL[q] - HL[q]), pd = PSR[q] - PSL[q];
        const double fmL = RSL[q] * VL[q], fmR = RSR[q] * VR[q];
        const double cr = 0.5 * CS * (fmR - fmL);
        const double mcs = MRS * CS, facs = FA * CS, mf = MF4P + MF4N;
        {
          const bool sh = (sub >> q) & 1;
          const double MP =
              quot(at(GR_KP) * f1 * (sh ? pdh : pd), mcs * (facs + at(GR_DC) * idt));
          const double NV = CS * (mf - MP);
          NPp[q] = (sh ? (MPS - MHPS) : MPS) - at(GR_KU) * cr;
          FRp[q] = (NV >= 0.0 ? RSL[q] : RSR[q]) * NV;
          FMp[q] = (NV >= 0.0 ? fmL : fmR) * NV;
          bp = (q == 0) ? RS2 * NV : bp + RS2 * NV;
          GV_HERE(NPp[q]);
          GV_HERE(FRp[q]);
          GV_HERE(FMp[q]);
        }
        {
          const bool sh = (subUp >> q) & 1;
          const double MP =
              quot(at(GR_KP, 1) * f1 * (sh ? pdh : pd), mcs * (facs + at(GR_DC, 1) * idt));
          const double NV = CS * (mf - MP);
          spc(GP_NP, q) = (sh ? (MPS - MHPS) : MPS) - at(GR_KU, 1) * cr;
          spc(GP_FR, q) = (NV >= 0.0 ? RSL[q] : RSR[q]) * NV;
          spc(GP_FM, q) = (NV >= 0.0 ? fmL : fmR) * NV;
          bm = (q == 0) ? RS2 * NV : bm + RS2 * NV;
        }
        GV_ORDER();
      }
      own(GP_BP) = bp;
      own(GP_BM) = bm;
    }
    GV_ORDER();
    // d ln(rho_s/rho)/dz (:649-688), here where the face states are done with
    // and the old LogNS still in place
    double glc[SPW];
#pragma unroll
    for (int q = 0; q < SPW; q++) {
      const double lm = kp.lmass[s0 + q];
      double a = at(GR_GLC) * ((lm + spc(GU_LN, q, -2)) - at(GU_LR, -2));
      a = a + at(GR_GLC + 1) * ((lm + spc(GU_LN, q, -1)) - at(GU_LR, -1));
      a = a + at(GR_GLC + 2) * ((lm + spc(GU_LN, q)) - at(GU_LR));
      a = a + at(GR_GLC + 3) * ((lm + spc(GU_LN, q, 1)) - at(GU_LR, 1));
      glc[q] = a + at(GR_GLC + 4) * ((lm + spc(GU_LN, q, 2)) - at(GU_LR, 2));
      GV_HERE(glc[q]);
    }
    cx.sync();
    // --- G: flux divergences (:2042-2068), new densities and the species
    // winds before friction (:802-930).  The new densities and winds take the
    // LDS places of the old LogNS and VertVel, which nothing reads any more.
    double nrs[SPW], W0[SPW], LN[SPW], ef = 0.0;
    if (cell()) {
      // energy (group 0), east and north momentum (1, 2): flux of the upper
      // face, then of the lower one (:1973-2026)
      double fl[2];
#pragma unroll
      for (int u = 0; u < 2; u++) {
        const int b = u ? GP_BM : GP_BP;
        const double bnv = ((at(b, -u) + at(b + 1, -u)) + at(b + 2, -u)) * at(GR_IRLR, -u);
        const bool pos = bnv >= 0.0;
        double q;
        if (g == 0) {
          q = pos ? at(GR_EPL, -u) : at(GR_EPR, -u);
        } else {
          const double *v = &spc(GR_VEL - 2, 0, -u);
          q = pos ? at(GR_RL, -u) * v[0] : at(GR_RR, -u) * v[1];
        }
        fl[u] = q * bnv;
      }
      const double ap = at(GR_AP), am = at(GR_AM), ivol = at(GR_IVOL);
      ef = (ap * fl[0] - am * fl[1]) * ivol;
      GV_HERE(ef);
      const double ve = at(GU_VE), vn = at(GU_VN), gradT = at(GR_GT);
#pragma unroll
      for (int q = 0; q < SPW; q++) {
        const double im = kp.imass[s0 + q];
        LN[q] = spc(GU_LN, q);
        W0[q] = spc(GU_W, q);
        const double rsf = (ap * FRp[q] - am * spc(GP_FR, q, -1)) * ivol;
        const double msf = (ap * FMp[q] - am * spc(GP_FM, q, -1)) * ivol +
                           (NPp[q] - spc(GP_NP, q, -1)) * idC;
        nrs[q] = rhos[q] - dtin * rsf;
        const double src = ((sub >> q) & 1) ? dev[q] : rhos[q];
        const double nm = rhos[q] * W0[q] - dtin * msf + dtin * src * eg;
        double ww = nm / nrs[q];  // (nrs may lie below quot's range)
        ww = ww + dtin * (vn * vn + ve * ve) * at(GR_INVR);
        if (kp.coriolis) ww = ww + dtin * (sc(GS_COR) * ve);
        ww = ww - dtin * (kp.tdc[s0 + q] * KB * gradT) * im;
        spc(GU_LN, q) = nrs[q] * im;
        spc(GU_W, q) = ww;
        GV_ORDER();
      }
      own(GP_NRHO) = nrs[0] + nrs[1];
    }
    cx.sync();
    // --- H: friction solve (group 0); new logarithms, horizontal winds and
    // LogRho (groups 1, 2; :931-960)
    double inrho = 0.0, nrho = 0.0, nnt = 0.0, w[NSP];
    if (cell()) {
      nrho = (at(GP_NRHO) + at(GP_NRHO + 1)) + at(GP_NRHO + 2);
      inrho = recip(nrho);
#pragma unroll
      for (int q = 0; q < SPW; q++) {
        spc(GP_KGLC, q) = glc[q];
        spc(GP_KNRS, q) = nrs[q];
        spc(GP_KW, q) = W0[q];
        spc(GP_KL, q) = LN[q];
      }
      GV_ORDER();
      if (g == 0) {
        double ns[NSP], pw[6];
#pragma unroll
        for (int s = 0; s < NSP; s++) {
          ns[s] = at(GU_LN + s);
          w[s] = at(GU_W + s);
          pw[s] = at(GP_PW + s);
        }
        nnt = ((ns[0] + ns[1]) + (ns[2] + ns[3])) + (ns[4] + ns[5]);
        if (kp.friction) {
          const double sum = friction_solve(kp, dtin, ns, nnt, at(GU_T), pw, w);
          if (!(fabs(sum) < __builtin_inf()) && friction_singular(&at(GU_LN), at(GU_T)))
            fail(GITM_VERT_ESINGULAR, k);
#pragma unroll
          for (int s = 0; s < NSP; s++) at(GU_W + s) = w[s];
        }
      } else {
        const int sl = (g - 1) * 3;
        double *const n = lds + (oj + sl);
#pragma unroll
        for (int q = 0; q < 3; q++) {
          n[GP_KLN + q] = ln(n[GU_LN + q]);
          GV_ORDER();
        }
        const double v = own(GU_T);
        double nv = (rho * v - dtin * ef) * inrho;
        nv = nv + at(GR_HF) * dtin * kept;
        at(GR_VEL + g - 1) = nv;
        own(GU_T) = commit(stg, nv, v, Yr[0], Ar[0]);
        if (g == 1) {
          double sr = 0.0;
#pragma unroll
          for (int s = 0; s < NSP; s++) sr = sr + kp.mass[s] * at(GU_LN + s);
          at(GU_LR) = commit(stg, ln(sr), at(GU_LR), Yr[1], Ar[1]);
        }
      }
    }
    cx.sync();
    // --- I: species winds after friction (:961-975), bulk vertical wind and
    // temperature (group 0, :976-997)
    if (cell()) {
      const double ec = kp.friction ? at(GR_EDDY) : 0.0;
      if (g == 0) {
        double m[NSP];
#pragma unroll
        for (int s = 0; s < NSP; s++) {
          const double ww = dmin(kp.maxvv, dmax(-kp.maxvv, w[s] - ec * at(GP_KGLC + s)));
          m[s] = ww * at(GP_KNRS + s);
        }
        const double nvu = (((m[0] + m[1]) + (m[2] + m[3])) + (m[4] + m[5])) * inrho;
        const double nvE = at(GR_VEL), nvN = at(GR_VEL + 1), vu = at(GU_VU);
        const double nte = kept - dtin * ef + dtin * rho * vu * eg;
        const double np = (nte - 0.5 * nrho * (nvu * nvu + nvN * nvN + nvE * nvE)) * gm1;
        at(GU_VU) = commit(stg, nvu, vu, Yr[1], Ar[1]);
        at(GU_T) = commit(stg, quot(np, KB * nnt), at(GU_T), Yr[0], Ar[0]);
      }
#pragma unroll
      for (int q = 0; q < SPW; q++) {
        const double ww = dmin(kp.maxvv, dmax(-kp.maxvv, spc(GU_W, q) - ec * spc(GP_KGLC, q)));
        spc(GU_W, q) = commit(stg, ww, spc(GP_KW, q), Yw[q], Aw[q]);
        spc(GU_LN, q) = commit(stg, spc(GP_KLN, q), spc(GP_KL, q), Yn[q], An[q]);
      }
    }
    if (IONS && !cell()) {  // the boundary reads the step's first ghost ions
#pragma unroll
      for (int q = 0; q < IPW; q++) own(GR_LEN + NG * q) = Yi[q];
    }
  }

  // advance_vertical_1d_ausm, vertical_solver_ausm.f90:26-433.
  GV_MEM void step() {
    bottom_values(true);
    cx.sync();
    bcs();
#pragma unroll
    for (int q = 0; q < SPW; q++) {
      Yn[q] = spc(GU_LN, q);
      Yw[q] = spc(GU_W, q);
      An[q] = Aw[q] = 0.0;
    }
    Yr[0] = own(GU_T);
    Yr[1] = own(GU_VU);
    Ar[0] = Ar[1] = 0.0;
    if (IONS) {
#pragma unroll
      for (int q = 0; q < IPW; q++) {
        Yi[q] = own(GR_LEN + NG * q);
        Ai[q] = 0.0;
      }
    }
    // dt may be 0 (a member's step from the prep, at EndTime): what it divides
    // is then so large that MPn is 0, and recip takes no infinite operand
    const double idt = dmax(-0x1p300, dmin(1.0 / dt, 0x1p300));
#pragma unroll 1
    for (int stg = 0; stg < 4; stg++) {
      stage(stg == 2 ? dt : 0.5 * dt, stg == 2 ? idt : 2.0 * idt, stg);  // :160-377
      bottom_values(false);
      cx.sync();
      bcs();
    }
  }
};

// One column of `io` (col = its index there, n_alts its nAlts): gather,
// n_steps steps of Dt = dt, scatter (advance_vertical.f90:84-219).  err_col:
// the column number that error reports carry.
template <bool IONS, class Ctx>
GV_FN void run_group_column(Ctx &cx, const KParams &kp, const gitm_vert_columns &io, int col,
                            double *lds, double dt, int err_col, int n_alts) {
  GroupColumn<IONS, Ctx> c(cx, kp, lds, err_col, dt, n_alts);
  if (!c.active()) return;
  // the column's indices, formed anew where they are used: kept, the offsets
  // of 25 fields would hold more scalar registers through the step than there
  // are
  const auto at_column = [&](int &ci, int &cj, int &cb) {
    int q = col;
#ifndef GV_HOST_EMULATION
    asm volatile("" : "+s"(q));
#endif
    ci = q % io.n_lons;
    cj = (q / io.n_lons) % io.n_lats;
    cb = q / (io.n_lons * io.n_lats);
  };
  int ci, cj, cb;
  at_column(ci, cj, cb);
  const int g = c.g, j = c.j, k = c.k, nA = c.nA, s0 = c.s0;
  double nds[SPW], r0, r1 = 0.0;  // r0, r1: the group's own fields
  {
#define GV_LD(F) (*fld(io.F, col_base(io.F, ci, cj, cb), k, 0))
    const long long bn = col_base(io.ndensity_s, ci, cj, cb);
    const long long bw = col_base(io.vertical_velocity, ci, cj, cb);
    const long long bv = col_base(io.velocity, ci, cj, cb);
    double w[SPW];
#pragma unroll
    for (int q = 0; q < SPW; q++) {
      nds[q] = *fld(io.ndensity_s, bn, k, s0 + q);
      w[q] = *fld(io.vertical_velocity, bw, k, s0 + q);
    }
    if (g == 0) {
      r0 = GV_LD(temperature);
      r1 = *fld(io.velocity, bv, k, 2);
    } else {
      r0 = *fld(io.velocity, bv, k, g - 1);
      if (g == 1) r1 = GV_LD(rho);
    }
    const double alt = GV_LD(altitude), grav = GV_LD(gravity), dalt = GV_LD(dalt),
                 gam = GV_LD(gamma);
    const double invr = GV_LD(inv_radial_distance), eddy = c.cell() ? GV_LD(eddy) : 0.0;
    const double cmax = (g == 0 && k >= 0 && k <= nA + 1) ? GV_LD(cmax) : 0.0;
    const double mmm = (g == 0 && j <= 1) ? GV_LD(mean_major_mass) : 0.0;
    const double coslat = io.cos_latitude.ptr[col_base(io.cos_latitude, ci, cj, cb)];
    if (IONS) {
      // LogINS (linear densities with UseImprovedIonAdvection) and IVel(up)
      // (:120-130); SZA and MLat of the column for the nighttime BCs (:84-85)
      const long long bi = col_base(io.idensity_s, ci, cj, cb);
#pragma unroll
      for (int q = 0; q < IPW; q++) {
        const double v = *fld(io.idensity_s, bi, k, g + NG * q);
        c.own(GR_LEN + NG * q) = kp.improved_ions ? v : ln(v);
      }
      if (c.cell() && g < NI_ADVECT)
        c.ivu = *fld(io.ivelocity, col_base(io.ivelocity, ci, cj, cb), k, 2);
      if (kp.nighttime_ion_bcs) {
        const double sza = io.sza.ptr[col_base(io.sza, ci, cj, cb)];
        const double mlat = io.mlat.ptr[col_base(io.mlat, ci, cj, cb)];
        c.plasma =
            sza > PI / 2 && ((mlat > 30.0 && mlat < 70.0) || (mlat > -60.0 && mlat < -30.0));
      }
    }
    // the caller's MSIS values of level 0, or the tides' winds after them
    // (set_vertical_bcs.Earth.f90:113-159)
    if (kp.msis && c.t < 9) {
      const gitm_vert_field &f = io.msis_bc;
      c.sc(GS_MSIS + c.t) = f.ptr[col_base(f, ci, cj, cb) + (long long)c.t * f.s_comp];
    }
    if (kp.tides && c.t >= 7 && c.t < 10) {
      const gitm_vert_field &f = c.t == 7 ? io.tides_east : c.t == 8 ? io.tides_north
                                                                     : io.tides_temp;
      c.sc(c.t == 9 ? GS_TIDE : GS_MSIS + c.t) = *fld(f, col_base(f, ci, cj, cb), 0, 0);
    }
    c.setup(alt, grav, invr, dalt, gam, cmax, eddy, mmm, coslat);
#pragma unroll
    for (int q = 0; q < SPW; q++) c.spc(GU_W, q) = w[q];
  }
  for (int step = 0; step < kp.n_steps; step++) {
    // gather (:96-116): the densities must be positive on every level
    bool bad = false;
#pragma unroll
    for (int q = 0; q < SPW; q++) bad = bad || !(nds[q] > 0.0);
    if (cx.sync_or(bad)) {
      c.own(GP_SUB) = bad ? k : 1 << 20;
      cx.sync();
      if (c.t == 0) {
        double lo = 1 << 20;
        for (int q = 0; q < c.L; q++)
          for (int h = 0; h < NG; h++) lo = dmin(lo, c.x(GP_SUB + h, q));
        c.fail(GITM_VERT_ENONPOSITIVE, (int)lo);
      }
      return;  // the column is left as it was
    }
#pragma unroll
    for (int q = 0; q < SPW; q++) c.spc(GU_LN, q) = ln(nds[q]);
    c.own(GU_T) = (g == 0) ? r0 * GV_LD(temp_unit) : r0;
    if (g == 0) c.at(GU_VU) = r1;
    if (g == 1) c.at(GU_LR) = ln(r1);
    cx.sync();
    c.step();
    // scatter (:163-185)
    at_column(ci, cj, cb);
#pragma unroll
    for (int q = 0; q < SPW; q++) nds[q] = exp(c.spc(GU_LN, q));
    r0 = c.own(GU_T);
    r1 = c.own(GU_VU);
    if (g == 0) r0 = r0 / GV_LD(temp_unit);
    if (g == 1) r1 = exp(r1);
    if (IONS) {
      // IDensityS as the scatter writes it (:187-212) and the next gather
      // reads it back: floored at 1 on 1..nAlts, or exp(LogINS)
#pragma unroll
      for (int q = 0; q < IPW; q++) {
        double &u = c.own(GR_LEN + NG * q);
        if (kp.improved_ions) {
          if (c.cell() && u < 1) u = 1.0;
        } else if (step + 1 < kp.n_steps) {
          u = ln(exp(u));
        }
      }
    }
  }
#undef GV_LD
  const long long bn = col_base(io.ndensity_s, ci, cj, cb);
  const long long bw = col_base(io.vertical_velocity, ci, cj, cb);
  const long long bv = col_base(io.velocity, ci, cj, cb);
#pragma unroll
  for (int q = 0; q < SPW; q++) {
    const int s = s0 + q;
    *fld(io.ndensity_s, bn, k, s) = nds[q];
    *fld(io.vertical_velocity, bw, k, s) = c.spc(GU_W, q);
    if (io.log_ns.ptr) *fld(io.log_ns, col_base(io.log_ns, ci, cj, cb), k, s) = c.spc(GU_LN, q);
  }
  if (g == 0) {
    *fld(io.temperature, col_base(io.temperature, ci, cj, cb), k, 0) = r0;
    *fld(io.velocity, bv, k, 2) = r1;
  } else {
    *fld(io.velocity, bv, k, g - 1) = r0;
    if (g == 1) *fld(io.rho, col_base(io.rho, ci, cj, cb), k, 0) = r1;
  }
  if (io.ndensity.ptr || IONS) {
    // sums over the species and the ions (:187-212), from the lanes' values
#pragma unroll
    for (int q = 0; q < SPW; q++) c.x(GR_POOL + s0 + q, j) = nds[q];
    double v[IPW];
    if (IONS) {
#pragma unroll
      for (int q = 0; q < IPW; q++) {
        const int f = g + NG * q;
        v[q] = kp.improved_ions ? c.ion(f, j) : exp(c.ion(f, j));
        *fld(io.idensity_s, col_base(io.idensity_s, ci, cj, cb), k, f) = v[q];
        c.x(GR_POOL + NSP + f, j) = v[q];
      }
    }
    cx.sync();
    if (g == 1 && io.ndensity.ptr) {
      double n = 0.0;
#pragma unroll
      for (int s = 0; s < NSP; s++) n = n + c.x(GR_POOL + s, j);
      *fld(io.ndensity, col_base(io.ndensity, ci, cj, cb), k, 0) = n;
    }
    if (IONS && g == 2) {
      double e = 0.0;
#pragma unroll
      for (int f = 0; f < NI; f++) e = e + c.x(GR_POOL + NSP + f, j);
      *fld(io.idensity_s, col_base(io.idensity_s, ci, cj, cb), k, NI) = e;
    }
  }
}

}  // namespace gv
