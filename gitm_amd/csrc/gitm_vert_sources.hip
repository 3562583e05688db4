// gitm_vert_sources.hip -- the operator-split sources step's neutral terms
// (gitm_vert_sources of include/gitm_vert.h): thermal conduction
// (calc_conduction.f90:19-125) and viscosity (calc_viscosity.f90:4-189),
// each three implicit solves of calc_conduction_1d
// (calc_conduction.f90:132-244) and the second-order combination
// (2H - F) - Q, then the updates of add_sources.f90:53-70,94-107.
//
// Mapping: one workgroup per column, one lane per level, as the vertical
// step's.  The tridiagonal (Thomas) solves are serial in altitude and the
// results are the oracle's bit for bit, so neither a parallel solver nor a
// multiplication by a rounded reciprocal will do; what is left is to make
// the serial part short and to keep enough columns on a CU to hide it:
//  * the quotients are the hardware's own division sequence without its
//    scaling and special cases (vert_sources_chain.h), whose reciprocal a
//    pivot's two quotients share; range tests beside the chains tell whether
//    that was exact, and a column where it may not have been is done again with
//    plain divisions.  Zeros pass: after a vertical step the east and north
//    winds of level 0 are zero in every column;
//  * a chain reads ahead, two levels per LDS access (rows of the LDS image
//    run along altitude), and holds little but its arithmetic: per level the
//    first sweeps take 150 clocks, of which 88 are the serial operations, the
//    back substitutions 42;
//  * the second Dt/2 solve finds the pivots and their reciprocals formed by
//    the level lanes, so a level of its sweep is five dependent operations,
//    70 clocks;
//  * the LDS image is 45 doubles per level (five rows per quantity, each
//    reused as soon as it is read), four columns of 100 levels per CU.
// What bounds it is the serial chains of the few columns that the LDS holds:
// 34 of a column's 65 thousand clocks (LDS writes of 26 clocks each on top of
// the arithmetic), with 1.6 TB/s of HBM in use.  64,800 columns of 100 levels
// took 3.25 ms with a division in each link of the chains, 63 doubles per
// level and no read ahead; they take 1.74 ms, before and after a vertical step.
// Were all of them done again it would be 3.7 ms: the quick pass up to the test
// that fails, then a plain one without read ahead.
#include "vert_gpu.h"
#include "vert_sources_chain.h"

namespace {

using namespace gv::chain;

struct SrcParams {
  double dt;
  double mass[gv::NSP];
  int use_turbulent_cond, apply;
  int n_alts, n_cols;
};

struct SrcFields {
  gitm_vert_field kappa_temp, visc_coef, visc_coef_s, cp, raddist, heating, chem_heating,
      user_heating, conduction, viscosity, vvisc;
};

struct SrcArgs {
  SrcParams p;
  gitm_vert_columns io;
  SrcFields f;
};

constexpr int NQ = 3 + gv::NSP;  // temperature, two winds, six species winds

// Rows of the LDS image, one per quantity q (RS doubles each, level k at
// k + 1):
//   W_A   the tridiagonal a, shared by the three solves (it does not depend
//         on the step, but at the top level);
//   W_C   c, read by both solves, then the Dt solve's dp and its solution;
//         at the top level, where c is 0, the Dt solve's a; then the second
//         Dt/2 solve's right side, its dp and its solution;
//   W_BA  b of the Dt/2 solves, then their cp;
//   W_BC  b of the Dt solve, then its cp; then the reciprocals of the Dt/2
//         solves' pivots;
//   W_D   d of the Dt solve (the Dt/2 solve's is twice that in the
//         interior), then the first Dt/2 solve's dp and its solution; then
//         the Dt/2 solves' pivots.
// The two solves' lanes share a wavefront, so both have read c and d of a
// level before either writes over them.  Until the coefficients are formed
// the first rows hold the diffusion coefficients times r^2 (one for the two
// winds, whose coefficients are equal) and the altitude.
enum {
  W_A = 0, W_C = W_A + NQ, W_BA = W_C + NQ, W_BC = W_BA + NQ, W_D = W_BC + NQ, W_LEN = W_D + NQ,
  W_DI = 0, W_ALT = NQ - 1
};
constexpr int ND = NQ - 1;  // distinct diffusion coefficients
constexpr int di_slot(int q) { return q == 0 ? 0 : (q < 3 ? 1 : q - 1); }
static_assert(di_slot(NQ - 1) == ND - 1 && W_ALT >= ND, "diffusion rows below the altitude's");
static_assert(2 * NQ <= 64, "both solves' lanes in one wavefront");

// Doubles of a row: even, so that level 1 and every second one after it are
// 16-byte aligned, and odd in pairs, so that the chain lanes' rows fall on
// different LDS banks.
constexpr int row_len(int n_alts) { return (n_alts + 4) + ((2 - (n_alts + 4)) & 3); }

struct SrcCol {
  const SrcArgs *args;
  double *lds;
  int ci, cj, cb;
  int rs;

  // A later phase's view of the arguments: field descriptors and the column's
  // offsets in them are otherwise read and formed at the kernel's start, and
  // what the scalar registers do not hold of them is spilled.
  __device__ __forceinline__ void locate() {
    asm volatile("" : "+s"(args), "+s"(ci), "+s"(cj), "+s"(cb));
  }

  __device__ double *row(int w) const { return lds + w * rs + 1; }  // level 0
  __device__ double &rec(int k, int w) const { return row(w)[k]; }
  __device__ double at(const gitm_vert_field &g, int k, int comp = 0) const {
    return *gv::fld(g, gv::col_base(g, ci, cj, cb), k, comp);
  }
  __device__ double *ptr(const gitm_vert_field &g, int k, int comp = 0) const {
    return gv::fld(g, gv::col_base(g, ci, cj, cb), k, comp);
  }
  __device__ double quantity(int q, int k) const {
    const gitm_vert_columns &io = args->io;
    if (q == 0) return at(io.temperature, k);
    if (q < 3) return at(io.velocity, k, q - 1);
    return at(io.vertical_velocity, k, q - 3);
  }
};

// One quantity's coefficients at one level (calc_conduction.f90:181-230).
struct Coef {
  double a, c, ba, bc, d, ma;
};
// The grid factors that a level's quantities share.
struct Grid {
  double r, du12, du22, r12, r22;
};
template <bool FAST>
__device__ __forceinline__ Coef coefficients(Range &range, int k, int nA, double dtA, double dtC,
                                             const Grid &g, double told, double mr, double di0,
                                             double dl) {
  const auto div = [](double n, double d, double r) { return FAST ? div_pos(n, d, r) : n / d; };
  const double r = g.r;
  // Dt is twice Dt/2 without rounding, so the fast form has the Dt solve's
  // quotients from the Dt/2 solve's
  const double mA = div(dtA, mr, FAST ? div_recip(mr) : 0.0);
  const double mC = FAST ? 2.0 * mA : dtC / mr;
  const double rm = FAST ? div_recip(mA) : 0.0;
  const bool top = k > nA;
  const double h = r * (1.0 + r) * di0;
  const double xn = top ? h * mA : di0;
  const double x = div(xn, g.du22, g.r22), y = div(dl, g.du12, g.r12);
  const double i = div(1.0, mA, rm);
  Coef o;
  o.ma = mA;
  o.a = x * r - y * r * r;
  o.c = x + y;
  o.ba = -i - x * (1 + r) - y * (1 - r * r);
  o.bc = (FAST ? -0.5 * i : -1 / mC) - x * (1 + r) - y * (1 - r * r);
  o.d = FAST ? -0.5 * div(told, mA, rm) : -told / mC;
  if (FAST) {
    range.divisor(mr);
    range.divisor(mA);
    range.numerator(xn);
    range.numerator(dl);
    range.numerator(told);
    range.numerator(o.c);
    range.numerator(o.a);
    range.element(o.ba);
    range.element(o.bc);
  }
  if (k < 1) {  // a = 0, b = -1, c = 0, d = -told (:210-213)
    o.a = o.c = 0.0;
    o.ba = o.bc = -1.0;
  }
  if (top) {  // Neumann, :221-230
    o.a = x;
    o.c = FAST ? 2.0 * x : h * mC / g.du22;
    o.ba = -1.0 * (1.0 + o.a);
    o.bc = -1.0 * (1.0 + o.c);
  }
  if (k < 1 || top) o.d = -told;
  return o;
}

// A level's values that outlive the solves.
struct Level {
  double qin[NQ], s1[NQ], fv[NQ], h[NQ];  // in, first Dt/2 step, Dt step, second Dt/2 step
  double unit, vup, vu, heat[3];
};

// Phases of one column (barriers between them):
//  1. stage: one lane per level -1..nAlts+2 loads its level; the diffusion
//     coefficients and the altitude go to LDS, the rest stays in registers;
//  2. one lane per level 0..nAlts+1 reads its neighbours', forms the grid
//     factors and, after a barrier, every solve's a, b, c and d;
//  3. the forward sweeps and back substitutions of the first Dt/2 solve and
//     the Dt solve, one lane per (solve, quantity) of the first wavefront,
//     serial in altitude (:232-247);
//  4. one lane per level: the first stage's value, the full step's, and the
//     second Dt/2 solve's right side, pivots and reciprocals;
//  5. the second Dt/2 solve, one lane per quantity, and its values.
// With FAST the phases end early, for the whole workgroup, once a range test
// fails; returns whether none did.  Each phase has its own word of failed[]:
// it is written before a barrier and only read after it.
template <bool FAST>
__device__ __forceinline__ bool solves(const SrcCol &c, volatile int *failed, int j,
                                       Level &v) {
  const SrcParams &p = c.args->p;
  const gitm_vert_columns &io = c.args->io;
  const SrcFields &f = c.args->f;
  const int k = j - 1, nA = p.n_alts;
  const bool lev = k >= 0 && k <= nA + 1;
  const double dtA = p.dt / 2.0, dtC = p.dt;
  double mr[NQ];
  // 1. stage
  if (FAST && j < 5) failed[j] = 0;
  if (k <= nA + 2) c.rec(k, W_ALT) = c.at(io.altitude, k);
  if (lev) {
    v.unit = c.at(io.temp_unit, k);
    const double rd = c.at(f.raddist, k), rho = c.at(io.rho, k), eddy = c.at(io.eddy, k),
                 cpk = c.at(f.cp, k), kappa = c.at(f.kappa_temp, k), visc = c.at(f.visc_coef, k);
    double n[gv::NSP], vs[gv::NSP];
#pragma unroll
    for (int s = 0; s < gv::NSP; s++) {
      n[s] = c.at(io.ndensity_s, k, s);
      vs[s] = c.at(f.visc_coef_s, k, s);
    }
#pragma unroll
    for (int q = 0; q < NQ; q++) v.qin[q] = c.quantity(q, k);
    // what the updates add to, read while nothing waits for it
    if (p.apply) {
      v.vu = c.at(io.velocity, k, 2);
      if (k >= 1 && k <= nA) {
        if (f.heating.ptr) v.heat[0] = c.at(f.heating, k);
        if (f.chem_heating.ptr) v.heat[1] = c.at(f.chem_heating, k);
        if (f.user_heating.ptr) v.heat[2] = c.at(f.user_heating, k);
      }
    }
    GV_ORDER();  // every load is under way before the first is waited for
    const double r2 = rd * rd;
    // calc_conduction.f90:59-73
    const double prandtl = p.use_turbulent_cond ? eddy * rho * cpk : 0.0;
    c.rec(k, W_DI + di_slot(0)) = (kappa + prandtl) * r2;
    mr[0] = (rho * cpk) * r2;
    // calc_viscosity.f90:66-67
    c.rec(k, W_DI + di_slot(1)) = (visc + rho * eddy) * r2;
    mr[1] = rho * r2;
    mr[2] = rho * r2;
#pragma unroll
    for (int s = 0; s < gv::NSP; s++) {  // :125-128
      const double mn = p.mass[s] * n[s];
      c.rec(k, W_DI + di_slot(3 + s)) = ((4.0 / 3.0) * vs[s] + mn * eddy) * r2;
      mr[3 + s] = mn * r2;
    }
  }
  __syncthreads();
  // 2. coefficients
  Grid g;
  double di[ND], dl[ND], ba[NQ], ma[NQ];
  Range range;
  if (lev) {
    const double altm = c.rec(k - 1, W_ALT), alt0 = c.rec(k, W_ALT),
                 altp = c.rec(k + 1, W_ALT);
    const double du = altp - alt0, dl0 = alt0 - altm;  // :181-186
    const double r = du / dl0;
    g.r = r;
    g.du12 = du * du * (1 + r) * (1 + r);
    g.du22 = 0.5 * (dl0 * du + du * du);
    if (FAST) {
      g.r12 = div_recip(g.du12);
      g.r22 = div_recip(g.du22);
      range.divisor(g.du12);
      range.divisor(g.du22);
    }
#pragma unroll
    for (int s = 0; s < ND; s++) di[s] = dl[s] = c.rec(k, W_DI + s);
    if (k >= 1 && k <= nA)
#pragma unroll
      for (int s = 0; s < ND; s++)
        dl[s] = c.rec(k + 1, W_DI + s) - r * r * c.rec(k - 1, W_DI + s) -
                (1 - r * r) * di[s];  // :188-190
  }
  __syncthreads();
  if (lev) {
#pragma unroll
    for (int q = 0; q < NQ; q++) {
      const double told = q == 0 ? v.qin[0] * v.unit : v.qin[q];
      const Coef o = coefficients<FAST>(range, k, nA, dtA, dtC, g, told, mr[q], di[di_slot(q)],
                                        dl[di_slot(q)]);
      c.rec(k, W_A + q) = o.a;
      c.rec(k, W_C + q) = o.c;
      c.rec(k, W_BA + q) = ba[q] = o.ba;
      c.rec(k, W_BC + q) = o.bc;
      c.rec(k, W_D + q) = o.d;
      ma[q] = o.ma;
    }
    if (FAST && !range.good()) failed[0] = 1;
  }
  __syncthreads();
  if (FAST && __builtin_amdgcn_readfirstlane(failed[0])) return false;
  // 3. the first Dt/2 solve (A) and the Dt solve (C), at once
  if (j < 2 * NQ) {
    const bool isA = j < NQ;
    const int q = isA ? j : j - NQ, top = nA + 1;
    const double *ra = c.row(W_A + q), *rc = c.row(W_C + q), *rd = c.row(W_D + q);
    double *rb = c.row((isA ? W_BA : W_BC) + q), *wd = c.row((isA ? W_D : W_C) + q);
    const double a = (isA ? ra : rc)[top], b = rb[top], d = rd[top];
    double cp = 0.0 / -1.0;
    double dp = rd[0] / -1.0;
    rb[0] = cp;
    wd[0] = dp;
    if (!sweep<FAST>(ra, rc, rb, rd, wd, isA ? 2.0 : 1.0, nA, cp, dp)) failed[1] = 1;
    const double t = (d - dp * a) / (b - cp * a);  // temp(nAlts+1) = dp(nAlts+1)
    wd[top] = t;
    back<FAST>(rb, wd, nA, t);
  }
  __syncthreads();
  if (FAST && __builtin_amdgcn_readfirstlane(failed[1])) return false;
  // 4. the first stage's value s1 and the full step's fv (dTdt_cond,
  // :249-250), and the second Dt/2 solve's operands
  if (lev) {
    double finite = 0.0;
    Range told_range;
#pragma unroll
    for (int q = 0; q < NQ; q++) {
      const double in = q == 0 ? v.qin[0] * v.unit : v.qin[q];
      const double ra = c.rec(k, W_D + q) - in, rc = c.rec(k, W_C + q) - in;
      v.s1[q] = q == 0 ? v.qin[0] + ra / v.unit : v.qin[q] + ra;
      v.fv[q] = q == 0 ? v.qin[0] + rc / v.unit : v.qin[q] + rc;
      // Viscosity(:,:,:,iUp_) keeps the last species' full-step result
      // (calc_viscosity.f90:161)
      if (q == NQ - 1) v.vup = rc;
      const double told = q == 0 ? v.s1[0] * v.unit : v.s1[q];
      double rhs;
      if (FAST) {
        finite = __builtin_fma(ra, 0.0, __builtin_fma(rc, 0.0, finite));
        told_range.numerator(told);
        rhs = -div_pos(told, ma[q], div_recip(ma[q]));
      } else {
        rhs = -told / ma[q];
      }
      c.rec(k, W_C + q) = k >= 1 && k <= nA ? rhs : -told;
      if (k >= 1) {
        const double den = ba[q] - c.rec(k - 1, W_BA + q) * c.rec(k, W_A + q);
        c.rec(k, W_D + q) = den;
        if (FAST) c.rec(k, W_BC + q) = div_recip(den);
      }
    }
    if (FAST && !(told_range.good() && finite == 0.0)) failed[2] = 1;
  }
  __syncthreads();
  if (FAST && __builtin_amdgcn_readfirstlane(failed[2])) return false;
  // 5. the second Dt/2 solve (B)
  if (j < NQ) {
    const double *ra = c.row(W_A + j), *rden = c.row(W_D + j), *rr = c.row(W_BC + j);
    double *rn = c.row(W_C + j);
    const int top = nA + 1;
    const double a = ra[top], b = rden[top], d = rn[top];
    double dp = rn[0] / -1.0;
    rn[0] = dp;
    if (!sweep2<FAST>(ra, rn, rden, rr, nA, dp)) failed[3] = 1;
    const double t = (d - dp * a) / b;
    rn[top] = t;
    back<FAST>(c.row(W_BA + j), rn, nA, t);
  }
  __syncthreads();
  if (FAST && __builtin_amdgcn_readfirstlane(failed[3])) return false;
  if (lev) {
    double finite = 0.0;
#pragma unroll
    for (int q = 0; q < NQ; q++) {
      v.h[q] = c.rec(k, W_C + q);
      finite = __builtin_fma(v.h[q], 0.0, finite);
    }
    if (FAST && !(finite == 0.0)) failed[4] = 1;
  }
  if (!FAST) return true;
  __syncthreads();
  return __builtin_amdgcn_readfirstlane(failed[4]) == 0;
}

// Two wavefronts per SIMD are what the LDS image leaves room for: 256 VGPRs.
template <int NT>
__global__ void __launch_bounds__(NT, 2)
    sources_kernel(SrcArgs) {
  extern __shared__ __align__(16) double lds[];
  const auto *args = (const SrcArgs *)(const __attribute__((address_space(4))) SrcArgs *)
      __builtin_amdgcn_kernarg_segment_ptr();
  const int col = xcd_column((int)blockIdx.x, (int)gridDim.x), j = (int)threadIdx.x, k = j - 1;
  const int nA = args->p.n_alts, nlon = args->io.n_lons, nlat = args->io.n_lats;
  SrcCol c{args, lds, col % nlon, (col / nlon) % nlat, col / (nlon * nlat), row_len(nA)};
  volatile int *failed = reinterpret_cast<volatile int *>(lds + W_LEN * c.rs + PAD);
  Level v;
  v.unit = 1.0;
  v.vu = v.heat[0] = v.heat[1] = v.heat[2] = 0.0;
  if (!solves<true>(c, failed, j, v)) {
    __syncthreads();  // every lane is through with LDS
    c.locate();
    solves<false>(c, failed, j, v);
  }
  c.locate();
  const SrcParams &p = c.args->p;
  const gitm_vert_columns &io = c.args->io;
  const SrcFields &f = c.args->f;
  if (k < 0 || k > nA + 1) return;
  // 6. the combination (2H - F) - Q (:117-121, calc_viscosity.f90:110-114),
  // the increments and add_sources' updates (:53-70, :94-114), one level per
  // lane
  double out[NQ];
#pragma unroll
  for (int q = 0; q < NQ; q++) {
    const double in = q == 0 ? v.s1[0] * v.unit : v.s1[q];
    const double rb = v.h[q] - in;
    const double h = q == 0 ? v.s1[0] + rb / v.unit : v.s1[q] + rb;
    out[q] = (2.0 * h - v.fv[q]) - v.qin[q];
  }
  const double cond = out[0];
  if (f.conduction.ptr) *c.ptr(f.conduction, k) = cond;
  if (f.viscosity.ptr) {
    *c.ptr(f.viscosity, k, 0) = out[1];
    *c.ptr(f.viscosity, k, 1) = out[2];
    *c.ptr(f.viscosity, k, 2) = v.vup;
  }
  if (f.vvisc.ptr)
#pragma unroll
    for (int s = 0; s < gv::NSP; s++) *c.ptr(f.vvisc, k, s) = out[3 + s];
  if (!p.apply) return;
  double tt = v.qin[0];
  if (k >= 1 && k <= nA) {
    tt = tt + p.dt * v.heat[0];
    if (f.chem_heating.ptr) tt = tt + v.heat[1];
    if (f.user_heating.ptr) tt = tt + v.heat[2];
  }
  *c.ptr(io.temperature, k) = tt + cond;
  *c.ptr(io.velocity, k, 0) = v.qin[1] + out[1];
  *c.ptr(io.velocity, k, 1) = v.qin[2] + out[2];
  *c.ptr(io.velocity, k, 2) = v.vu + v.vup;
#pragma unroll
  for (int s = 0; s < gv::NSP; s++) *c.ptr(io.vertical_velocity, k, s) = v.qin[3 + s] + out[3 + s];
}

}  // namespace

extern "C" int gitm_vert_sources(gitm_vert_handle *h, const gitm_vert_sources_params *sp,
                                 const gitm_vert_columns *c,
                                 const gitm_vert_sources_fields *sf) {
  if (!h || !sp || !c || !sf) return GITM_VERT_EINVAL;
  if (c->n_alts < 10 || c->n_alts > GITM_VERT_MAX_NALTS) return GITM_VERT_EINVAL;
  if (c->n_lons < 1 || c->n_lats < 1 || c->n_blocks < 1) return GITM_VERT_EINVAL;
  const long long ncols = (long long)c->n_lons * c->n_lats * c->n_blocks;
  if (ncols > 0x7fffffffLL) return GITM_VERT_EINVAL;
  const gitm_vert_field *req[] = {&c->temperature, &c->temp_unit, &c->rho, &c->eddy,
                                  &c->ndensity_s, &c->velocity, &c->vertical_velocity,
                                  &c->altitude, &sf->kappa_temp, &sf->visc_coef,
                                  &sf->visc_coef_s, &sf->cp, &sf->radial_distance};
  for (const gitm_vert_field *g : req)
    if (!g->ptr) return GITM_VERT_EINVAL;
  if (!(sp->dt > 0.0)) return GITM_VERT_EINVAL;
  for (int s = 0; s < gv::NSP; s++)
    if (!(sp->mass[s] > 0.0)) return GITM_VERT_EINVAL;
  GV_HIP(hipSetDevice(h->device));
  SrcArgs args;
  SrcParams &p = args.p;
  args.io = *c;
  p.dt = sp->dt;
  for (int s = 0; s < gv::NSP; s++) p.mass[s] = sp->mass[s];
  p.use_turbulent_cond = sp->use_turbulent_cond != 0;
  p.apply = sp->apply != 0;
  p.n_alts = c->n_alts;
  p.n_cols = (int)ncols;
  SrcFields &f = args.f;
  f.kappa_temp = sf->kappa_temp;
  f.visc_coef = sf->visc_coef;
  f.visc_coef_s = sf->visc_coef_s;
  f.cp = sf->cp;
  f.raddist = sf->radial_distance;
  f.heating = sf->heating;
  f.chem_heating = sf->chem_heating;
  f.user_heating = sf->user_heating;
  f.conduction = sf->conduction;
  f.viscosity = sf->viscosity;
  f.vvisc = sf->vertical_viscosity;
  const size_t lds = ((size_t)W_LEN * row_len(c->n_alts) + PAD + 3) * sizeof(double);  // 91 KB at 252
  const int waves = gv::auto_waves(c->n_alts);
  const dim3 grid((unsigned)ncols), block(64 * waves);
  switch (waves) {
    case 1: hipLaunchKernelGGL(sources_kernel<64>, grid, block, lds, h->stream, args); break;
    case 2: hipLaunchKernelGGL(sources_kernel<128>, grid, block, lds, h->stream, args); break;
    case 3: hipLaunchKernelGGL(sources_kernel<192>, grid, block, lds, h->stream, args); break;
    case 4: hipLaunchKernelGGL(sources_kernel<256>, grid, block, lds, h->stream, args); break;
    default: return GITM_VERT_EINVAL;
  }
  GV_HIP(hipGetLastError());
  return GITM_VERT_OK;
}

// Host arrays (GITM's own): every field staged on the device over the levels
// the step touches (the altitude on -1..nAlts+2, the heating terms on
// 1..nAlts, the rest on 0..nAlts+1), the written ones copied back.
extern "C" int gitm_vert_sources_host(gitm_vert_handle *h, const gitm_vert_sources_params *sp,
                                      const gitm_vert_columns *c,
                                      const gitm_vert_sources_fields *sf) {
  if (!h || !sp || !c || !sf) return GITM_VERT_EINVAL;
  const int n = c->n_lons, m = c->n_lats, nA = c->n_alts, nb = c->n_blocks;
  if (n < 1 || m < 1 || nA < 1 || nb < 1) return GITM_VERT_EINVAL;
  gitm_vert_columns d = *c;
  gitm_vert_sources_fields g = *sf;
  const bool apply = sp->apply != 0;
  std::vector<HostSpan> spans;
  auto add = [&](gitm_vert_field *f, int nc, int lo, int hi, bool written) {
    spans.push_back({f, 1, n, 1, m, lo, hi, nc, written});
  };
  add(&d.altitude, 1, -1, nA + 2, false);
  add(&d.temperature, 1, 0, nA + 1, apply);
  add(&d.velocity, 3, 0, nA + 1, apply);
  add(&d.vertical_velocity, gv::NSP, 0, nA + 1, apply);
  add(&d.temp_unit, 1, 0, nA + 1, false);
  add(&d.rho, 1, 0, nA + 1, false);
  add(&d.eddy, 1, 0, nA + 1, false);
  add(&d.ndensity_s, gv::NSP, 0, nA + 1, false);
  add(&g.kappa_temp, 1, 0, nA + 1, false);
  add(&g.visc_coef, 1, 0, nA + 1, false);
  add(&g.visc_coef_s, gv::NSP, 0, nA + 1, false);
  add(&g.cp, 1, 0, nA + 1, false);
  add(&g.radial_distance, 1, 0, nA + 1, false);
  add(&g.heating, 1, 1, nA, false);
  add(&g.chem_heating, 1, 1, nA, false);
  add(&g.user_heating, 1, 1, nA, false);
  add(&g.conduction, 1, 0, nA + 1, true);
  add(&g.viscosity, 3, 0, nA + 1, true);
  add(&g.vertical_viscosity, gv::NSP, 0, nA + 1, true);
  GV_HIP(hipSetDevice(h->device));
  HostStaging st;
  int rc = stage_in(h, spans, nb, 96, st);  // slots after the other host entries'
  if (rc) return rc;
  rc = gitm_vert_sources(h, sp, &d, &g);
  if (rc) return rc;
  rc = stage_out(h, spans, 96, st);
  if (rc) return rc;
  GV_HIP(hipStreamSynchronize(h->stream));
  return GITM_VERT_OK;
}
