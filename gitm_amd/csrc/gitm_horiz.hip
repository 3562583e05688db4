// gitm_horiz.hip -- the horizontal step (gitm_horiz_advance of
// include/gitm_vert.h): advance_horizontal(iBlock)
// (advance_horizontal.f90:58-924) for every block, each altitude 1..nAlts
// an independent 2-D problem on the block's cells with the halo cells
// (-1:0, n+1:n+2) held at their input values (the caller's message
// exchange fills them, :20).
//
// Mapping: a lane takes one cell of one altitude.  The workgroup stages the
// slices of the advected variables (halo cells included) in LDS; each stage of
// the RK4 (:154-345) then runs horizontal_solver (:535-818) lane by lane: the
// lane forms the MC-limited face values of its own two faces in each direction
// (calc_facevalues_lons/lats, :928-1034) from the slopes at its cell and
// its two neighbours, the gradient and the Rusanov flux difference
// (calc_rusanov_lons/lats, :821-922), and the updates, holding the new
// values in registers until every lane has read the stage's state.  Density,
// temperature and winds advance together; the species, whose equations read
// the winds and nothing reads, are carried along.  Every
// value is formed by the reference's operations in the reference's order,
// so the results equal the reference's bit for bit (sin(latitude) aside,
// which is the device's).  With UseImprovedIonAdvection a second kernel
// applies the divergence of the ion velocity afterwards.
#include <type_traits>

#include "vert_gpu.h"

namespace {

constexpr int NIA = 2;  // nIonsAdvect (ModEarth.f90:39)
constexpr int V_RHO = 0, V_TEMP = 1, V_VEL = 2, V_NUM = 5, V_VV = 11, V_INUM = 17;
constexpr int NV_NEUTRAL = V_INUM, NV_IONS = V_INUM + NIA;

struct HzParams {
  double dt, omega, beta;
  int use_coriolis;
  int n_lons, n_lats, n_alts, n_blocks;
  int apw;         // altitudes per workgroup
  int alt_groups;  // workgroups per block
};

struct HzFields {
  gitm_vert_field inv_dlon_gb, inv_dlon_fb, dlon_fb, inv_dlat_gb, inv_dlat_fb, dlat_fb,
      raddist, latitude, tan_latitude, cmax, temp_source;
  gitm_vert_field dalt, dalt_dlon, dalt_dlat;  // UseTopography
};

// Element (iLon, iLat, level, comp) of block b: the descriptor's ptr is at
// (1, 1, first_level) of block 0.
__device__ __forceinline__ double *hf(const gitm_vert_field &f, int lon, int lat, int lev,
                                      int comp, int b) {
  return f.ptr + (long long)(lon - 1) * f.s_lon + (long long)(lat - 1) * f.s_lat +
         (long long)(lev - f.first_level) * f.s_lev + (long long)comp * f.s_comp +
         (long long)b * f.s_blk;
}

// The geometry of one cell i (1..n) along one line: InvD*Dist_FB at faces
// i-1..i+2, d*Dist_FB at faces i and i+1, InvD*Dist_GB(i), half the larger
// cMax of the cells on either side of faces i and i+1, and whether the cell
// is the line's first or last.
struct LineGeo {
  double ifb[4], dfb0, dfb1, igb, hc0, hc1;
  bool first, last;
};

// One cell of one line: v[m * S] = Var(i + m), m = -3..3.  Gradient and flux
// difference (calc_facevalues_lons/lats, calc_rusanov_lons/lats).  The slope
// of a cell takes the fourth-order difference of its two faces; a face's is
// the same seen from either cell, so the three slopes need four.  The faces
// beyond the line's outermost slopes take the plain difference; there m = -3
// or 3 lies outside the line, is read from whatever the LDS holds and not
// used.
template <class P>
__device__ __forceinline__ void rusanov_cell(const P v, int S, const LineGeo &g, double beta,
                                             double &grad, double &diff) {
  const double F1 = 0.6250000, F2 = 0.0416667;
  const double vm3 = v[-3 * S], vm2 = v[-2 * S], vm1 = v[-S], v0 = v[0], v1 = v[S],
               v2 = v[2 * S], v3 = v[3 * S];
  const double dm = vm1 - vm2, dp = v2 - v1;
  double f0 = (g.ifb[0] * 2) * (F1 * dm - F2 * (v0 - vm3));
  const double f1 = (g.ifb[1] * 2) * (F1 * (v0 - vm1) - F2 * (v1 - vm2));
  const double f2 = (g.ifb[2] * 2) * (F1 * (v1 - v0) - F2 * (v2 - vm1));
  double f3 = (g.ifb[3] * 2) * (F1 * dp - F2 * (v3 - v0));
  f0 = g.first ? dm * g.ifb[0] : f0;
  f3 = g.last ? dp * g.ifb[3] : f3;
  const double s0 = gv::limiter_sel(beta, f1, f0), s1 = gv::limiter_sel(beta, f2, f1),
               s2 = gv::limiter_sel(beta, f3, f2);
  const double l0 = vm1 + 0.5 * s0 * g.dfb0, r0 = v0 - 0.5 * s1 * g.dfb0;
  const double l1 = v0 + 0.5 * s1 * g.dfb1, r1 = v1 - 0.5 * s2 * g.dfb1;
  grad = 0.5 * (l1 + r1 - l0 - r0) * g.igb;
  diff = (g.hc1 * (r1 - l1) - g.hc0 * (r0 - l0)) * g.igb;
}

// The advected fields (advance_horizontal.f90:154-167) by number.
__device__ __forceinline__ const gitm_vert_field &hz_field(const gitm_vert_columns &io, int v,
                                                           int &comp) {
  if (v == V_RHO) { comp = 0; return io.rho; }
  if (v == V_TEMP) { comp = 0; return io.temperature; }
  if (v < V_NUM) { comp = v - V_VEL; return io.velocity; }
  if (v < V_VV) { comp = v - V_NUM; return io.ndensity_s; }
  if (v < V_INUM) { comp = v - V_VV; return io.vertical_velocity; }
  comp = v - V_INUM;
  return io.idensity_s;
}

// One lane's cell of one altitude: its geometry, and what the core's four
// stages leave for the other variables.
struct HzCell {
  int i, jl, k, b;
  LineGeo lo, la;
  double hz, slon, slat;     // UseTopography: 0.5 / dAlt_GB, the surface's slopes
  double ve[4], vn[4], div[4];
};

__device__ __forceinline__ double at_stage(const double (&x)[4], int s) {
  return s == 0 ? x[0] : s == 1 ? x[1] : s == 2 ? x[2] : x[3];
}
__device__ __forceinline__ void set_stage(double (&x)[4], int s, double v) {
  x[0] = s == 0 ? v : x[0];
  x[1] = s == 1 ? v : x[1];
  x[2] = s == 2 ? v : x[2];
  x[3] = s == 3 ? v : x[3];
}

template <bool TOPO>
__device__ __forceinline__ void hz_geometry(HzCell &c, const gitm_vert_columns &io,
                                            const HzFields &f, int nlo, int nla) {
  const int i = c.i, jl = c.jl, k = c.k, b = c.b;
#pragma unroll
  for (int m = -1; m <= 2; m++) {
    c.lo.ifb[m + 1] = *hf(f.inv_dlon_fb, i + m, jl, k, 0, b);
    c.la.ifb[m + 1] = *hf(f.inv_dlat_fb, i, jl + m, k, 0, b);
  }
  c.lo.dfb0 = *hf(f.dlon_fb, i, jl, k, 0, b);
  c.lo.dfb1 = *hf(f.dlon_fb, i + 1, jl, k, 0, b);
  c.la.dfb0 = *hf(f.dlat_fb, i, jl, k, 0, b);
  c.la.dfb1 = *hf(f.dlat_fb, i, jl + 1, k, 0, b);
  c.lo.igb = *hf(f.inv_dlon_gb, i, jl, k, 0, b);
  c.la.igb = *hf(f.inv_dlat_gb, i, jl, k, 0, b);
  const double o0 = *hf(f.cmax, i, jl, k, 0, b), a0 = *hf(f.cmax, i, jl, k, 1, b);
  c.lo.hc0 = 0.5 * fmax(*hf(f.cmax, i - 1, jl, k, 0, b), o0);
  c.lo.hc1 = 0.5 * fmax(o0, *hf(f.cmax, i + 1, jl, k, 0, b));
  c.la.hc0 = 0.5 * fmax(*hf(f.cmax, i, jl - 1, k, 1, b), a0);
  c.la.hc1 = 0.5 * fmax(a0, *hf(f.cmax, i, jl + 1, k, 1, b));
  c.lo.first = i == 1;
  c.lo.last = i == nlo;
  c.la.first = jl == 1;
  c.la.last = jl == nla;
  if (TOPO) {
    // 0.5 / dAlt and the slopes of the level surface (advance_horizontal.f90
    // :581-582, :870-871, :919-920)
    c.hz = 0.5 / *hf(f.dalt, i, jl, k, 0, b);
    c.slon = *hf(f.dalt_dlon, i, jl, k, 0, b);
    c.slat = *hf(f.dalt_dlat, i, jl, k, 0, b);
  }
}

// The RK4 bookkeeping of one variable (:184-345): the stage's new value nw
// and state x give the next stage's state (the last stage's: the result).
__device__ __forceinline__ double hz_rk(int stage, double nw, double x, double orig,
                                        double &acc) {
  const double K = nw - x;
  if (stage == 3) return orig + (1.0 / 6.0) * (acc + K);
  acc = stage == 0 ? K : acc + 2.0 * K;
  return (stage == 2 ? K : 0.5 * K) + orig;
}

constexpr int NCORE = 5;  // Rho, Temperature and the winds advance together

// Grad and Diff of one variable in both directions (:588-662); dz: the
// variable's 0.5 (Var(k+1) - Var(k-1)) / dAlt (:583-586)
template <bool TOPO>
__device__ __forceinline__ void hz_gd(const HzCell &c, const double *x, int NLo, double beta,
                                      double dz, double &glon, double &glat, double &dsum) {
  double dlon, dlat;
  rusanov_cell(x, 1, c.lo, beta, glon, dlon);
  GV_ORDER();
  rusanov_cell(x, NLo, c.la, beta, glat, dlat);
  if (TOPO) {
    glon = glon - dz * c.slon;
    glat = glat - dz * c.slat;
  }
  dsum = dlon + dlat;
  GV_HERE(glon);
  GV_HERE(glat);
  GV_HERE(dsum);
  GV_ORDER();
}

// New values (:667-816) of the core variables from the stage's state, the
// gradients and the flux differences.
__device__ __forceinline__ void hz_core_update(const HzParams &p, const double (&g)[6],
                                               double rho, double tmp, double ve, double vn,
                                               double vu, double div, const double (&go)[NCORE],
                                               const double (&ga)[NCORE],
                                               const double (&d)[NCORE], double (&nw)[NCORE]) {
  constexpr int E = V_VEL, N = V_VEL + 1, U = V_VEL + 2;
  const double dt = p.dt;
  const double invr = g[0], rd = g[1], gam = g[2], tl = g[3], cosl = g[4], sinl = g[5];
  const double csin = sinl * 2 * p.omega, ccos = cosl * 2 * p.omega;
  const double cent = p.omega * p.omega * cosl * sinl;
  nw[V_RHO] = rho - dt * (rho * div + ga[V_RHO] * vn + go[V_RHO] * ve) + dt * d[V_RHO];
  double we = ve -
              dt * (vn * ga[E] + ve * go[E] + ve * (vu - tl * vn) * invr + go[V_TEMP] +
                    go[V_RHO] * tmp / rho) +
              dt * d[E];
  double wn = vn -
              dt * (vn * ga[N] + ve * go[N] + (vn * vu + tl * (ve * ve)) * invr + ga[V_TEMP] +
                    ga[V_RHO] * tmp / rho) +
              dt * d[N];
  if (p.use_coriolis) {
    we = we + dt * (+csin * vn - ccos * vu);
    wn = wn - dt * (cent * rd + csin * ve);
  }
  nw[E] = we;
  nw[N] = wn;
  nw[V_TEMP] =
      tmp - dt * ((gam - 1) * tmp * div + ga[V_TEMP] * vn + go[V_TEMP] * ve) + dt * d[V_TEMP];
  nw[U] = vu - dt * (vn * ga[U] + ve * go[U]) + dt * d[U];
}

// New value of one of the variables that the core carries along: 0 NDensityS,
// 1 VerticalVelocity, 2 IDensityS (with the ion velocity in ve, vn).
template <int KIND>
__device__ __forceinline__ double hz_carried_update(double q, double dt, double go, double ga,
                                                    double d, double ve, double vn, double div) {
  if (KIND == 0) return q - dt * (q * div + ga * vn + go * ve) + dt * d;
  if (KIND == 1) return q - dt * (vn * ga + ve * go) + dt * d;
  return q - dt * (+ga * vn + go * ve) + dt * d;
}

// Per-cell inputs of the core's updates.
__device__ __forceinline__ void hz_cell_inputs(const HzCell &c, const gitm_vert_columns &io,
                                               const HzFields &f, double (&g)[6]) {
  g[0] = *hf(io.inv_radial_distance, c.i, c.jl, c.k, 0, c.b);
  g[1] = *hf(f.raddist, c.i, c.jl, c.k, 0, c.b);
  g[2] = *hf(io.gamma, c.i, c.jl, c.k, 0, c.b);
  g[3] = *hf(f.tan_latitude, 1, c.jl, 0, 0, c.b);
  g[4] = *hf(io.cos_latitude, 1, c.jl, 0, 0, c.b);
  g[5] = sin(*hf(f.latitude, 1, c.jl, 0, 0, c.b));
}

// Write back (:349-429).
__device__ __forceinline__ void hz_store_core(const HzCell &c, const gitm_vert_columns &io,
                                              const HzFields &f, const double (&u)[NCORE],
                                              double told) {
  *hf(io.rho, c.i, c.jl, c.k, 0, c.b) = u[V_RHO];
#pragma unroll
  for (int q = 0; q < 3; q++) *hf(io.velocity, c.i, c.jl, c.k, q, c.b) = u[V_VEL + q];
  if (f.temp_source.ptr) *hf(f.temp_source, c.i, c.jl, c.k, 0, c.b) = u[V_TEMP] - told;
  *hf(io.temperature, c.i, c.jl, c.k, 0, c.b) = u[V_TEMP];
}
__device__ __forceinline__ void hz_report(const HzCell &c, int nlo, int nla,
                                          unsigned long long *err) {
  const int column = (c.b * nla + (c.jl - 1)) * nlo + (c.i - 1);
  atomicMin(err, gv::error_key(column, GITM_VERT_ENONPOSITIVE, c.k));
}
// The floored advected ion (:405-417) s of the cell.
__device__ __forceinline__ double hz_store_ion(const HzCell &c, const gitm_vert_columns &io,
                                               int s, double v) {
  if (v < 1.0e2) v = 1.0e2;
  *hf(io.idensity_s, c.i, c.jl, c.k, s, c.b) = v;
  return v;
}
__device__ __forceinline__ void hz_store_electrons(const HzCell &c,
                                                   const gitm_vert_columns &io) {
  double e = 0.0;  // :420-425
  for (int s = 0; s < gv::NIONS - 1; s++)
    e = e + *hf(io.idensity_s, c.i, c.jl, c.k, s, c.b);
  *hf(io.idensity_s, c.i, c.jl, c.k, gv::NIONS - 1, c.b) = e;
}

// LDS doubles before the first and after the last slice: the reads of m = -3
// and 3 past a line's end stay inside the block.
__host__ __device__ constexpr int hz_pad(int nlo) { return nlo + 4 + 4; }

// ---------------------------------------------------------------------------
// Level surfaces (no UseTopography): the altitudes are independent.  A
// workgroup takes apw altitudes of one block, a lane one cell of one of them.
// The core variables run their four stages first (:154-345); the others do
// not feed back on them, so they follow in groups that reuse the same LDS
// slices, with the core's winds and divergence of each stage kept in
// registers, as are the RK4's starting values and sums.
// Six slices per altitude instead of seventeen and their new values, so that
// the lanes can be packed (three 9x9 altitudes on 243 of 256 lanes) and three
// wavefronts share a SIMD.  FP64 issue bounds it: 800 blocks of 9x9 x 100
// levels, 8.8 -> 3.1 ms (all variables at once, one altitude on 81 of 128
// lanes, the RK4 sums and starting values in device memory, six face
// differences per cell and direction before).  Three wavefronts per SIMD (168
// registers, no spills) against four (128, 42 spilled): 3.1 against 3.5 ms.
// BLON, BLAT: the block's cells per direction when fixed at compile time
// (GITM's are, 9 x 9 by default), so that the LDS and cell indexing is
// constant; 0 takes them from the parameters.
// ---------------------------------------------------------------------------
constexpr int HZ_GROUP = 6;

template <bool IONS, int BLON, int BLAT>
__global__ void __launch_bounds__(256, 3)
    horiz_flat_kernel(HzParams p, gitm_vert_columns io, HzFields f, unsigned long long *err) {
  extern __shared__ double lds[];
  const int nlo = BLON ? BLON : p.n_lons, nla = BLAT ? BLAT : p.n_lats, NLo = nlo + 4,
            NLg = nla + 4;
  const int cells = nlo * nla, plane = NLg * NLo;
  const int k0 = 1 + ((int)blockIdx.x % p.alt_groups) * p.apw;
  const int napw = min(p.apw, p.n_alts - k0 + 1);
  const int tid = (int)threadIdx.x, a = tid / cells, cell = tid % cells;
  const bool active = a < napw;
  HzCell c;
  c.b = (int)blockIdx.x / p.alt_groups;
  c.i = cell % nlo + 1;
  c.jl = cell / nlo + 1;
  c.k = k0 + (active ? a : 0);
  double *const slices = lds + hz_pad(nlo);
  double *const x = slices + (active ? a : 0) * HZ_GROUP * plane + (c.jl + 1) * NLo + c.i + 1;
  // variables v0..v0+n-1, halo cells included: [altitude][variable][lat][lon];
  // each thread takes the cells r2 = tid, tid + 256, .. of a slice
  auto stage_in = [&](int v0, int n) {
    for (int r2 = tid; r2 < plane; r2 += (int)blockDim.x) {
      const int lat = r2 / NLo - 1, lon = r2 % NLo - 1;
      for (int aa = 0; aa < napw; aa++) {
        double *d = slices + aa * HZ_GROUP * plane + r2;
#pragma unroll
        for (int v = 0; v < HZ_GROUP; v++)
          if (v < n) {
            int comp;
            const gitm_vert_field &g = hz_field(io, v0 + v, comp);
            d[v * plane] = *hf(g, lon, lat, k0 + aa, comp, c.b);
          }
      }
    }
  };
  stage_in(V_RHO, NCORE);
  double g[6];
  if (active) {
    hz_geometry<false>(c, io, f, nlo, nla);
    hz_cell_inputs(c, io, f, g);
  }
  __syncthreads();
  {
    double orig[NCORE], acc[NCORE];
#pragma unroll
    for (int v = 0; v < NCORE; v++) orig[v] = x[v * plane];
    double u[NCORE];
#pragma unroll 1
    for (int stage = 0; stage < 4; stage++) {
      if (active) {
        double go[NCORE], ga[NCORE], d[NCORE];
#pragma unroll
        for (int v = 0; v < NCORE; v++)
          hz_gd<false>(c, x + v * plane, NLo, p.beta, 0.0, go[v], ga[v], d[v]);
        const double ve = x[V_VEL * plane], vn = x[(V_VEL + 1) * plane];
        const double div = ga[V_VEL + 1] + go[V_VEL] - g[3] * vn * g[0];
        set_stage(c.ve, stage, ve);
        set_stage(c.vn, stage, vn);
        set_stage(c.div, stage, div);
        hz_core_update(p, g, x[V_RHO * plane], x[V_TEMP * plane], ve, vn,
                       x[(V_VEL + 2) * plane], div, go, ga, d, u);
      }
      __syncthreads();  // every lane has read the stage's state
      if (active)
#pragma unroll
        for (int v = 0; v < NCORE; v++) {
          u[v] = hz_rk(stage, u[v], x[v * plane], orig[v], acc[v]);
          x[v * plane] = u[v];
        }
      __syncthreads();
    }
    if (active) hz_store_core(c, io, f, u, orig[V_TEMP]);
  }
  auto carried = [&](auto kind, int v0, auto count, auto &&store) {
    constexpr int KIND = decltype(kind)::value, N = decltype(count)::value;
    stage_in(v0, N);
    double ive = 0.0, ivn = 0.0;
    if (KIND == 2 && active) {
      ive = *hf(io.ivelocity, c.i, c.jl, c.k, 0, c.b);
      ivn = *hf(io.ivelocity, c.i, c.jl, c.k, 1, c.b);
    }
    __syncthreads();
    double orig[N], acc[N], u[N];
#pragma unroll
    for (int v = 0; v < N; v++) orig[v] = x[v * plane];
#pragma unroll 1
    for (int stage = 0; stage < 4; stage++) {
      if (active) {
        const double ve = KIND == 2 ? ive : at_stage(c.ve, stage),
                     vn = KIND == 2 ? ivn : at_stage(c.vn, stage), div = at_stage(c.div, stage);
#pragma unroll
        for (int v = 0; v < N; v++) {
          double go, ga, d;
          hz_gd<false>(c, x + v * plane, NLo, p.beta, 0.0, go, ga, d);
          u[v] = hz_carried_update<KIND>(x[v * plane], p.dt, go, ga, d, ve, vn, div);
          GV_HERE(u[v]);
          GV_ORDER();
        }
      }
      __syncthreads();
      if (active)
#pragma unroll
        for (int v = 0; v < N; v++) {
          u[v] = hz_rk(stage, u[v], x[v * plane], orig[v], acc[v]);
          x[v * plane] = u[v];
        }
      __syncthreads();
    }
    if (active) store(u);
  };
  carried(std::integral_constant<int, 0>(), V_NUM, std::integral_constant<int, gv::NSP>(),
          [&](const double (&u)[gv::NSP]) {
            bool negative = false;
#pragma unroll
            for (int s = 0; s < gv::NSP; s++) {
              negative = negative || u[s] < 0.0;
              *hf(io.ndensity_s, c.i, c.jl, c.k, s, c.b) = u[s];
            }
            if (negative) hz_report(c, nlo, nla, err);
          });
  carried(std::integral_constant<int, 1>(), V_VV, std::integral_constant<int, gv::NSP>(),
          [&](const double (&u)[gv::NSP]) {
#pragma unroll
            for (int s = 0; s < gv::NSP; s++)
              *hf(io.vertical_velocity, c.i, c.jl, c.k, s, c.b) = u[s];
          });
  if (IONS)
    carried(std::integral_constant<int, 2>(), V_INUM, std::integral_constant<int, NIA>(),
            [&](const double (&u)[NIA]) {
#pragma unroll
              for (int s = 0; s < NIA; s++) hz_store_ion(c, io, s, u[s]);
              hz_store_electrons(c, io);
            });
}

// ---------------------------------------------------------------------------
// UseTopography: dVarDAlt reads the level below as the step leaves it and the
// level above as it was (:583-586), so a block's levels follow one another.
// One workgroup walks a block's levels: no launch per level, and the chain of
// levels is shortened by giving the variables to teams of wavefronts that
// work side by side.  Team 0 takes the core variables, the others VP of the
// carried ones each (the ions' team the two ions); all have the cells of the
// level.  In each stage the teams form their gradients, the core's team puts
// its winds and divergence in LDS, and after a barrier every team updates.
// The chain of levels bounds it where blocks are few: 32 blocks of 9x9 x 50
// levels with ions 6.45 -> 1.5 ms (one launch per level before).
// A lane keeps its own cell's result for the level above.
// ---------------------------------------------------------------------------
enum { TEAM_CORE = 0, TEAM_DENSITY, TEAM_WIND, TEAM_ION };

template <int KIND, int N, int BLON, int BLAT>
__device__ __forceinline__ void topo_team(const HzParams &p, const gitm_vert_columns &io,
                                          const HzFields &f, unsigned long long *err,
                                          double *slices, double *pub, int cell,
                                          int team_threads, int s0) {
  const int nlo = BLON ? BLON : p.n_lons, nla = BLAT ? BLAT : p.n_lats, NLo = nlo + 4,
            NLg = nla + 4;
  const int cells = nlo * nla, plane = NLg * NLo;
  constexpr int V0 = KIND == TEAM_CORE ? V_RHO : KIND == TEAM_DENSITY ? V_NUM
                     : KIND == TEAM_WIND ? V_VV : V_INUM;
  const bool active = cell < cells;
  HzCell c;
  c.b = (int)blockIdx.x;
  c.i = active ? cell % nlo + 1 : 1;
  c.jl = active ? cell / nlo + 1 : 1;
  double *const mine = slices + (V0 + s0) * plane;
  double *const x = mine + (c.jl + 1) * NLo + c.i + 1;
  // a variable of the team at (lon, lat, k)
  const auto at = [&](int v, int lon, int lat, int k) -> double * {
    if (KIND == TEAM_CORE)
      return v == 0   ? hf(io.rho, lon, lat, k, 0, c.b)
             : v == 1 ? hf(io.temperature, lon, lat, k, 0, c.b)
                      : hf(io.velocity, lon, lat, k, v - 2, c.b);
    const gitm_vert_field &g = KIND == TEAM_DENSITY ? io.ndensity_s
                               : KIND == TEAM_WIND  ? io.vertical_velocity
                                                    : io.idensity_s;
    return hf(g, lon, lat, k, s0 + v, c.b);
  };
  double below[N];  // own cell at the level below, as the step leaves it
#pragma unroll
  for (int v = 0; v < N; v++) below[v] = *at(v, c.i, c.jl, 0);
#pragma unroll 1
  for (int k = 1; k <= p.n_alts; k++) {
    c.k = k;
    for (int r2 = cell; r2 < plane; r2 += team_threads) {
      const int lat = r2 / NLo - 1, lon = r2 % NLo - 1;
#pragma unroll
      for (int v = 0; v < N; v++) mine[v * plane + r2] = *at(v, lon, lat, k);
    }
    double g[6], ive = 0.0, ivn = 0.0;
    hz_geometry<true>(c, io, f, nlo, nla);
    if (KIND == TEAM_CORE) hz_cell_inputs(c, io, f, g);
    if (KIND == TEAM_ION) {
      ive = *hf(io.ivelocity, c.i, c.jl, k, 0, c.b);
      ivn = *hf(io.ivelocity, c.i, c.jl, k, 1, c.b);
    }
    double dz[N], orig[N], acc[N], u[N];
#pragma unroll
    for (int v = 0; v < N; v++) {
      dz[v] = c.hz * (*at(v, c.i, c.jl, k + 1) - below[v]);
      GV_HERE(dz[v]);
    }
    __syncthreads();
#pragma unroll
    for (int v = 0; v < N; v++) orig[v] = x[v * plane];
#pragma unroll 1
    for (int stage = 0; stage < 4; stage++) {
      double go[N], ga[N], d[N];
      if (active) {
#pragma unroll
        for (int v = 0; v < N; v++)
          hz_gd<true>(c, x + v * plane, NLo, p.beta, dz[v], go[v], ga[v], d[v]);
        if (KIND == TEAM_CORE) {
          const double vn = x[(V_VEL + 1) * plane];
          pub[cell] = x[V_VEL * plane];
          pub[cells + cell] = vn;
          pub[2 * cells + cell] = ga[V_VEL + 1] + go[V_VEL] - g[3] * vn * g[0];
        }
      }
      __syncthreads();
      if (active) {
        const double ve = KIND == TEAM_ION ? ive : pub[cell],
                     vn = KIND == TEAM_ION ? ivn : pub[cells + cell], div = pub[2 * cells + cell];
        if constexpr (KIND == TEAM_CORE) {
          hz_core_update(p, g, x[V_RHO * plane], x[V_TEMP * plane], ve, vn,
                         x[(V_VEL + 2) * plane], div, go, ga, d, u);
        } else {
#pragma unroll
          for (int v = 0; v < N; v++)
            u[v] = hz_carried_update<KIND - 1>(x[v * plane], p.dt, go[v], ga[v], d[v], ve, vn, div);
        }
#pragma unroll
        for (int v = 0; v < N; v++) {
          u[v] = hz_rk(stage, u[v], x[v * plane], orig[v], acc[v]);
          // the slices are a team's own, and its lanes have read the stage's
          // state before the barrier
          x[v * plane] = u[v];
        }
      }
      __syncthreads();
    }
    if (active) {
      if constexpr (KIND == TEAM_CORE) {
        hz_store_core(c, io, f, u, orig[V_TEMP]);
      } else if (KIND == TEAM_ION) {
#pragma unroll
        for (int v = 0; v < N; v++) u[v] = hz_store_ion(c, io, v, u[v]);
        hz_store_electrons(c, io);
      } else {
        bool negative = false;
#pragma unroll
        for (int v = 0; v < N; v++) {
          negative = negative || u[v] < 0.0;
          *at(v, c.i, c.jl, k) = u[v];
        }
        if (KIND == TEAM_DENSITY && negative) hz_report(c, nlo, nla, err);
      }
    }
#pragma unroll
    for (int v = 0; v < N; v++) below[v] = u[v];
  }
}

// (VP 3: blocks of up to 128 cells, six teams of two wavefronts; VP 6: up to
// 256 cells, four teams, as a workgroup holds 1,024 threads and six teams of
// three wavefronts are more.  32 blocks x 40 levels, one launch per level before:
// 9x9 cells 4.60 -> 1.16 ms, 12x9 6.25 -> 1.22, 12x12 6.40 -> 2.22, 16x16 6.46 -> 2.43.)
template <bool IONS, int VP, int BLON, int BLAT>
__global__ void __launch_bounds__(VP == 3 ? 768 : 1024)
    horiz_topo_kernel(HzParams p, gitm_vert_columns io, HzFields f, unsigned long long *err,
                      int team_threads) {
  extern __shared__ double lds[];
  const int nlo = BLON ? BLON : p.n_lons, nla = BLAT ? BLAT : p.n_lats;
  const int plane = (nla + 4) * (nlo + 4);
  const int team = __builtin_amdgcn_readfirstlane((int)threadIdx.x / team_threads);
  const int cell = (int)threadIdx.x - team * team_threads;
  double *const slices = lds + hz_pad(nlo);
  // ve, vn and div of each cell
  double *const pub = slices + (IONS ? NV_IONS : NV_NEUTRAL) * plane + hz_pad(nlo);
  constexpr int T = gv::NSP / VP;  // teams per species field
  if (team == 0)
    topo_team<TEAM_CORE, NCORE, BLON, BLAT>(p, io, f, err, slices, pub, cell, team_threads, 0);
  else if (team <= T)
    topo_team<TEAM_DENSITY, VP, BLON, BLAT>(p, io, f, err, slices, pub, cell, team_threads,
                                            (team - 1) * VP);
  else if (team <= 2 * T)
    topo_team<TEAM_WIND, VP, BLON, BLAT>(p, io, f, err, slices, pub, cell, team_threads,
                                         (team - 1 - T) * VP);
  else if (IONS)
    topo_team<TEAM_ION, NIA, BLON, BLAT>(p, io, f, err, slices, pub, cell, team_threads, 0);
}

// UseImprovedIonAdvection (advance_horizontal.f90:432-518), after the
// step: the divergence of the field-aligned ion velocity from UAM_Gradient
// (gradient.f90:1-86) divides the advected ions by 1 + Dt div on the
// interior cells of levels 1..nAlts; then the electrons are re-summed on
// every cell and level of the block.  One thread per element of the
// block's (-1:nLons+2,-1:nLats+2,-1:nAlts+2) array; each touches its own
// cell's ions only.
struct DivFields {
  gitm_vert_field ivel_par, glm, gl0, glp, gam, ga0, gap;
};

__global__ void __launch_bounds__(256)
    ion_divergence_kernel(HzParams p, gitm_vert_columns io, HzFields f, DivFields g) {
  const int nlo = p.n_lons, nla = p.n_lats, nA = p.n_alts;
  const long long NLo = nlo + 4, NLg = nla + 4, per_block = NLo * NLg * (nA + 4);
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= per_block * p.n_blocks) return;
  const int b = (int)(e / per_block);
  long long r = e % per_block;
  const int k = (int)(r / (NLo * NLg)) - 1;
  r %= NLo * NLg;
  const int lat = (int)(r / NLo) - 1, lon = (int)(r % NLo) - 1;
  if (lon >= 1 && lon <= nlo && lat >= 1 && lat <= nla && k >= 1 && k <= nA) {
    const double ir = *hf(io.inv_radial_distance, lon, lat, k, 0, b);
    auto v = [&](int comp, int lo, int la, int kk) {
      return *hf(g.ivel_par, lo, la, kk, comp, b);
    };
    double div = 0.0;
    if (nlo > 1) {  // east (gradient.f90:27-41)
      const double icl = 1. / fmax(*hf(io.cos_latitude, 1, lat, 0, 0, b), 0.17);
      const double gr = (*hf(g.glm, lon, 1, 0, 0, b) * v(0, lon - 1, lat, k) +
                         *hf(g.gl0, lon, 1, 0, 0, b) * v(0, lon, lat, k) +
                         *hf(g.glp, lon, 1, 0, 0, b) * v(0, lon + 1, lat, k)) *
                        ir * icl;
      div = div + gr;
    }
    {  // north (:44-56), then the tan(latitude) term (:462-477)
      const double gr = nla > 1 ? (*hf(g.gam, 1, lat, 0, 0, b) * v(1, lon, lat - 1, k) +
                                   *hf(g.ga0, 1, lat, 0, 0, b) * v(1, lon, lat, k) +
                                   *hf(g.gap, 1, lat, 0, 0, b) * v(1, lon, lat + 1, k)) *
                                      ir
                                : 0.0;
      div = div + gr;
      double tl = *hf(f.tan_latitude, 1, lat, 0, 0, b);
      if (tl > 5.0) tl = 5.0;
      if (tl < -5.0) tl = -5.0;
      div = div - tl * v(1, lon, lat, k) * ir;
    }
    {  // radial (:59-78), then 2 w / r (:480-493)
      const double r0 = *hf(f.raddist, lon, lat, k, 0, b);
      const double drp = *hf(f.raddist, lon, lat, k + 1, 0, b) - r0;
      const double drm = r0 - *hf(f.raddist, lon, lat, k - 1, 0, b);
      const double q = drm / drp;
      const double q2 = q * q;
      const double bottom = drm * (1 + q);
      const double gr =
          nA > 1 ? (q2 * v(2, lon, lat, k + 1) - v(2, lon, lat, k - 1) - (q2 - 1) * v(2, lon, lat, k)) /
                       bottom
                 : 0.0;
      div = div + gr;
      div = div + 2 * v(2, lon, lat, k) * ir;
    }
    div = div * *hf(io.cos_latitude, 1, lat, 0, 0, b);  // :498-502
    const double change = p.dt * div;
#pragma unroll
    for (int s = 0; s < NIA; s++) {  // :505-510
      double *n = hf(io.idensity_s, lon, lat, k, s, b);
      *n = *n / (1 + change);
    }
  }
  double el = 0.0;  // :512-516, every cell and level
  for (int s = 0; s < gv::NIONS - 1; s++) el = el + *hf(io.idensity_s, lon, lat, k, s, b);
  *hf(io.idensity_s, lon, lat, k, gv::NIONS - 1, b) = el;
}

// The message exchange on one device (exchange_messages_sphere.f90:4-95).
// One thread per (block, halo cell, level -1..nAlts+2): on levels 1..nAlts
// it copies every carried field from the global-grid cell the halo cell
// overlaps (past a pole: the mirrored row, the longitude turned by 180
// degrees); in the halo rows past a pole it then turns the east and north
// winds around on every level (:30-72).  Sources are blocks' own cells,
// which no thread writes.
struct XParams {
  int n_lons, n_lats, n_alts, nbl, nbt, ions;
};

struct XFields {
  gitm_vert_field itemp, etemp, ivel, latitude;
};

__global__ void __launch_bounds__(256)
    exchange_kernel(XParams p, gitm_vert_columns io, XFields f) {
  const int nlo = p.n_lons, nla = p.n_lats, nA = p.n_alts;
  const int NLo = nlo + 4, NLg = nla + 4, halo = NLo * NLg - nlo * nla;
  const long long per_block = (long long)halo * (nA + 4);
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= per_block * p.nbl * p.nbt) return;
  const int b = (int)(e / per_block);
  const int rem = (int)(e % per_block);
  const int k = rem / halo - 1, hc = rem % halo;
  // halo cell hc: the two bottom rows, the side columns of the block's
  // rows, the two top rows
  int lo, la;
  if (hc < 2 * NLo) {
    la = hc / NLo - 1;
    lo = hc % NLo - 1;
  } else if (hc < 2 * NLo + 4 * nla) {
    const int q = hc - 2 * NLo;
    la = q / 4 + 1;
    const int c = q % 4;
    lo = c < 2 ? c - 1 : nlo + c - 1;
  } else {
    const int q = hc - 2 * NLo - 4 * nla;
    la = nla + 1 + q / NLo;
    lo = q % NLo - 1;
  }
  const long long NLON = (long long)p.nbl * nlo, NLAT = (long long)p.nbt * nla;
  if (k >= 1 && k <= nA) {
    long long J = (long long)(b % p.nbl) * nlo + lo - 1, I = (long long)(b / p.nbl) * nla + la - 1;
    if (I < 0) {
      I = -1 - I;
      J += NLON / 2;
    } else if (I >= NLAT) {
      I = 2 * NLAT - 1 - I;
      J += NLON / 2;
    }
    J = ((J % NLON) + NLON) % NLON;
    const int sb = (int)(I / nla) * p.nbl + (int)(J / nlo);
    const int slo = (int)(J % nlo) + 1, sla = (int)(I % nla) + 1;
    auto cp = [&](const gitm_vert_field &g, int nc) {
      for (int c = 0; c < nc; c++) *hf(g, lo, la, k, c, b) = *hf(g, slo, sla, k, c, sb);
    };
    cp(io.rho, 1);
    cp(io.temperature, 1);
    cp(f.itemp, 1);
    cp(f.etemp, 1);
    cp(io.velocity, 3);
    cp(io.vertical_velocity, gv::NSP);
    cp(io.ndensity_s, gv::NSP);
    if (p.ions) {
      cp(io.idensity_s, gv::NIONS);
      cp(f.ivel, 3);
    }
  }
  const double half_pi = 3.14159265358979323846 / 2.0;
  const bool south = la <= 0 && *hf(f.latitude, 1, 0, 0, 0, b) < -half_pi;
  const bool north = la >= nla + 1 && *hf(f.latitude, 1, nla + 1, 0, 0, b) > half_pi;
  if (south || north) {
    for (int c = 0; c < 2; c++) {
      double *v = hf(io.velocity, lo, la, k, c, b);
      *v = -*v;
      if (f.ivel.ptr) {
        double *w = hf(f.ivel, lo, la, k, c, b);
        *w = -*w;
      }
    }
  }
}

// The checks after the exchange (:74-84): one thread per cell and level
// 1..nAlts of the blocks.
__global__ void __launch_bounds__(256)
    exchange_check_kernel(XParams p, gitm_vert_columns io, unsigned long long *err) {
  const int nlo = p.n_lons, nla = p.n_lats, nA = p.n_alts;
  const long long per_block = (long long)nlo * nla * nA;
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= per_block * p.nbl * p.nbt) return;
  const int b = (int)(e / per_block);
  const int rem = (int)(e % per_block);
  const int k = rem / (nlo * nla) + 1, cell = rem % (nlo * nla);
  const int lo = cell % nlo + 1, la = cell / nlo + 1;
  const int column = (b * nla + la - 1) * nlo + lo - 1;
  if (*hf(io.temperature, lo, la, k, 0, b) < 100.0)
    atomicMin(err, gv::error_key(column, GITM_VERT_ELOWTEMP, k));
  if (*hf(io.rho, lo, la, k, 0, b) < 0.0)
    atomicMin(err, gv::error_key(column, GITM_VERT_ENONPOSITIVE, k));
}

}  // namespace

extern "C" int gitm_horiz_exchange(gitm_vert_handle *h, const gitm_horiz_exchange_params *xp,
                                   const gitm_vert_columns *c,
                                   const gitm_horiz_exchange_fields *xf) {
  if (!h || !xp || !c || !xf) return GITM_VERT_EINVAL;
  const int nlo = c->n_lons, nla = c->n_lats;
  if (nlo < 1 || nla < 2 || c->n_alts < 1 || xp->n_blocks_lon < 1 || xp->n_blocks_lat < 1)
    return GITM_VERT_EINVAL;
  if ((long long)xp->n_blocks_lon * xp->n_blocks_lat != c->n_blocks) return GITM_VERT_EINVAL;
  if (((long long)xp->n_blocks_lon * nlo) % 2) return GITM_VERT_EINVAL;
  const gitm_vert_field *req[] = {&c->rho, &c->temperature, &c->velocity,
                                  &c->vertical_velocity, &c->ndensity_s, &xf->i_temperature,
                                  &xf->e_temperature, &xf->latitude};
  for (const gitm_vert_field *g : req)
    if (!g->ptr) return GITM_VERT_EINVAL;
  const bool ions = xp->use_ion_advection != 0;
  if (ions && (!c->idensity_s.ptr || !xf->ion_velocity.ptr)) return GITM_VERT_EINVAL;
  XParams p;
  p.n_lons = nlo;
  p.n_lats = nla;
  p.n_alts = c->n_alts;
  p.nbl = xp->n_blocks_lon;
  p.nbt = xp->n_blocks_lat;
  p.ions = ions;
  XFields f;
  f.itemp = xf->i_temperature;
  f.etemp = xf->e_temperature;
  f.ivel = xf->ion_velocity;
  f.latitude = xf->latitude;
  const long long halo = (long long)(nlo + 4) * (nla + 4) - (long long)nlo * nla;
  const long long n1 = halo * (c->n_alts + 4) * c->n_blocks;
  const long long n2 = (long long)nlo * nla * c->n_alts * c->n_blocks;
  if ((n1 + 255) / 256 > 0x7fffffffLL || (n2 + 255) / 256 > 0x7fffffffLL) return GITM_VERT_EINVAL;
  GV_HIP(hipSetDevice(h->device));
  hipLaunchKernelGGL(exchange_kernel, dim3((unsigned)((n1 + 255) / 256)), dim3(256), 0,
                     h->stream, p, *c, f);
  GV_HIP(hipGetLastError());
  hipLaunchKernelGGL(exchange_check_kernel, dim3((unsigned)((n2 + 255) / 256)), dim3(256), 0,
                     h->stream, p, *c, h->d_err);
  GV_HIP(hipGetLastError());
  return GITM_VERT_OK;
}

extern "C" int gitm_horiz_advance(gitm_vert_handle *h, const gitm_horiz_params *hp,
                                  const gitm_vert_columns *c, const gitm_horiz_fields *hf_) {
  if (!h || !hp || !c || !hf_) return GITM_VERT_EINVAL;
  const int nlo = c->n_lons, nla = c->n_lats;
  if (nlo < 1 || nla < 1 || c->n_blocks < 1 || c->n_alts < 1) return GITM_VERT_EINVAL;
  const int cells = nlo * nla;
  if (cells > 256) return GITM_VERT_EUNSUPPORTED;  // one lane per cell
  if (!(hp->dt > 0.0)) return GITM_VERT_EINVAL;
  const gitm_vert_field *req[] = {&c->rho, &c->temperature, &c->velocity,
                                  &c->vertical_velocity, &c->ndensity_s, &c->gamma,
                                  &c->inv_radial_distance, &c->cos_latitude,
                                  &hf_->inv_dlon_gb, &hf_->inv_dlon_fb, &hf_->dlon_fb,
                                  &hf_->inv_dlat_gb, &hf_->inv_dlat_fb, &hf_->dlat_fb,
                                  &hf_->radial_distance, &hf_->latitude, &hf_->tan_latitude,
                                  &hf_->cmax_horizontal};
  for (const gitm_vert_field *g : req)
    if (!g->ptr) return GITM_VERT_EINVAL;
  const bool ions = hp->use_ion_advection != 0;
  if (ions && (!c->idensity_s.ptr || !c->ivelocity.ptr)) return GITM_VERT_EINVAL;
  const bool improved = ions && hp->use_improved_ion_advection != 0;
  const bool topo = hp->use_topography != 0;
  if (topo && (!hf_->d_alt.ptr || !hf_->dalt_dlon.ptr || !hf_->dalt_dlat.ptr))
    return GITM_VERT_EINVAL;
  DivFields dv;
  dv.ivel_par = hf_->ivelocity_par;
  dv.glm = hf_->grad_lon_m;
  dv.gl0 = hf_->grad_lon_0;
  dv.glp = hf_->grad_lon_p;
  dv.gam = hf_->grad_lat_m;
  dv.ga0 = hf_->grad_lat_0;
  dv.gap = hf_->grad_lat_p;
  if (improved)
    for (const gitm_vert_field *g : {&dv.ivel_par, &dv.glm, &dv.gl0, &dv.glp, &dv.gam, &dv.ga0,
                                     &dv.gap})
      if (!g->ptr) return GITM_VERT_EINVAL;
  const int nv = ions ? NV_IONS : NV_NEUTRAL, plane = (nla + 4) * (nlo + 4);
  // altitudes per workgroup: what the caller asks (at most 256 lanes, and the
  // slab of every variable with its new values in a CU's LDS), else as many as
  // fill 256 lanes with 40 KB of LDS, but no more than leave two workgroups
  // for each of the 256 CUs; with topography a workgroup takes a block,
  // whatever is asked
  const size_t slab = (size_t)nv * (plane + cells) * sizeof(double);
  int apw = 1;
  if (topo) {
    if (slab > 160 * 1024) return GITM_VERT_EINVAL;
  } else if (hp->altitudes_per_workgroup > 0) {
    apw = hp->altitudes_per_workgroup;
    if (apw * cells > 256 || apw * slab > 160 * 1024) return GITM_VERT_EINVAL;
  } else {
    if (slab > 160 * 1024) return GITM_VERT_EINVAL;
    const size_t group = (size_t)HZ_GROUP * plane * sizeof(double);
    const long long most = (long long)c->n_alts * c->n_blocks / 512;
    while ((apw + 1) * cells <= 256 && (apw + 1) * group <= 40 * 1024 && apw + 1 <= most) apw++;
  }
  apw = std::min(apw, c->n_alts);
  HzParams p;
  p.dt = hp->dt;
  p.omega = hp->omega_body;
  p.beta = hp->beta_limiter;
  p.use_coriolis = hp->use_coriolis != 0;
  p.n_lons = nlo;
  p.n_lats = nla;
  p.n_alts = c->n_alts;
  p.n_blocks = c->n_blocks;
  p.apw = apw;
  p.alt_groups = topo ? 1 : (c->n_alts + apw - 1) / apw;
  const long long nwg = (long long)p.alt_groups * c->n_blocks;
  if (nwg > 0x7fffffffLL) return GITM_VERT_EINVAL;
  HzFields f;
  f.inv_dlon_gb = hf_->inv_dlon_gb;
  f.inv_dlon_fb = hf_->inv_dlon_fb;
  f.dlon_fb = hf_->dlon_fb;
  f.inv_dlat_gb = hf_->inv_dlat_gb;
  f.inv_dlat_fb = hf_->inv_dlat_fb;
  f.dlat_fb = hf_->dlat_fb;
  f.raddist = hf_->radial_distance;
  f.latitude = hf_->latitude;
  f.tan_latitude = hf_->tan_latitude;
  f.cmax = hf_->cmax_horizontal;
  f.temp_source = hf_->temp_source;
  f.dalt = hf_->d_alt;
  f.dalt_dlon = hf_->dalt_dlon;
  f.dalt_dlat = hf_->dalt_dlat;
  GV_HIP(hipSetDevice(h->device));
  // GITM's default 9 x 9 blocks take the kernels with the block shape fixed
  const bool b99 = nlo == 9 && nla == 9;
  const int lanes = ((apw * cells + 63) / 64) * 64;
  const dim3 grid((unsigned)nwg);
  if (topo) {
    // teams of three variables where six of them fit a workgroup, else of six
    const bool three = lanes <= 128;
    const dim3 block((1 + (three ? 4 : 2) + (ions ? 1 : 0)) * lanes);
    const size_t lds =
        ((size_t)nv * plane + 2 * hz_pad(nlo) + 3 * (size_t)cells) * sizeof(double);
    const auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, grid, block, lds, h->stream, p, *c, f, h->d_err, lanes);
    };
    if (three && b99)
      ions ? launch(horiz_topo_kernel<true, 3, 9, 9>) : launch(horiz_topo_kernel<false, 3, 9, 9>);
    else if (three)
      ions ? launch(horiz_topo_kernel<true, 3, 0, 0>) : launch(horiz_topo_kernel<false, 3, 0, 0>);
    else
      ions ? launch(horiz_topo_kernel<true, 6, 0, 0>) : launch(horiz_topo_kernel<false, 6, 0, 0>);
  } else {
    const size_t lds =
        ((size_t)apw * HZ_GROUP * plane + 2 * hz_pad(nlo)) * sizeof(double);
    const auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, grid, dim3(lanes), lds, h->stream, p, *c, f, h->d_err);
    };
    if (b99)
      ions ? launch(horiz_flat_kernel<true, 9, 9>) : launch(horiz_flat_kernel<false, 9, 9>);
    else
      ions ? launch(horiz_flat_kernel<true, 0, 0>) : launch(horiz_flat_kernel<false, 0, 0>);
  }
  GV_HIP(hipGetLastError());
  if (improved) {
    const long long n =
        (long long)(nlo + 4) * (nla + 4) * (c->n_alts + 4) * (long long)c->n_blocks;
    const long long nb = (n + 255) / 256;
    if (nb > 0x7fffffffLL) return GITM_VERT_EINVAL;
    hipLaunchKernelGGL(ion_divergence_kernel, dim3((unsigned)nb), dim3(256), 0, h->stream, p,
                       *c, f, dv);
    GV_HIP(hipGetLastError());
  }
  return GITM_VERT_OK;
}

// ---------------------------------------------------------------------------
// Host-array entry point (the Fortran drop-in): every field the step reads is
// staged on the device over exactly the index ranges the step touches, halo
// cells included; the written ones come back.
// ---------------------------------------------------------------------------
namespace {
constexpr size_t kHostStageBase = 64;  // staging slots after the vertical entry's
}  // namespace

extern "C" int gitm_horiz_advance_host(gitm_vert_handle *h, const gitm_horiz_params *hp,
                                       const gitm_vert_columns *c,
                                       const gitm_horiz_fields *hf_) {
  if (!h || !hp || !c || !hf_) return GITM_VERT_EINVAL;
  gitm_vert_columns d = *c;
  gitm_horiz_fields g = *hf_;
  const int n = c->n_lons, m = c->n_lats, nA = c->n_alts, nb = c->n_blocks;
  if (n < 1 || m < 1 || nA < 1 || nb < 1) return GITM_VERT_EINVAL;
  const bool ions = hp->use_ion_advection != 0;
  const bool improved = ions && hp->use_improved_ion_advection != 0;
  std::vector<HostSpan> sp;
  auto full = [&](gitm_vert_field *f, int nc, bool w) {
    sp.push_back({f, -1, n + 2, -1, m + 2, -1, nA + 2, nc, w});
  };
  auto lat1 = [&](gitm_vert_field *f) {  // (-1:nLats+2, nBlocks)
    sp.push_back({f, 1, 1, -1, m + 2, f->first_level, f->first_level, 1, false});
  };
  full(&d.rho, 1, true);
  full(&d.temperature, 1, true);
  full(&d.velocity, 3, true);
  full(&d.vertical_velocity, gv::NSP, true);
  full(&d.ndensity_s, gv::NSP, true);
  full(&d.gamma, 1, false);
  full(&d.inv_radial_distance, 1, false);
  lat1(&d.cos_latitude);
  if (ions) {
    full(&d.idensity_s, gv::NIONS, true);
    full(&d.ivelocity, 3, false);
  }
  for (gitm_vert_field *f : {&g.inv_dlon_gb, &g.inv_dlon_fb, &g.dlon_fb, &g.inv_dlat_gb,
                             &g.inv_dlat_fb, &g.dlat_fb, &g.radial_distance})
    full(f, 1, false);
  lat1(&g.latitude);
  lat1(&g.tan_latitude);
  sp.push_back({&g.cmax_horizontal, 0, n + 1, 0, m + 1, 0, nA + 1, 2, false});
  if (g.temp_source.ptr) sp.push_back({&g.temp_source, 1, n, 1, m, 1, nA, 1, true});
  if (hp->use_topography)
    for (gitm_vert_field *f : {&g.d_alt, &g.dalt_dlon, &g.dalt_dlat})
      sp.push_back({f, 1, n, 1, m, 1, nA, 1, false});
  if (improved) {
    full(&g.ivelocity_par, 3, false);
    for (gitm_vert_field *f : {&g.grad_lon_m, &g.grad_lon_0, &g.grad_lon_p})
      sp.push_back({f, 1, n, 1, 1, f->first_level, f->first_level, 1, false});
    for (gitm_vert_field *f : {&g.grad_lat_m, &g.grad_lat_0, &g.grad_lat_p})
      sp.push_back({f, 1, 1, 1, m, f->first_level, f->first_level, 1, false});
  }
  GV_HIP(hipSetDevice(h->device));
  HostStaging st;
  int rc = stage_in(h, sp, nb, kHostStageBase, st);
  if (rc) return rc;
  rc = gitm_horiz_advance(h, hp, &d, &g);
  if (rc) return rc;
  rc = stage_out(h, sp, kHostStageBase, st);
  if (rc) return rc;
  return gitm_vert_get_error(h, nullptr);
}
