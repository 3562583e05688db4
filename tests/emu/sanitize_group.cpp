// sanitize_group.cpp -- TEST INFRASTRUCTURE ONLY.
//
// The AUSM step split over the species (gitm_amd/csrc/vert_group.h) as a program
// of its own, for the host sanitizers: each thread of a column's workgroup is a
// CPU thread, a workgroup barrier a std::barrier over all of them and a
// wavefront's ordering (wave_sync) one over its own lanes only, so that
// ThreadSanitizer reports what wavefronts exchange without a workgroup barrier
// between; the LDS block has the size of a launch's.  Reads sanitize_main.cpp's
// case file.  Two runs, over LDS filled with NaN and with -1e300, must give the
// same bits: nothing that is read comes from a slot never written.
#include <stdio.h>
#include <string.h>

#define GV_HOST_EMULATION 1
#include <atomic>
#include <barrier>
#include <memory>
#include <thread>
#include <vector>

#include "vert_group.h"
#include "vert_params.h"

namespace {

struct Shared {
  std::barrier<> bar;
  std::vector<std::unique_ptr<std::barrier<>>> wave;
  std::atomic<int> orflag{0};
  std::atomic<unsigned long long> err{~0ULL};
  explicit Shared(int n) : bar(n) {}
};

struct Ctx {
  using real = double;
  int lane_;
  Shared *sh;
  int lane() const { return lane_; }
  int uniform(int x) const { return x / 64 * 64; }
  void sync() { sh->bar.arrive_and_wait(); }
  void wave_sync() { sh->wave[lane_ / 64]->arrive_and_wait(); }
  bool sync_or(bool p) {
    if (p) sh->orflag.store(1);
    sync();
    const bool r = sh->orflag.load() != 0;
    sync();
    if (lane_ == 0) sh->orflag.store(0);
    sync();
    return r;
  }
  void report(unsigned long long key) {
    unsigned long long cur = sh->err.load();
    while (key < cur && !sh->err.compare_exchange_weak(cur, key)) {
    }
  }
  void diff_powers(double temp, double sign, double (&out)[6]) const {
    const double lt = log(temp);
    for (int u = 0; u < 6; u++) out[u] = exp((sign * gv::DEXU[u]) * lt);
  }
};

gitm_vert_field field(double *p, int per_col, int lev, int comp, int first) {
  gitm_vert_field f{};
  f.ptr = p;
  f.s_lon = per_col;
  f.s_lev = lev;
  f.s_comp = comp;
  f.first_level = first;
  return f;
}

}  // namespace

int main(int argc, char **argv) {
  FILE *fp = argc == 2 ? fopen(argv[1], "rb") : nullptr;
  int hdr[8];
  if (!fp || fread(hdr, sizeof(int), 8, fp) != 8 || hdr[0] != 1196840532) return 2;
  const int nc = hdr[1], na = hdr[2], n_steps = hdr[4], flags = hdr[5], L = na + 4;
  const bool ions = flags & 1, msis = flags & 2, gswm = flags & 4, waccm = flags & 8;
  // values per column of each array in the file
  std::vector<int> per = {6 * L, 6 * L, 3 * L, L, L, L, L, L, L, L, L, L, L, L, 1};
  if (ions) per.insert(per.end(), {10 * L, 3 * L, 1, 1});
  if (msis) per.push_back(9);
  if (gswm || waccm) per.push_back(6);
  std::vector<std::vector<double>> in;
  for (int n : per) {
    in.emplace_back((size_t)n * nc);
    if (fread(in.back().data(), sizeof(double), in.back().size(), fp) != in.back().size()) return 2;
  }
  fclose(fp);

  gitm_vert_params p;
  gv::default_params(&p);
  p.use_ion_advection = ions;
  p.use_msis = msis;
  p.use_gswm_tides = gswm;
  p.use_waccm_tides = waccm;

  auto run = [&](double fill) {
    std::vector<std::vector<double>> a = in;
    a.emplace_back((size_t)nc * 6 * L);
    a.emplace_back((size_t)nc * L);
    gitm_vert_columns c{};
    c.n_lons = nc;
    c.n_lats = c.n_blocks = 1;
    c.n_alts = na;
    gitm_vert_field *lf[] = {&c.ndensity_s, &c.vertical_velocity, &c.velocity, &c.temperature,
                             &c.rho, &c.temp_unit, &c.mean_major_mass, &c.gamma, &c.cmax,
                             &c.eddy, &c.altitude, &c.gravity, &c.inv_radial_distance, &c.dalt};
    size_t i = 0;
    for (; i < 14; i++) *lf[i] = field(a[i].data(), per[i], 1, L, -1);
    c.cos_latitude = field(a[i++].data(), 1, 0, 0, 0);
    if (ions) {
      c.idensity_s = field(a[i++].data(), 10 * L, 1, L, -1);
      c.ivelocity = field(a[i++].data(), 3 * L, 1, L, -1);
      c.sza = field(a[i++].data(), 1, 0, 0, 0);
      c.mlat = field(a[i++].data(), 1, 0, 0, 0);
    }
    if (msis) c.msis_bc = field(a[i++].data(), 9, 0, 1, 0);
    if (gswm || waccm) {
      gitm_vert_field *tf[] = {&c.tides_east, &c.tides_north, &c.tides_temp};
      for (int d = 0; d < 3; d++) *tf[d] = field(a[i].data() + 2 * d, 6, 1, 0, -1);
      i++;
    }
    c.log_ns = field(a[i++].data(), 6 * L, 1, L, -1);
    c.ndensity = field(a[i++].data(), L, 1, L, -1);
    if (gv::check_args(&p, &c, GITM_VERT_AUSM, n_steps)) exit(2);
    const gv::KParams kp = gv::make_kparams(&p, &c, GITM_VERT_AUSM, n_steps, nullptr);
    const int stride = gv::group_stride(na), threads = gv::group_threads(na);
    Shared sh(gv::NG * L);
    for (int w = 0; w < threads; w += 64) {
      int n = 0;
      for (int t = w; t < w + 64; t++) n += t % stride < L;
      sh.wave.push_back(std::make_unique<std::barrier<>>(n));
    }
    std::vector<double> lds(gv::group_lds_bytes(na, ions) / sizeof(double), fill);
    std::vector<std::thread> th;
    for (int t = 0; t < threads; t++) {
      if (t % stride >= L) continue;
      th.emplace_back([&, t] {
        Ctx cx{t, &sh};
        for (int q = 0; q < nc; q++) {
          if (ions)
            gv::run_group_column<true>(cx, kp, c, q, lds.data(), kp.dt, q, na);
          else
            gv::run_group_column<false>(cx, kp, c, q, lds.data(), kp.dt, q, na);
          cx.sync();
        }
      });
    }
    for (auto &x : th) x.join();
    if (sh.err.load() != ~0ULL) {
      fprintf(stderr, "error word %llx\n", (unsigned long long)sh.err.load());
      exit(1);
    }
    return a;
  };

  const auto a = run(__builtin_nan("")), b = run(-1e300);
  for (size_t i = 0; i < a.size(); i++)
    if (memcmp(a[i].data(), b[i].data(), a[i].size() * sizeof(double)) != 0) {
      fprintf(stderr, "array %zu depends on what LDS held\n", i);
      return 1;
    }
  printf("ok\n");
  return 0;
}
