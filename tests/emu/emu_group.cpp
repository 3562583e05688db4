// emu_group.cpp -- TEST INFRASTRUCTURE ONLY.
//
// Host build of the AUSM step split over the species (gitm_amd/csrc/
// vert_group.h): each thread of a column's workgroup that owns a level runs as
// a CPU thread, a barrier is a std::barrier and the LDS block an array of
// exactly the size that a launch gets.
#define GV_HOST_EMULATION 1
#include <atomic>
#include <barrier>
#include <thread>
#include <vector>

#include "vert_group.h"
#include "vert_params.h"

namespace {

struct Shared {
  std::barrier<> bar;
  std::atomic<int> orflag{0};
  std::atomic<unsigned long long> err{~0ULL};
  explicit Shared(int n) : bar(n) {}
};

struct EmuCtx {
  using real = double;
  int lane_;
  Shared *sh;
  int lane() const { return lane_; }
  int uniform(int x) const { return x / 64 * 64; }
  void sync() { sh->bar.arrive_and_wait(); }
  void wave_sync() { sync(); }
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

}  // namespace

// n_steps AUSM steps of columns 0..n_cols-1 of `c`.
extern "C" int gv_emu_group(const gitm_vert_params *p, const gitm_vert_columns *c, int n_steps,
                            int n_cols, gitm_vert_error *e) {
  const int rc = gv::check_args(p, c, GITM_VERT_AUSM, n_steps);
  if (rc) return rc;
  const gv::KParams kp = gv::make_kparams(p, c, GITM_VERT_AUSM, n_steps, nullptr);
  const int L = c->n_alts + 4, stride = gv::group_stride(c->n_alts);
  Shared sh(gv::NG * L);
  std::vector<double> lds(gv::group_lds_bytes(c->n_alts, kp.ions != 0) / sizeof(double), 0.0);
  std::vector<std::thread> th;
  for (int t = 0; t < gv::group_threads(c->n_alts); t++) {
    if (t % stride >= L) continue;
    th.emplace_back([&, t] {
      EmuCtx cx{t, &sh};
      for (int q = 0; q < n_cols; q++) {
        if (kp.ions)
          gv::run_group_column<true>(cx, kp, *c, q, lds.data(), kp.dt, q, kp.n_alts);
        else
          gv::run_group_column<false>(cx, kp, *c, q, lds.data(), kp.dt, q, kp.n_alts);
        cx.sync();
      }
    });
  }
  for (auto &x : th) x.join();
  gv::decode_error(sh.err.load(), e);
  return e->code;
}

extern "C" int gv_emu_group_max_alts(int ions) {
  int m = 0;
  for (int n = 10; n <= GITM_VERT_MAX_NALTS; n++)
    if (gv::group_fits(n, ions != 0)) m = n;
  return m;
}
