// The cascade lane's hull test on the host: a sub-step that compare_quick passes must hold no crossing for the exact
// search. Lanes run random samples through the lane program with stage time constants a factor `ratio` apart (either one
// the longer, up to argv[3]); at every sub-step the reference is also moved so that the hull ends a hair inside the
// test's margin of either level, where the test has least to spare. Prints the counts; exit status 1 where a passed
// sub-step has a crossing.
#include <cfloat>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "cascade.h"

using Lane = bsx::CascadeLane<1>;

struct NoSink {
  void push(const bsx::RawEventDev&) {}
};

static long long n_quick = 0, n_near = 0, n_bad = 0;

static void check(const Lane& lane, bool near) {
  Lane q = lane;
  const int64_t t_a = q.pc_.t_a + q.cmp_a_, t_b = q.pc_.t_a + q.cmp_b_;
  if (q.blind_until != bsx::kNotBlind || q.t_search >= t_b || !q.compare_quick()) return;
  ++n_quick;
  n_near += near;
  const int64_t lo = bsx::vmax(lane.t_search, t_a);
  bsx::cascade::SubStep sub;
  sub.t_a = t_a;
  sub.s3 = lane.s3_fn_;
  const bsx::cascade::Hit hit = bsx::cascade::search(lane.delta_fn(sub, lo), lo, t_b, lo, lane.theta_on, lane.theta_off);
  if (!hit.found) return;
  if (n_bad++ < 5)
    std::printf("passed, but fires %s at +%lld of %lld ns (tau_o %g tau_sf %g, C %g %g, c0 %g)\n", hit.on ? "on" : "off",
                (long long)(hit.t - t_a), (long long)(t_b - t_a), lane.cc.tau_o, lane.cc.tau_sf, lane.s3_fn_.C[0],
                lane.s3_fn_.C[1], lane.s3_fn_.c[0]);
}

int main(int argc, char** argv) {
  const int trials = argc > 1 ? std::atoi(argv[1]) : 1000;
  const unsigned long long seed = argc > 2 ? std::strtoull(argv[2], nullptr, 10) : 1;
  const double max_ratio = argc > 3 ? std::atof(argv[3]) : 1e3;
  std::mt19937_64 rng(seed);
  std::uniform_real_distribution<double> U(0.0, 1.0);
  std::normal_distribution<double> N01(0.0, 1.0);
  for (int it = 0; it < trials; ++it) {
    const int n = 60;
    std::vector<int64_t> ts(n);
    std::vector<float> irr(n);
    const double ratio = 1.1 * std::pow(max_ratio / 1.1, U(rng)), shorter = std::exp(U(rng) * 9.0 - 14.0);
    const double step = std::exp(U(rng) * 9.0 - 14.0), level = std::exp(U(rng) * 12.0 - 2.0);
    const double vol = std::exp(U(rng) * 8.0 - 7.0);
    const int64_t t0 = static_cast<int64_t>(U(rng) * 1e9);
    double lv = std::log(level);
    int64_t t = t0;
    for (int i = 0; i < n; ++i) {
      t += 1 + static_cast<int64_t>(step * 1e9 * U(rng));
      ts[i] = t;
      if (U(rng) < 0.8) lv += vol * N01(rng);
      irr[i] = static_cast<float>(std::exp(std::fmin(std::fmax(lv, -3.0), 14.0)));
    }
    Lane L{};
    L.pixel = 0;
    L.G = 1;
    L.theta_on = static_cast<float>(0.2 + 0.1 * U(rng));
    L.theta_off = static_cast<float>(0.2 + 0.1 * U(rng));
    if (it % 5 == 0) L.theta_on = L.theta_off = 40.0f;  // long stretches without an event
    L.leak = it % 3 == 0 ? 0.0f : static_cast<float>(0.2 * std::exp(8.0 * U(rng) - 3.0));
    L.dark = 0.2f;
    L.scale = 1.0f;
    L.irr_max = 1e9f;
    L.eps_ci = 0.0f;
    L.label_cut = 0.5f;
    L.refractory_ns = it % 2 == 0 ? 0 : 3000;
    L.ideal_reset = it % 4 == 1;
    L.t_state = t0;
    L.ts = ts.data();
    L.irr = irr.data();
    L.n = n;
    L.held[0] = irr[0];
    const double tau_a = shorter, tau_b = shorter * ratio, eps_h = 1e-3 / 8.0;
    const bool swap = U(rng) < 0.5;
    const double tau_o = swap ? tau_b : tau_a, tau_sf = swap ? tau_a : tau_b;
    L.cc = bsx::cascade::Consts{10.0f, static_cast<float>(1.0 / tau_o), static_cast<float>(1.0 / tau_sf),
                                static_cast<float>(tau_o), static_cast<float>(tau_sf), static_cast<float>(eps_h / 1.5),
                                static_cast<float>(std::fmax(eps_h / 1024.0, 32.0 * FLT_EPSILON))};
    L.i_scale = static_cast<float>(level);
    const float I = L.dark + irr[0];
    L.z = 1.0f / I;
    L.x1 = -bsx::pm::log(L.z * L.i_scale);
    L.s2 = L.s3 = L.x1;
    L.s3_ref = L.s3;
    L.t_ref = t0;
    L.blind_until = bsx::kNotBlind;
    L.t_search = t0;
    NoSink sink;
    L.start(t + 1000);
    for (long n_steps = 0;;) {
      if (L.comparing_) {
        check(L, false);
        for (int side = 0; side < 2; ++side) {
          // the reference that puts the hull's end just inside the level (the last that passes, by bisection)
          const float over = side == 0 ? L.hull_.hi - L.theta_on : L.hull_.lo + L.theta_off;
          const float drift = L.leak * bsx::ns_to_s64<float>(L.pc_.t_a + L.cmp_a_ - L.t_ref) + L.dr_ref;
          const auto at = [&](double margin) {
            Lane moved = L;
            moved.s3_ref = drift + over + (side == 0 ? 1.0f : -1.0f) * static_cast<float>(margin);
            return moved;
          };
          double no = 0.0, yes = std::fmin(L.theta_on, L.theta_off);
          if (!at(yes).compare_quick()) continue;
          for (int k = 0; k < 24; ++k) {
            const double m = 0.5 * (no + yes);
            (at(m).compare_quick() ? yes : no) = m;
          }
          check(at(yes), true);
        }
      }
      const int due = L.prepare();
      if (due == Lane::kFinished) break;
      if (due == Lane::kExact) L.compare_exact(sink);
      else if (due != Lane::kMove) L.attempt(due == Lane::kFast ? L.fast_coef() : L.slow_coef());
      if (L.n_attempts > 2000 || ++n_steps > 20000) break;  // (time constants far below the samples' spacing; an event a ns)
    }
  }
  std::printf("quick %lld near %lld crossings %lld\n", n_quick, n_near, n_bad);
  return n_bad != 0;
}
