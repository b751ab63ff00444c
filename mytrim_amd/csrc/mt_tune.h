// The flights a cascade is expected to have, and the launch phases of a cascade
// launch with the rate they project for a launch of more histories (host code
// of the runs and of the autotuner, mt_autotune).
//
// A launch ramps up until the admission of its middle primary, runs at a
// steady rate until the admission of its last one, then drains: the last
// cascades' longest flight chains run on an emptying device.  The kernel
// stamps both admissions (wall clock, flights ended by then).  A launch of N
// collisions is projected to take the sample's ramp and drain (their time
// and the collisions done in them) plus the rest of its collisions at the
// steady rate.
#pragma once
#include <algorithm>
#include <cmath>
#include <vector>

#include "mytrim_gpu.h"

namespace mt {

// Flights of one cascade expected from an ion (Z1, m1) of energy E in atoms
// (Z2, m2) with displacement energy Ed, before any has been counted: the
// damage energy T of the Lindhard partition with Robinson's fit
// (T = E / (1 + k g(eps))) over Ed, twice the Kinchin-Pease count T / (2 Ed).
// Full cascades ran 0.64 to 1.0 of it (H/He to Xe, 10 keV to 2 MeV); E / (2 Ed)
// alone is 13 times too many for 100 keV He in Fe and 23 for 2 MeV C in W,
// which left their batches with too small a share of the queue.
inline double flights_estimate(double Z1, double m1, double E, double Z2, double m2, double Ed) {
  const double z = std::pow(Z1, 2.0 / 3.0) + std::pow(Z2, 2.0 / 3.0);
  const double a = 0.8853 * 0.5292 / std::sqrt(z);
  const double eps = a * m2 * E / (Z1 * Z2 * 14.4 * (m1 + m2));
  const double k = 0.0793 * std::pow(Z1, 2.0 / 3.0) * std::sqrt(Z2) * std::pow(m1 + m2, 1.5) /
                   (std::pow(z, 0.75) * std::pow(m1, 1.5) * std::sqrt(m2));
  const double g = eps + 0.40244 * std::pow(eps, 0.75) + 3.4008 * std::pow(eps, 1.0 / 6.0);
  return 1.0 + E / (1.0 + k * g) / std::max(Ed, 1.0);
}

struct LaunchPhases {
  double kernel_s = 0.0;             // kernel time
  double half_s = 0.0;               // start to the middle admission (0: not stamped)
  double admit_s = 0.0;              // start to the last admission (0: not stamped)
  long long n_coll = 0, n_flight = 0;
  long long flights_half = 0;        // flights ended by the middle admission
  long long flights_admit = 0;       // flights ended by the last admission
  long long n_hist = 0;              // histories of the launch
};

// Collisions per second projected for a launch of n_batch histories at the
// sample's collisions per history.  The sample's own rate (collisions over
// kernel time) where n_batch is not larger than the sample, where the stamps
// are missing or out of order, or where the steady phase holds under a
// quarter of the flights (all admissions in the first round: fewer histories
// than the cascades the device admits at once).
inline double projected_rate(const LaunchPhases& p, long long n_batch) {
  const double whole = p.kernel_s > 0.0 ? double(p.n_coll) / p.kernel_s : 0.0;
  if (n_batch <= p.n_hist || p.n_hist <= 0 || p.n_flight <= 0 || p.kernel_s <= 0.0) return whole;
  if (!(p.half_s > 0.0 && p.admit_s > p.half_s && p.flights_admit > p.flights_half)) return whole;
  if (4 * (p.flights_admit - p.flights_half) < p.n_flight) return whole;
  const double cpf = double(p.n_coll) / double(p.n_flight);
  const double steady = double(p.flights_admit - p.flights_half) * cpf / (p.admit_s - p.half_s);
  const double w_ramp = double(p.flights_half) * cpf;
  const double w_drain = double(p.n_flight - p.flights_admit) * cpf;
  const double drain = std::max(0.0, p.kernel_s - p.admit_s);
  const double n = double(p.n_coll) / double(p.n_hist) * double(n_batch);
  return n / (p.half_s + std::max(0.0, n - w_ramp - w_drain) / steady + drain);
}

// A launch shape timed by the autotuner: its tuning, its (projected) rate and
// the waves per CU its launch ran at.
struct TimedShape {
  mt_tuning t;
  double rate;
  int occ;
};

inline bool same_shape(const mt_tuning& a, const mt_tuning& b) {
  return a.block == b.block && a.blocks_per_cu == b.blocks_per_cu && a.stack_cap == b.stack_cap;
}

// Index of the pick among v (-1 if none has a rate): the fastest, except that
// among shapes within 2 % of it (the spread of one timing) the deepest LDS
// stack wins, the fastest of those at that depth.  On full launches shallower
// stacks than a sample's pick measured slower (C3: 96 entries picked over
// 128, -8 %).
inline int pick_shape(const std::vector<TimedShape>& v) {
  double top = 0.0;
  for (const auto& e : v) top = std::max(top, e.rate);
  int best = -1;
  for (int i = 0; i < (int)v.size(); ++i) {
    const TimedShape& e = v[size_t(i)];
    if (!(e.rate > 0.0) || e.rate < 0.98 * top) continue;
    if (best < 0 || e.t.stack_cap > v[size_t(best)].t.stack_cap ||
        (e.t.stack_cap == v[size_t(best)].t.stack_cap && e.rate > v[size_t(best)].rate))
      best = i;
  }
  return best;
}

// Finalists of one group of timed shapes: for each occupancy (ascending), its
// pick if that is within `within` of the group's fastest; with runner_up,
// also the fastest shape of another block size, blocks per CU or stack depth
// at that occupancy within the same margin.
inline std::vector<TimedShape> occupancy_finalists(const std::vector<TimedShape>& v, bool runner_up,
                                                   double within = 0.9) {
  std::vector<TimedShape> out;
  double top = 0.0;
  for (const auto& e : v) top = std::max(top, e.rate);
  if (!(top > 0.0)) return out;
  std::vector<int> occs;
  for (const auto& e : v) occs.push_back(e.occ);
  std::sort(occs.begin(), occs.end());
  occs.erase(std::unique(occs.begin(), occs.end()), occs.end());
  for (int oc : occs) {
    std::vector<TimedShape> g;
    for (const auto& e : v)
      if (e.occ == oc) g.push_back(e);
    const int p = pick_shape(g);
    if (p < 0 || g[size_t(p)].rate < within * top) continue;
    out.push_back(g[size_t(p)]);
    if (!runner_up) continue;
    int second = -1;
    for (int i = 0; i < (int)g.size(); ++i)
      if (!same_shape(g[size_t(i)].t, g[size_t(p)].t) && g[size_t(i)].rate >= within * top &&
          (second < 0 || g[size_t(i)].rate > g[size_t(second)].rate))
        second = i;
    if (second >= 0) out.push_back(g[size_t(second)]);
  }
  return out;
}

}  // namespace mt
