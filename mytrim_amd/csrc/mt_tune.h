// The flights and direct recoils a cascade is expected to have, how a launch
// admits its primaries, and the launch phases of a cascade launch with the rate
// they project for a launch of more histories (host code of the runs and of the
// autotuner, mt_autotune).
//
// A launch ramps up until the admission of its middle primary, runs at a
// steady rate until the admission of its last one, then drains: the last
// cascades' longest flight chains run on an emptying device.  The kernel
// stamps both admissions (wall clock, flights ended by then).  A launch of N
// collisions is projected to take the sample's ramp and drain (their time
// and the collisions done in them) plus the rest of its collisions at the
// steady rate.
#pragma once
#include <stdint.h>

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

// Direct recoils of that ion above Ed: collisions that transfer more than Ed, over
// the stopping, by the Thomas-Fermi cross-section of Winterbon, Sigmund and
// Sanders, d sigma = pi a^2 f(sqrt t) / (2 t^1.5) dt with f(x) = 1.309 x^(1/3) /
// (1 + (2.618 x^(4/3))^(2/3))^1.5, and Lindhard's k sqrt(eps), for heavy ions
// falling off as 1 / sqrt(eps) above 25 keV/amu Z1^(4/3).  0.9 to 1.9 times what
// cascades have (H to U, 1 keV to 1 GeV); the integrals run on a grid of 64 steps in
// log eps.
inline double direct_estimate(double Z1, double m1, double E, double Z2, double m2, double Ed) {
  constexpr int N = 64;
  const double z = std::pow(Z1, 2.0 / 3.0) + std::pow(Z2, 2.0 / 3.0);
  const double a = 0.8853 * 0.5292 / std::sqrt(z);
  const double per_eV = a * m2 / (Z1 * Z2 * 14.4 * (m1 + m2));
  const double gamma = 4.0 * m1 * m2 / ((m1 + m2) * (m1 + m2));
  const double k = 0.0793 * std::pow(Z1, 2.0 / 3.0) * std::sqrt(Z2) * std::pow(m1 + m2, 1.5) /
                   (std::pow(z, 0.75) * std::pow(m1, 1.5) * std::sqrt(m2));
  const double e0 = per_eV * std::max(Ed, 1.0) / gamma, e1 = per_eV * E;  // eps of threshold and ion
  if (!(e1 > e0)) return 0.0;
  const double step = std::log(e1 / e0) / N, fast = Z1 > 2.0 ? 2.5e4 * m1 * std::pow(Z1, 4.0 / 3.0) : 1e300;
  double over[N + 1];  // integral of f / x^2 from e0, x = sqrt t
  double loss = 0.0, sum = 0.0, f0 = 0.0, x0 = 0.0, y0 = 0.0;
  for (int i = 0; i <= N; ++i) {
    const double x = e0 * std::exp(step * i), c = std::cbrt(x);
    const double d = 1.0 + 1.899 * std::pow(x, 8.0 / 9.0);
    const double f = 1.309 * c / (d * std::sqrt(d));
    over[i] = i == 0 ? 0.0 : over[i - 1] + 0.5 * step * (f0 / x0 + f / x);
    loss = i == 0 ? 0.75 * x * f : loss + 0.5 * step * (f0 * x0 + f * x);  // integral of f from 0
    // transfers from Ed (x = sqrt(e0 eps), halfway to e0 on this grid) to the largest
    const double n = over[i] - 0.5 * (over[i / 2] + over[(i + 1) / 2]);
    const double e = x / per_eV;
    const double se = k * std::sqrt(x) * std::min(1.0, fast / e);
    const double y = n / gamma / (loss / x + se) * x;
    if (i > 0) sum += 0.5 * step * (y0 + y);
    f0 = f;
    x0 = x;
    y0 = y;
  }
  return sum;
}

// What a batch is expected to bring: flights of the largest cascade and of the mean
// one, direct recoils of all its primaries and of the one with the most.
struct BatchWork {
  long long n = 0;
  double flights = 1.0, flights_mean = 1.0, direct_all = 0.0, direct_max = 0.0;
};

// How a launch admits its primaries (see Params)
struct AdmitPlan {
  bool strict = false;       // cascades reserved before they start
  int share = 0;             // small batch: primaries a wave admits at once, without the budget
  int late_block = 0;        // small batch: first block to start late (0: none)
  int stagger = 0;           // naps over which the blocks of another batch start
  double budget = 0.0;       // flights of live cascades
  double flights = 1.0;      // a cascade's, until 64 have ended
  long long live_floor = 0;  // cascades that may always be live
  double live_cap = 1e18;    // cascades that may be live at most
  double first_live = 1e18;  // and at most until 64 cascades have ended
};

constexpr uint64_t kMaxQueue = uint64_t(1) << 27;  // most queue slots a run takes by itself

// A queue that has room for the batch's flights needs no care; of one that has not
// (capped at kMaxQueue, a fixed scratch, a tuning), the recoils that wait decide.
// Measured, per live cascade (D: direct recoils):
//  - light ions (He in Fe, 2 MeV C in W): 0.5 to 0.9 D, while most lanes hold
//    primaries: they bring their recoils faster than lanes come free
//  - heavy ions on fewer cascades than lanes, which widen the tree: 4.4 D (Cu 500
//    keV) to 5.9 D (Xe 2 MeV in UO2) with a primary on every 16th lane, 1.8 to 3.6 D
//    on every second one, 0.2 to 0.8 D on every lane; 3 to 10 % of the flights
// So everything may start at once while 5, 3 and 1 times the estimate of D (1.1 to
// 1.5 times the truth for these ions) of what starts fits the slots.
// Else cascades are reserved first (strict) and bounded twice: by flights, 12 times
// the slots and 16 a lane in a small queue (of which lanes and stacks hold the most:
// 3 % wait), 7.5 times the slots in one that is large beside them (10 % wait); and
// by D, nine tenths of the slots.  By flights alone, 65 536 histories of 2 MeV C in W
// overflowed 2^21 slots (D is 17 % of their flights).
inline AdmitPlan plan_admission(const BatchWork& b, uint64_t qcap, int waves, int simds, int block, int stack_cap,
                                int feeders64) {
  AdmitPlan p;
  const double slots = double(qcap), n = double(b.n), lanes = 64.0 * waves;
  const bool roomy = n * b.flights <= 2.0 * slots;
  const double x = n / lanes;  // primaries per lane
  const double widen = x < 0.5 ? 5.0 - 2.0 / 3.0 * std::log2(16.0 * std::max(x, 1.0 / 16.0))
                               : std::max(1.0, 3.0 - 4.0 * (x - 0.5));
  const bool at_once = widen * std::min(b.direct_all, lanes * b.direct_max) <= slots;
  p.strict = !roomy && (qcap < kMaxQueue || !at_once);
  const int first = std::min(waves, simds);  // one wave per SIMD of a small batch admits all of it
  if (feeders64 == 0 && !p.strict && b.n <= 64ll * first) {
    p.share = int((b.n + first - 1) / first);
    p.late_block = waves > first ? first * 64 / block : 0;
  }
  const double d = std::min(b.direct_max, 2.0 * b.direct_all / std::max(n, 1.0));
  const double cap = roomy ? 1e18 : (0.9 * slots + 0.5 * stack_cap * waves) / std::max(d, 1.0);
  // The blocks of a large batch start over 256 naps (0.27 ms): started together,
  // the waves empty their lanes and crowd the shared words together (2e5 He
  // histories 30 -> 24 ms, 2e5 of 1 keV Cu 5.9 -> 5.6).  With fewer primaries than
  // lanes the first blocks would take them all, 64 a wave: 1e5 He histories take 12 ms
  // over 48 or 8 naps, 21 to 26 over 256; 7e4 of 1 keV Cu 2.0, 2.0 and 2.2 ms, 1e5 3.1,
  // 2.3 and 3.1, 7e4 He 9.0, 9.9 and 9.0, 7e4 of 2 MeV C in W 37, 42 and 59.  With three
  // waves per SIMD 8 naps are better: 1e5 He 20, 19 and 27 ms, 1.4e5 21, 20 and 39,
  // 1.4e5 of 1 keV Cu 4.2, 3.2 and 4.3.
  p.stagger = n >= lanes ? 256 : waves > 2 * simds ? 8 : 48;
  p.budget = 0.5 * slots;
  p.flights = b.flights;
  p.live_floor = waves;
  if (feeders64 > 0 && !p.strict) {
    // With wave roles the feeders' first admission is what counts.  A batch that it
    // takes nearly whole (64 a feeder) is not held back for the rest: feeders that
    // wait for the budget poll four words that every wave writes (2e5 He histories,
    // 62 feeders of 64: 47 against 32 ms).  A larger one floods the queue before the
    // few other waves have taken anything in, so until 64 cascades have ended 16 per
    // wave may be live (4e5 He histories 62 -> 46 ms, 3e5 of 2 MeV C in W 167 -> 150);
    // after that 224 per wave, counted by the flights expected, as far as the queue
    // bears it (1e6: 114 -> 84 ms unbounded against so, and 522 -> 460).  Blocks over
    // 256 naps: 1e5 He 27 ms, over 8 17; the larger ones over 16.
    const double feeders = waves * (feeders64 / 64.0);
    if (n <= 96.0 * feeders) {
      p.budget = 4.0 * slots;
      p.stagger = 8;
    } else {
      p.budget = std::min(std::max(0.5 * slots, 224.0 * waves * b.flights), 7.5 * slots + 6144.0 * waves);
      p.live_cap = cap;
      p.first_live = 16.0 * waves;
      p.stagger = 16;
    }
  }
  if (p.strict) {
    p.budget = std::min(12.0 * slots + 1024.0 * waves, 7.5 * slots + 6144.0 * waves);
    p.live_cap = cap;
    // The first cascades of a mixed batch are hardly all of its largest kind.  What may
    // start at first may stay live: the measured flights per cascade count those of
    // unfinished ones too (20 000 histories of H to Xe ions, 10 keV to 2 MeV, through
    // 2^21 slots: 54 ms with 561 live at first and 512 later, 50 with 1900; all at once
    // they take 37, but with twice as many live 1e5 of them, heaviest first, overflow)
    p.flights = std::min(b.flights, 4.0 * b.flights_mean);
    p.live_floor = (long long)std::max(std::min(512.0, double(waves)),
                                       std::min(std::min(double(waves), p.budget / p.flights), cap));
  }
  return p;
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
