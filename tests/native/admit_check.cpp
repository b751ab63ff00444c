// Reads lines of stdin.  "direct Z1 m1 E Z2 m2 Ed" prints direct_estimate;
// "plan n flights direct_all direct_max qcap waves simds block stack feeders"
// prints plan_admission's strict share late_block budget live_floor live_cap
// stagger first_live.
#include <cstdio>
#include <cstring>

#include "mt_tune.h"

int main() {
  char what[16];
  while (std::scanf("%15s", what) == 1) {
    if (!std::strcmp(what, "direct")) {
      double v[6];
      for (double& x : v)
        if (std::scanf("%lf", &x) != 1) return 1;
      std::printf("%.17g\n", mt::direct_estimate(v[0], v[1], v[2], v[3], v[4], v[5]));
    } else {
      mt::BatchWork b;
      unsigned long long qcap;
      int w, simds, block, stack, k;
      if (std::scanf("%lld %lf %lf %lf %llu %d %d %d %d %d", &b.n, &b.flights, &b.direct_all, &b.direct_max, &qcap, &w,
                     &simds, &block, &stack, &k) != 10)
        return 1;
      b.flights_mean = b.flights;
      const mt::AdmitPlan p = mt::plan_admission(b, qcap, w, simds, block, stack, k);
      std::printf("%d %d %d %.17g %lld %.17g %d %.17g\n", int(p.strict), p.share, p.late_block, p.budget, p.live_floor,
                  p.live_cap, p.stagger, p.first_live);
    }
  }
}
