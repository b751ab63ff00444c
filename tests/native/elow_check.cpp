// For each heavy (ion, element): e_low of the tables, the largest energy
// (keV/amu) at which the stopping's velocity yr stays at its branch limit, found
// by bisection of the reference's expressions (material.C:213-233), and vfermi.
#include <cmath>
#include <cstdio>

#include "mt_host.h"

int main() {
  using namespace mt;
  HostTarget t;
  HostMaterial m;
  for (int Z : {1, 3, 6, 14, 29, 47, 74, 92}) m.el.push_back(HostElement{Z, 2.0 * Z + 1.0, 1.0, 25.0, 3.0});
  m.rho = 5.0;
  m.prepare();
  t.mat.push_back(m);
  for (int Z = 3; Z <= 92; ++Z) {
    std::vector<Species> sp{Species{Z, 2.0 * Z + 1.0}};
    for (const auto& e : m.el)
      if (e.Z != Z) sp.push_back(Species{e.Z, e.m});
    std::vector<unsigned char> blob;
    if (!build_tables(default_coefs(), t, sp, blob).empty()) return 1;
    const TableHeader* H = reinterpret_cast<const TableHeader*>(blob.data());
    const StopConst* S = reinterpret_cast<const StopConst*>(blob.data() + H->off_stop);
    for (size_t k = 0; k < m.el.size(); ++k) {
      const double vf = S[k].vfermi, z23 = std::pow(std::cbrt(double(Z)), 2), branch = std::fmax(0.13, 1.0 / z23);
      auto low = [&](double e) {
        const double v = std::sqrt(e / 25.0) / vf;
        const double vr = v >= 1.0 ? v * vf * (1.0 + 1.0 / (5.0 * v * v))
                                   : 3.0 * vf / 4.0 * (1.0 + 2.0 * v * v / 3.0 - v * v * v * v / 15.0);
        return std::fmax(0.13, std::fmax(vr / z23, 1.0 / z23)) <= branch;
      };
      double lo = 0.0, hi = 1e6;
      if (!low(0.0)) hi = 0.0;
      for (int i = 0; i < 200; ++i) (low(0.5 * (lo + hi)) ? lo : hi) = 0.5 * (lo + hi);
      std::printf("%d %d %.9g %.9g %.9g\n", Z, m.el[k].Z, double(S[k].e_low), hi == 0.0 ? 0.0 : lo, vf);
    }
  }
}
