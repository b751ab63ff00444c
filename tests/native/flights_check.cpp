// Prints flights_estimate (mt_tune.h) for each line "Z1 m1 E Z2 m2 Ed" of stdin.
#include <cstdio>

#include "mt_tune.h"

int main() {
  double Z1, m1, E, Z2, m2, Ed;
  while (std::scanf("%lf %lf %lf %lf %lf %lf", &Z1, &m1, &E, &Z2, &m2, &Ed) == 6)
    std::printf("%.17g\n", mt::flights_estimate(Z1, m1, E, Z2, m2, Ed));
}
