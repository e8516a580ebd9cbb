// root_replay_check.cpp -- shock_raref_root of flux64.hpp (a bisection replayed from the root)
// against the bisection itself, written out here, on the host.
//
//   root_replay_check GAMMA SPEED N   N random shock + rarefaction faces, pressures and densities
//                                     over six decades, speeds scaled by SPEED
// Prints the faces whose p* differs by more than 2e-16 relative, whose iteration count differs,
// the largest relative difference, and the mean iteration count.
#include <math.h>
#include <stdio.h>
#include <stdlib.h>

#include "../asteriy_2d_amd/csrc/flux64.hpp"

using namespace ast::d64;

static unsigned long long st = 0x2545F4914F6CDD1Dull;
static double urand() {
  st ^= st >> 12;
  st ^= st << 25;
  st ^= st >> 27;
  return (double)((st * 2685821657736338717ull) >> 11) * (1.0 / 9007199254740992.0);
}

static double bisect(const GasD& a, double du, double pI, double rI, double pII, double cII,
                     int& it) {
  auto f = [&](double p) {
    const double s = sqrt((a.c2g2 / rI) / (p + a.g1g2 * pI));
    return (p - pI) * s + a.c2g1 * cII * (pow(p / pII, a.gm) - 1.0) - du;
  };
  double lo = pI, hi = pII, flo = f(lo);
  it = 0;
  if (fabs(flo) <= 1e-9) return lo;
  if (fabs(f(hi)) <= 1e-9) return hi;
  for (;;) {
    it++;
    const double mid = 0.5 * (lo + hi), fm = f(mid);
    if (fabs(fm) <= 1e-9 || it >= AST_ITER_CAP) return mid;
    if (flo * fm <= 0.0) {
      hi = mid;
    } else {
      lo = mid;
      flo = fm;
    }
  }
}

int main(int argc, char** argv) {
  if (argc != 4) return 2;
  const GasD a = make_gas(atof(argv[1]));
  const double speed = atof(argv[2]);
  const int n = atoi(argv[3]);
  int diff = 0, iters = 0;
  double worst = 0.0, sum = 0.0;
  for (int k = 0; k < n; k++) {
    // speed scales every sound speed: p by its square
    const double s2 = speed * speed;
    double pI = s2 * exp(-6.9 + 13.8 * urand()), pII = s2 * exp(-6.9 + 13.8 * urand());
    if (k % 8 == 0) pII = pI * (1.0 + 1e-6 * urand());
    if (pI > pII) { const double t = pI; pI = pII; pII = t; }
    const double rI = exp(-6.9 + 13.8 * urand()), rII = exp(-6.9 + 13.8 * urand());
    const double cII = sqrt(a.g * pII / rII);
    const double q = pow(pI / pII, a.gm);
    const double lo = a.c2g1 * cII * (q - 1.0);
    const double hi = (pII - pI) / sqrt(0.5 * rI * (a.g2 * pII + a.g1 * pI));
    double u = urand();
    if (k % 5 == 0) u = exp(-20.0 * u);  // near the two-rarefaction bound
    if (k % 7 == 0) u = 1.0 - exp(-20.0 * u);
    const double du = lo + (hi - lo) * u;
    int i0, i1;
    bool capped = false;
    const double p0 = bisect(a, du, pI, rI, pII, cII, i0);
    const double p1 = shock_raref_root(a, du, pI, rI, pII, cII, q, i1, capped);
    const double d = fabs(p1 - p0) / p0;
    if (!(d <= 2e-16)) diff++;
    if (i0 != i1) iters++;
    if (d > worst) worst = d;
    sum += i1;
  }
  printf("%d %d %.3g %.3g\n", diff, iters, worst, sum / n);
  return 0;
}
