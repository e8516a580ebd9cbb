// root_cost_check.cpp -- how many powers shock_raref_root of flux64.hpp takes on fast faces (host).
//
//   root_cost_check GAMMA N   N random shock + rarefaction faces, pressures and densities over six
//                             decades, whose speeds |du| + 2 c_II/(gamma-1) lie between 1e4 and 6e4
// Prints the faces, the mean and the largest number of powers of one face.  (A gas whose 1/gm is
// not an integer: each evaluation of the function and each Newton step is one power.)
#include <math.h>
#include <stdio.h>
#include <stdlib.h>

static long powers;
static double counted_pow(double x, double y) {
  powers++;
  return pow(x, y);
}
#define pow counted_pow
#include "../asteriy_2d_amd/csrc/flux64.hpp"
#undef pow

using namespace ast::d64;

static unsigned long long st = 0x2545F4914F6CDD1Dull;
static double urand() {
  st ^= st >> 12;
  st ^= st << 25;
  st ^= st >> 27;
  return (double)((st * 2685821657736338717ull) >> 11) * (1.0 / 9007199254740992.0);
}

int main(int argc, char** argv) {
  if (argc != 3) return 2;
  const GasD a = make_gas(atof(argv[1]));
  if (a.n != 0) return 3;
  const int n = atoi(argv[2]);
  int faces = 0;
  long sum = 0, most = 0;
  while (faces < n) {
    double pI = exp(-6.9 + 13.8 * urand()), pII = exp(-6.9 + 13.8 * urand());
    if (pI > pII) { const double t = pI; pI = pII; pII = t; }
    const double rI = exp(-6.9 + 13.8 * urand()), rII = exp(-6.9 + 13.8 * urand());
    // the densities' unit brings the speeds to 1e4 .. 6e4
    const double cII = sqrt(a.g * pII / rII), q = pow(pI / pII, a.gm);
    const double lo = a.c2g1 * cII * (q - 1.0);
    const double hi = (pII - pI) / sqrt(0.5 * rI * (a.g2 * pII + a.g1 * pI));
    const double du = lo + (hi - lo) * urand();
    const double f = (1e4 + 5e4 * urand()) / (fabs(du) + a.c2g1 * cII);
    int it;
    bool capped = false;
    powers = 0;
    shock_raref_root(a, f * du, pI, rI / (f * f), pII, f * cII, q, it, capped);
    sum += powers;
    if (powers > most) most = powers;
    faces++;
  }
  printf("%d %.3f %ld\n", faces, (double)sum / faces, most);
  return 0;
}
