// Host build of rbmd_amd/csrc/sincos.hpp's table variant: max |error| of
// sin(2 pi t), cos(2 pi t) against long double on a dense grid of t in
// [-1/2, 1/2], on both sides of every step between table entries, and on
// random t in [-50, 50]; then against itself at whole turns up to 2^40.
#include <cmath>
#include <cstdio>
#include <random>

#include "sincos.hpp"

int main() {
  const long double two_pi = 6.283185307179586476925286766559005768L;
  std::mt19937_64 g(1);
  std::uniform_real_distribution<double> u(-50.0, 50.0);
  long double e = 0;
  auto check = [&](double t) {
    double s, c;
    rbmd::sincos_turns_table(t, rbmd::kTurnTable, &s, &c);
    const long double th = two_pi * ((long double)t - rintl((long double)t));
    e = fmaxl(e, fmaxl(fabsl(s - sinl(th)), fabsl(c - cosl(th))));
  };
  for (int i = 0; i < 3000000; ++i) check(i < 1000001 ? (i - 500000) / 1000000.0 : u(g));
  for (int j = -129; j <= 129; ++j)
    for (double t : {j / 128.0, std::nextafter(j / 128.0, 9.0), std::nextafter(j / 128.0, -9.0)}) check(t);
  int differ = 0;
  for (int p = 0; p <= 40; ++p)
    for (int j = 0; j < 16; ++j) {
      double s0, c0, s1, c1;
      const double f = j / 4096.0;  // exact beside 2^40 turns
      rbmd::sincos_turns_table(f, rbmd::kTurnTable, &s0, &c0);
      rbmd::sincos_turns_table(std::ldexp(1.0, p) + f, rbmd::kTurnTable, &s1, &c1);
      differ += s0 != s1 || c0 != c1;
    }
  printf("%.6Le %d\n", e, differ);
  return 0;
}
