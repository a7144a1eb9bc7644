// Driver for the CPU run of the register stages of fft_device.h (cut out by
// tests/test_stage_error.py into stages_cpu.h): root mean square error, against
// long double butterflies with exact twiddles, of a tile's outermost stage of RB
// levels as first_stage computes it and with twiddles that are products.
#include <cmath>
#include <random>

#include "stages_cpu.h"

typedef long double ld;
struct cl {
  ld x, y;
};
static const ld PI = 3.14159265358979323846264338327950288L;

template <int L, int RB, bool INV>
void run() {
  constexpr int R = 1 << RB;
  std::vector<cd> tl(L / 2);
  for (int t = 0; t < L / 2; t++) tl[t] = make_double2((double)cosl(2 * PI * t / L), (double)sinl(2 * PI * t / L));
  std::mt19937_64 rng(L + RB);
  std::normal_distribution<double> nd;
  ld fine = 0, prod = 0, norm = 0;
  for (int rep = 0; rep < 200; rep++)
    for (int q = 0; q < L / R; q++) {
      cd a[R], b[R];
      cl e[R];
      for (int t = 0; t < R; t++) {
        a[t] = b[t] = make_double2(nd(rng), nd(rng));
        e[t] = {a[t].x, a[t].y};
      }
      first_stage<L, RB, INV>(a, tl.data(), q);
      cd tb[RB];
      level_bases<RB>(tl.data(), q, 1, tb);
      if constexpr (INV) dit_levels<RB>(b, tb);
      else dif_levels<RB>(b, tb);
      for (int n = 0; n < RB; n++) {
        const int l = INV ? RB - 1 - n : n, half = R >> (l + 1);
        for (int t = 0; t < R; t++) {
          if ((t & (2 * half - 1)) >= half) continue;
          const ld w = 2 * PI * (ld)(q + (t & (half - 1)) * (L / R)) * (1 << l) / L, c = cosl(w), s = sinl(w);
          cl u = e[t], v = e[t + half];
          if (INV) v = {v.x * c + v.y * s, v.y * c - v.x * s};
          e[t] = {u.x + v.x, u.y + v.y};
          u = {u.x - v.x, u.y - v.y};
          e[t + half] = INV ? u : cl{u.x * c - u.y * s, u.x * s + u.y * c};
        }
      }
      for (int t = 0; t < R; t++) {
        fine += (a[t].x - e[t].x) * (a[t].x - e[t].x) + (a[t].y - e[t].y) * (a[t].y - e[t].y);
        prod += (b[t].x - e[t].x) * (b[t].x - e[t].x) + (b[t].y - e[t].y) * (b[t].y - e[t].y);
        norm += e[t].x * e[t].x + e[t].y * e[t].y;
      }
    }
  printf("%d %d %d %.6Le %.6Le\n", L, RB, (int)INV, sqrtl(fine / norm), sqrtl(prod / norm));
}

int main() {
  run<64, 2, false>();
  run<64, 2, true>();
  run<128, 3, false>();
  run<128, 3, true>();
  run<2048, 3, false>();
  run<2048, 3, true>();
  run<256, 4, false>();
  run<256, 4, true>();
  run<4096, 4, false>();
  run<4096, 4, true>();
  return 0;
}
