// Host check of tm_div_by (tallymap_amd/csrc/tm_device.h: float32 division by a float64 reciprocal) against x / y, test
// infrastructure: special values x special values, pseudo-random pairs over the whole exponent range, pairs whose
// quotient is next to a midpoint of two floats, and quotients in and around the subnormal range.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include "../../tallymap_amd/csrc/tm_device.h"

static u64 st = 0x2545F4914F6CDD1Dull;
static u64 rnd() { st ^= st << 13; st ^= st >> 7; st ^= st << 17; return st; }

int main(int argc, char** argv) {
  const long n = argc > 1 ? atol(argv[1]) : 20000000;
  long bad = 0, tot = 0;
  auto chk = [&](float x, float y) {
    volatile float vy = y;
    const float g = tm_div_by(x, y, 1.0 / (double)vy), w = x / vy;
    ++tot;
    if (!((g != g && w != w) || tm_f2u(g) == tm_f2u(w)) && bad++ < 5) printf("%a / %a = %a, not %a\n", x, y, w, g);
  };
  const float fs[] = {0.0f, -0.0f, INFINITY, -INFINITY, NAN, 1e-45f, -1e-45f, 1.17549435e-38f, 3e-39f, 1.0f, -1.0f,
                      0.5f, 3.0f, 7.0f, -7.0f, 1e10f, 3.4028235e38f, 2.5f, 0.1f, 16777217.0f, 1.9999999f, 6.0f};
  for (float x : fs)
    for (float y : fs) chk(x, y);
  for (long i = 0; i < n; ++i) {
    const u64 r = rnd(), s = rnd();
    chk(tm_u2f((u32)r), tm_u2f((u32)(r >> 32)));
    const float y = tm_u2f((u32)(s & 0x7fffffu) | 0x3f800000u);
    // x next to m y, m a midpoint (25 significant bits) of two floats in [1, 2)
    const double m = 1.0 + (double)((s >> 23) & 0xffffffu) * 0x1p-24;
    chk((float)(m * y), y);
    // a quotient of up to 30 bits below and 4 above the smallest normal
    const float d = __builtin_ldexpf(tm_u2f((u32)(r & 0x7fffffu) | 0x3f800000u), -126 - 30 + (int)(s >> 58) % 34);
    chk(d, y);
    chk(d * (float)(1 + (int)(r >> 60)), (float)(1 + (int)((r >> 56) & 15u)));       // (exact and tied subnormals)
  }
  printf("%ld %ld\n", bad, tot);
  return bad != 0;
}
