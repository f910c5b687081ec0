// Host check of the exact and the scaled fixed-point accumulators of tallymap_amd/csrc/tm_device.h (test
// infrastructure).  Modes (argv[1]):
//   (none)  reads f32 values (one hex word per line on stdin), emits them into one bin with tm_xemit_with (a plain
//           add standing in for the device's int64 atomic), prints the readout's bits and the flag;
//   words   reads TM_XW int64 words (hex, two's complement) of one bin, prints tm_xread's bits, its flag and
//           tm_xread_f64's bits: the readout of words that are not canonical (any signed values, as concurrent carries leave them);
//   wide    reads pairs (low word hex u64, count decimal i32), prints tm_wide_f64's bits for each.
#include <cstdio>
#include <cstdint>
#include <cstring>
#include "../../tallymap_amd/csrc/tm_device.h"

struct PlainAdd {
  i64 operator()(u64* a, int j, i64 q) const { const i64 o = (i64)a[j]; a[j] = (u64)o + (u64)q; return o; }
};

int main(int argc, char** argv) {
  const char* mode = argc > 1 ? argv[1] : "";
  if (!strcmp(mode, "words")) {
    u64 w[TM_XW];
    for (int j = 0; j < TM_XW; ++j)
      if (scanf("%llx", &w[j]) != 1) return 2;
    bool bad = false;
    const float r = tm_xread(w, &bad);
    printf("%08x %d %016llx\n", tm_f2u(r), (int)bad, (unsigned long long)tm_d2u(tm_xread_f64(w)));
    return 0;
  }
  if (!strcmp(mode, "wide")) {
    unsigned long long lo;
    int c;
    while (scanf("%llx %d", &lo, &c) == 2) printf("%016llx\n", (unsigned long long)tm_d2u(tm_wide_f64(lo, c)));
    return 0;
  }
  u64 w[TM_XW] = {};
  bool flag = false;
  unsigned b;
  while (scanf("%x", &b) == 1) flag = tm_xemit_with(w, tm_u2f(b), PlainAdd()) || flag;
  bool bad = false;
  const float r = tm_xread(w, &bad);
  printf("%08x %d\n", tm_f2u(r), (int)(flag || bad));
  return 0;
}
