// Host checks of tallymap_amd/csrc/tm_libm.h against glibc (test infrastructure).
//   libm_check erfinv_normal   every f32 argument jax.random.normal passes to erf_inv (2^23 uniform values):
//                              tm_erfinvf vs the reference CPU target's formula with glibc log / sqrt
//   libm_check erfinv_all <stride>
//                              every stride-th f32 in (-1, 1) (stride 1: all 2,130,706,430, OpenMP): tm_erfinvf vs
//                              the reference formula, bitwise
//   libm_check log <n> <seed>  n random t in [2^-24, 1]: |tm_log_erfinv(t) - glibc log(t)| / max(1, |log t|)
//   libm_check f32 <fn> <stride> <offset>
//                              logf expf sinf cosf atanf exp2f log2f expm1f log1pf tanhf logistic asinf acosf
//                              sinhf coshf atanhf asinhf acoshf erff erfcf tanf lgammaf on every stride-th f32 bit pattern
//                              from offset
//                              (stride 1: all 2^32): bitwise mismatches and the largest ulp distance
//   libm_check uniform         every f32 that jax.random.uniform(key) produces (2^23 values u in [0, 1)), through
//                              the argument forms the configs use: logf(1 - u) (the slab's free path) and
//                              sinf / cosf(f32(2 pi) u) (the azimuths of the slab and of walk on spheres): bitwise
//   libm_check atan2 <n> <seed>
//                              n random (y, x) pairs of finite f32 over the full exponent range: tm_atan2f vs glibc
//   libm_check f64 <fn> <n> <seed>
//                              the float64 restatements (exp exp2 expm1 log1p tanh sinh cosh atanh erf erfc) on n
//                              sampled arguments and the special values, bitwise against glibc
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <cstdint>
#include "../../tallymap_amd/csrc/tm_device.h"
#include "../../tallymap_amd/csrc/tm_libm.h"

static double ref_giles(double y) {        // reference host.py:107-118 with glibc's log / sqrt
  const double a = fabs(y);
  double w = -log((1.0 - a) * (1.0 + a)), p;
  if (w < 5.0) { w -= 2.5; p = 2.81022636e-08; p = 3.43273939e-07 + p * w; p = -3.5233877e-06 + p * w;
    p = -4.39150654e-06 + p * w; p = 0.00021858087 + p * w; p = -0.00125372503 + p * w; p = -0.00417768164 + p * w;
    p = 0.246640727 + p * w; p = 1.50140941 + p * w; }
  else { w = sqrt(w) - 3.0; p = -0.000200214257; p = 0.000100950558 + p * w; p = 0.00134934322 + p * w;
    p = -0.00367342844 + p * w; p = 0.00573950773 + p * w; p = -0.0076224613 + p * w; p = 0.00943887047 + p * w;
    p = 1.00167406 + p * w; p = 2.83297682 + p * w; }
  return p * a; }
static float ref_erfinvf(float y) {
  if (!(y > -1.0f && y < 1.0f)) return y == 1.0f ? INFINITY : (y == -1.0f ? -INFINITY : NAN);
  return y == 0.0f ? y : (float)copysign(ref_giles(y), (double)y); }

static double ref_erfinv(double y) {      // reference host.py:117-129 with glibc's erf / erfc / exp / log
  if (!(y > -1.0 && y < 1.0)) return y == 1.0 ? INFINITY : (y == -1.0 ? -INFINITY : NAN);
  if (y == 0.0) return y;
  const double a = fabs(y);
  double x = ref_giles(y);
  for (int i = 0; i < 8; ++i) {
    const double f = a < 0.5 ? erf(x) - a : (1.0 - a) - erfc(x);
    const double d = 1.1283791670955126 * exp(-x * x);
    const double dx = f / (d * (1.0 + x * f / d));
    x -= dx;
    if (fabs(dx) <= 2.3e-16 * x) break;
  }
  return copysign(x, y); }

static float ref_logistic(float x) { return 1.0f / (1.0f + expf(-x)); }   // op_table.py:243-247

int main(int argc, char** argv) {
  if (argc > 1 && !strcmp(argv[1], "uniform")) {
    long n = 0, bad = 0;
    const float twopi = (float)(2.0 * M_PI);
    for (uint32_t m = 0; m < (1u << 23); ++m) {
      const float u = tm_fmax(0.0f, (tm_u2f(m | 0x3f800000u) - 1.0f) * 1.0f + 0.0f);
      const float a = 1.0f - u, phi = twopi * u;
      n += 3;
      if (tm_f2u(tm_logf(a)) != tm_f2u(logf(a))) { if (++bad < 10) printf("  logf(%a)\n", a); }
      if (tm_f2u(tm_sinf(phi)) != tm_f2u(sinf(phi))) { if (++bad < 10) printf("  sinf(%a)\n", phi); }
      if (tm_f2u(tm_cosf(phi)) != tm_f2u(cosf(phi))) { if (++bad < 10) printf("  cosf(%a)\n", phi); }
    }
    printf("uniform: %ld arguments, %ld mismatches\n", n, bad);
    return bad != 0;
  }
  if (argc > 1 && !strcmp(argv[1], "erfinv_normal")) {
    const float lo = tm_u2f(0xbf7fffffu), span = 1.0f - lo;
    long n = 0, bad = 0, logdiff = 0;
    for (uint32_t m = 0; m < (1u << 23); ++m) {
      const float f = tm_u2f(m | 0x3f800000u) - 1.0f;
      const float r = f * span;
      const float s = r + lo;
      const float u = tm_fmax(lo, s);
      const float a = tm_erfinvf(u), b = ref_erfinvf(u);
      const double ad = fabs((double)u);
      if (tm_log_erfinv((1.0 - ad) * (1.0 + ad)) != log((1.0 - ad) * (1.0 + ad))) ++logdiff;
      ++n;
      if (tm_f2u(a) != tm_f2u(b)) { if (++bad < 10) printf("  u=%a tm=%a ref=%a\n", u, a, b); }
    }
    printf("erfinv_normal: %ld arguments, %ld f32 mismatches (double log differs on %ld)\n", n, bad, logdiff);
    return bad != 0;
  }
  if (argc > 2 && !strcmp(argv[1], "erfinv_all")) {
    const int64_t stride = atoll(argv[2]);
    long n = 0, bad = 0;
#pragma omp parallel for reduction(+ : n, bad) schedule(dynamic, 64)
    for (int64_t blk = 0; blk < 0x3f800000ll; blk += 1 << 16) {
      for (int64_t b = blk; b < blk + (1 << 16) && b < 0x3f800000ll; b += stride) {
        for (int s = 0; s < 2; ++s) {
          const float y = tm_u2f((uint32_t)b | (s ? 0x80000000u : 0u));
          ++n;
          if (tm_f2u(tm_erfinvf(y)) != tm_f2u(ref_erfinvf(y))) ++bad;
        }
      }
    }
    printf("erfinv_all: %ld arguments, %ld f32 mismatches\n", n, bad);
    return bad != 0;
  }
  if (argc > 3 && !strcmp(argv[1], "log")) {
    long n = atol(argv[2]);
    srand48(atol(argv[3]));
    double worst = 0.0;
    for (long i = 0; i < n; ++i) {
      const double x = 0x1p-24 + (1.0 - 0x1p-24) * drand48();
      const double r = log(x);
      const double e = fabs(tm_log_erfinv(x) - r) / (fabs(r) > 1.0 ? fabs(r) : 1.0);
      if (e > worst) worst = e;
    }
    printf("log: %ld t in [2^-24, 1], max |error| / max(1, |log t|) = %a\n", n, worst);
    return worst > 0x1p-51;
  }
  if (argc > 4 && !strcmp(argv[1], "f32")) {
    float (*mine)(float) = nullptr;
    float (*ref)(float) = nullptr;
    if (!strcmp(argv[2], "logf")) { mine = tm_logf; ref = logf; }
    else if (!strcmp(argv[2], "expf")) { mine = tm_expf; ref = expf; }
    else if (!strcmp(argv[2], "sinf")) { mine = tm_sinf; ref = sinf; }
    else if (!strcmp(argv[2], "cosf")) { mine = tm_cosf; ref = cosf; }
    else if (!strcmp(argv[2], "sincosf_s")) { mine = [](float x) { float s, c; tm_sincosf(x, s, c); return s; }; ref = sinf; }
    else if (!strcmp(argv[2], "sincosf_c")) { mine = [](float x) { float s, c; tm_sincosf(x, s, c); return c; }; ref = cosf; }
    else if (!strcmp(argv[2], "atanf")) { mine = tm_atanf; ref = atanf; }
    else if (!strcmp(argv[2], "exp2f")) { mine = tm_exp2f; ref = exp2f; }
    else if (!strcmp(argv[2], "log2f")) { mine = tm_log2f; ref = log2f; }
    else if (!strcmp(argv[2], "expm1f")) { mine = tm_expm1f; ref = expm1f; }
    else if (!strcmp(argv[2], "log1pf")) { mine = tm_log1pf; ref = log1pf; }
    else if (!strcmp(argv[2], "tanhf")) { mine = tm_tanhf; ref = tanhf; }
    else if (!strcmp(argv[2], "logistic")) { mine = tm_logisticf; ref = ref_logistic; }
    else if (!strcmp(argv[2], "asinf")) { mine = tm_asinf; ref = asinf; }
    else if (!strcmp(argv[2], "acosf")) { mine = tm_acosf; ref = acosf; }
    else if (!strcmp(argv[2], "sinhf")) { mine = tm_sinhf; ref = sinhf; }
    else if (!strcmp(argv[2], "coshf")) { mine = tm_coshf; ref = coshf; }
    else if (!strcmp(argv[2], "atanhf")) { mine = tm_atanhf; ref = atanhf; }
    else if (!strcmp(argv[2], "asinhf")) { mine = tm_asinhf; ref = asinhf; }
    else if (!strcmp(argv[2], "acoshf")) { mine = tm_acoshf; ref = acoshf; }
    else if (!strcmp(argv[2], "erff")) { mine = tm_erff; ref = erff; }
    else if (!strcmp(argv[2], "erfcf")) { mine = tm_erfcf; ref = erfcf; }
    else if (!strcmp(argv[2], "tanf")) { mine = tm_tanf; ref = tanf; }
    else if (!strcmp(argv[2], "lgammaf")) { mine = tm_lgammaf; ref = lgammaf; }   // ((-15, -2): lgammaf itself)
    if (!mine) return 2;
    const uint64_t stride = strtoull(argv[3], nullptr, 0), off = strtoull(argv[4], nullptr, 0);
    long n = 0, bad = 0, maxulp = 0;
    // (OpenMP over 2^16 blocks of bit patterns; a block's first argument is the next multiple of stride past off)
#pragma omp parallel for reduction(+ : n, bad) reduction(max : maxulp) schedule(dynamic, 16)
    for (int64_t blk = 0; blk < (1ll << 16); ++blk) {
      const uint64_t lo = (uint64_t)blk << 16, hi = lo + (1ull << 16);
      uint64_t u = lo <= off ? off : off + (lo - off + stride - 1) / stride * stride;
      for (; u < hi; u += stride) {
        const float x = tm_u2f((uint32_t)u), a = mine(x), b = ref(x);
        ++n;
        if (std::isnan(a) && std::isnan(b)) continue;
        if (tm_f2u(a) == tm_f2u(b)) continue;
        ++bad;
        const long d = labs((long)(int32_t)tm_f2u(a) - (long)(int32_t)tm_f2u(b));
        if (d > maxulp) maxulp = d;
      }
    }
    printf("%s: %ld arguments, %ld mismatches, max %ld ulp\n", argv[2], n, bad, maxulp);
    return 0;
  }
  if (argc > 3 && !strcmp(argv[1], "powf")) {
    // n random (x, y) pairs: half over all bit patterns, half with x near 1 and |y| moderate (results in range),
    // then every pair of a grid of special values
    long n = atol(argv[2]);
    srand48(atol(argv[3]));
    long bad = 0, maxulp = 0, tot = 0;
    auto chk = [&](float x, float y) {
      const float a = tm_powf(x, y), b = powf(x, y);
      ++tot;
      if ((std::isnan(a) && std::isnan(b)) || tm_f2u(a) == tm_f2u(b)) return;
      if (++bad <= 5) printf("  powf(%a, %a) tm=%a glibc=%a\n", x, y, a, b);
      const long d = labs((long)(int32_t)tm_f2u(a) - (long)(int32_t)tm_f2u(b));
      if (d > maxulp) maxulp = d;
    };
    for (long i = 0; i < n; ++i) {
      const uint32_t bx = (uint32_t)mrand48(), by = (uint32_t)mrand48();
      chk(tm_u2f(bx), tm_u2f(by));
      const float x = (float)(0.5 + drand48() * 3.0) * (i & 1 ? 1.0f : -1.0f);
      const float y = (float)((drand48() - 0.5) * 120.0);
      chk(x, y);
      chk(x, (float)(int)y);
      chk(tm_u2f((bx & 0x007fffffu) | 0x3f800000u), (float)((drand48() - 0.5) * 2e7));
    }
    const float sp[] = {0.0f, -0.0f, 1.0f, -1.0f, 0.5f, -0.5f, 2.0f, -2.0f, 3.0f, -3.0f, INFINITY, -INFINITY, NAN,
                        1e-45f, -1e-45f, 1e-40f, 3.4e38f, -3.4e38f, 1.0000001f, 0.99999994f, 126.0f, -126.0f,
                        150.0f, -150.0f, 127.5f, 0.25f, 16777217.0f, -16777217.0f, 8388609.0f, 1e10f, -1e10f};
    for (float x : sp)
      for (float y : sp) chk(x, y);
    printf("powf: %ld pairs, %ld mismatches, max %ld ulp\n", tot, bad, maxulp);
    return 0;
  }
  if (argc > 3 && !strcmp(argv[1], "pow")) {
    // float64 pow on n random pairs, a sixth each: all bit patterns; |x| in [2^-20, 2^20) of both signs with y in
    // (-60, 60); the same with y an integer; x within 2^-16 of 1 with |y| up to 2^40; results near the subnormal
    // boundary (2^-1000 .. 2^-1080, the scaled underflow path, both signs of the base); results near overflow
    // (2^1000 .. 2^1030).  Then every pair of a grid of special values.  Bitwise, NaN == NaN.
    const long n = atol(argv[2]);
    const uint64_t seed = (uint64_t)atol(argv[3]);
    long bad = 0;
    auto mix = [](uint64_t u) {
      u ^= u >> 31; u *= 0xBF58476D1CE4E5B9ull; u ^= u >> 27; u *= 0x94D049BB133111EBull; u ^= u >> 31;
      return u;
    };
#pragma omp parallel for reduction(+ : bad) schedule(static)
    for (long i = 0; i < n; ++i) {
      const uint64_t u = mix((uint64_t)(i + 1) * 0x9E3779B97F4A7C15ull + seed), v = mix(u + 0x632BE59BD9B4E019ull);
      const double t = (double)(u >> 11) * 0x1p-53, s = (double)(v >> 11) * 0x1p-53;
      const double sg = (v & 1) ? -1.0 : 1.0;
      double x, y;
      switch (i % 6) {
        case 0: x = tm_u2d(u); y = tm_u2d(v); break;
        case 1: x = sg * ldexp(1.0 + t, (int)(v % 41) - 20); y = (s - 0.5) * 120.0; break;
        case 2: x = sg * ldexp(1.0 + t, (int)(v % 41) - 20); y = (double)(long)((s - 0.5) * 120.0); break;
        case 3: x = tm_u2d(0x3ff0000000000000ull | (u & 0xfffffffffull)) * ((v >> 9) & 1 ? 1.0 : 0.99999);
                y = (s - 0.5) * ldexp(1.0, (int)(v % 41)); break;
        case 4: x = sg * (1.5 + 2.5 * t); y = -(1000.0 + 80.0 * s) / log2(fabs(x));
                if ((v >> 5) & 1) y = (double)(long)y; break;
        default: x = sg * (1.5 + 2.5 * t); y = (1000.0 + 30.0 * s) / log2(fabs(x));
                if ((v >> 5) & 1) y = (double)(long)y; break;
      }
      const double a = tm_pow(x, y), b = pow(x, y);
      if (tm_d2u(a) != tm_d2u(b) && !(a != a && b != b)) {
        if (++bad <= 5) printf("  pow(%a, %a): tm %a glibc %a\n", x, y, a, b);
      }
    }
    const long rnd = bad;
    bad = 0;
    const double sp[] = {0.0, -0.0, 1.0, -1.0, 0.5, -0.5, 2.0, -2.0, 3.0, -3.0, INFINITY, -INFINITY, NAN, 5e-324,
                         -5e-324, 2.2250738585072014e-308, 1.7976931348623157e308, -1.7976931348623157e308,
                         1.0000000000000002, 0.99999999999999989, 1022.0, -1022.0, 1075.0, -1075.0, 0x1p53,
                         0x1p53 + 2.0, 0x1p52 + 1.0, -(0x1p52 + 1.0), 1e-20, 1e20, 0x1p-66, 0x1p63, -0x1p63, 0.25};
    for (double x : sp)
      for (double y : sp) {
        const double a = tm_pow(x, y), b = pow(x, y);
        if (tm_d2u(a) != tm_d2u(b) && !(a != a && b != b)) {
          if (++bad <= 5) printf("  pow(%a, %a): tm %a glibc %a\n", x, y, a, b);
        }
      }
    printf("f64 pow: %ld pairs, %ld mismatches; %zu special pairs, %ld mismatches\n", n, rnd,
           (sizeof(sp) / sizeof(sp[0])) * (sizeof(sp) / sizeof(sp[0])), bad);
    return rnd + bad != 0;
  }
  if (argc > 3 && !strcmp(argv[1], "atan2")) {
    long n = atol(argv[2]);
    srand48(atol(argv[3]));
    long bad = 0, maxulp = 0;
    for (long i = 0; i < n; ++i) {
      const uint32_t by = (uint32_t)mrand48(), bx = (uint32_t)mrand48();
      const float y = tm_u2f(by), x = tm_u2f(bx);
      if (!std::isfinite(y) || !std::isfinite(x)) { --i; continue; }
      const float a = tm_atan2f(y, x), b = atan2f(y, x);
      if (tm_f2u(a) == tm_f2u(b)) continue;
      ++bad;
      const long d = labs((long)(int32_t)tm_f2u(a) - (long)(int32_t)tm_f2u(b));
      if (d > maxulp) maxulp = d;
    }
    printf("atan2: %ld pairs, %ld mismatches, max %ld ulp\n", n, bad, maxulp);
    return 0;
  }
  if (argc > 4 && !strcmp(argv[1], "f64")) {
    // float64 exp exp2 expm1 log1p tanh sinh cosh atanh erf erfc against glibc: n samples, a quarter each of random
    // bit patterns (every class), uniform draws over the working range, random magnitudes 2^-60 .. 2^20 of both
    // signs, and arguments in the bands around each branch boundary of the restated code (a boundary high word
    // +- 2 with a random low word, both signs); then the special values.  Bitwise, NaN == NaN.
    struct Fn { const char* name; double (*mine)(double); double (*ref)(double); double lo, hi;
                uint32_t edges[12]; };
    static const Fn fns[] = {
        {"exp", [](double x) { return tm_exp(x); }, [](double x) { return exp(x); }, -746.0, 710.0,
         {0x3c900000u, 0x40800000u, 0x40900000u, 0x40862e42u, 0x408633ceu, 0x40874910u}},
        {"exp2", [](double x) { return tm_exp2(x); }, [](double x) { return exp2(x); }, -1080.0, 1025.0,
         {0x3c900000u, 0x40800000u, 0x40900000u, 0x408d0000u, 0x40910c00u, 0x408ff000u}},
        {"expm1", [](double x) { return tm_expm1(x); }, [](double x) { return expm1(x); }, -50.0, 710.0,
         {0x4043687au, 0x40862e42u, 0x3fd62e42u, 0x3ff0a2b2u, 0x3c900000u, 0x4035ffffu, 0x40340000u}},
        {"log1p", [](double x) { return tm_log1p(x); }, [](double x) { return log1p(x); }, -1.0, 1.0e6,
         {0x3fda827au, 0x3fd2bec3u, 0x3fd2bec4u, 0x3e200000u, 0x3c900000u, 0x43400000u, 0x3ff00000u}},
        {"tanh", [](double x) { return tm_tanh(x); }, [](double x) { return tanh(x); }, -25.0, 25.0,
         {0x40360000u, 0x3c800000u, 0x3ff00000u}},
        {"sinh", [](double x) { return tm_sinh(x); }, [](double x) { return sinh(x); }, -711.0, 711.0,
         {0x40360000u, 0x3e300000u, 0x3ff00000u, 0x40862e42u, 0x408633ceu}},
        {"cosh", [](double x) { return tm_cosh(x); }, [](double x) { return cosh(x); }, -711.0, 711.0,
         {0x40360000u, 0x3fd62e43u, 0x3c800000u, 0x40862e42u, 0x408633ceu}},
        {"atanh", [](double x) { return tm_atanh(x); }, [](double x) { return atanh(x); }, -1.0, 1.0,
         {0x3fe00000u, 0x3e300000u, 0x3ff00000u, 0x3fefffffu}},
        {"erf", [](double x) { return tm_erf(x); }, [](double x) { return erf(x); }, -7.0, 7.0,
         {0x3feb0000u, 0x3ff40000u, 0x4006db6du, 0x4006db6eu, 0x40180000u, 0x3e300000u, 0x00800000u}},
        {"log", [](double x) { return tm_log(x); }, [](double x) { return log(x); }, 0.0, 4.0,
         {0x3fee0000u, 0x3ff10900u, 0x3fe60000u, 0x3ff60000u, 0x00100000u, 0x000fffffu, 0x7fefffffu, 0x3ff00000u}},
        {"log2", [](double x) { return tm_log2(x); }, [](double x) { return log2(x); }, 0.0, 4.0,
         {0x3feea4afu, 0x3ff0b559u, 0x3fe60000u, 0x3ff60000u, 0x00100000u, 0x000fffffu, 0x7fefffffu, 0x3ff00000u}},
        {"erfinv", [](double x) { return tm_erfinv(x); }, [](double x) { return ref_erfinv(x); }, -1.0, 1.0,
         {0x3fe00000u, 0x3fefffffu, 0x3feffff0u, 0x3c900000u, 0x3e300000u}},
        {"lgamma", [](double x) { return tm_lgamma(x); }, [](double x) { return lgamma(x); }, 0.0, 40.0,
         {0x3b900000u, 0x3feccccdu, 0x3fe76944u, 0x3fcda661u, 0x3ffbb4c3u, 0x3ff3b4c4u, 0x40000000u, 0x40200000u,
          0x43900000u, 0x3ff00000u}},
        {"asinh", [](double x) { return tm_asinh(x); }, [](double x) { return asinh(x); }, -30.0, 30.0,
         {0x3e300000u, 0x41b00000u, 0x40000000u, 0x3ff00000u}},
        {"acosh", [](double x) { return tm_acosh(x); }, [](double x) { return acosh(x); }, 1.0, 30.0,
         {0x41b00000u, 0x40000000u, 0x3ff00000u, 0x3ff00001u, 0x40000001u}},
        {"erfc", [](double x) { return tm_erfc(x); }, [](double x) { return erfc(x); }, -7.0, 28.0,
         {0x3feb0000u, 0x3ff40000u, 0x4006db6du, 0x4006db6eu, 0x40180000u, 0x403c0000u, 0x3fd00000u,
          0x3c700000u}},
    };
    const Fn* f = nullptr;
    for (const Fn& c : fns)
      if (!strcmp(argv[2], c.name)) f = &c;
    if (!f) return 2;
    const long n = atol(argv[3]);
    int ne = 0;
    while (ne < 12 && f->edges[ne]) ++ne;
    long bad = 0;
    auto chk = [&](double x) {
      const double a = f->mine(x), b = f->ref(x);
      if (tm_d2u(a) == tm_d2u(b) || (a != a && b != b)) return;
      if (++bad <= 5) printf("  %s(%a): tm %a glibc %a\n", f->name, x, a, b);
    };
#pragma omp parallel for reduction(+ : bad) schedule(static)
    for (long i = 0; i < n; ++i) {
      uint64_t u = (uint64_t)(i + 1) * 0x9E3779B97F4A7C15ull + (uint64_t)atol(argv[4]);
      u ^= u >> 31; u *= 0xBF58476D1CE4E5B9ull; u ^= u >> 27; u *= 0x94D049BB133111EBull; u ^= u >> 31;
      const double t = (double)(u >> 11) * 0x1p-53;
      double x;
      switch (i & 3) {
        case 0: x = tm_u2d(u); break;
        case 1: x = f->lo + t * (f->hi - f->lo); break;
        case 2: x = ldexp(1.0 + t, (int)(u % 81) - 60) * ((u >> 8) & 1 ? -1.0 : 1.0); break;
        default: {
          const uint32_t hw = f->edges[(u >> 40) % ne] + (uint32_t)((u >> 36) % 5) - 2u;
          x = tm_u2d(((uint64_t)(hw | ((u >> 35) & 1 ? 0x80000000u : 0u)) << 32) | (u & 0xffffffffull));
        }
      }
      const double a = f->mine(x), b = f->ref(x);
      if (tm_d2u(a) != tm_d2u(b) && !(a != a && b != b)) ++bad;
    }
    const long rnd = bad;
    bad = 0;
    const double sp[] = {0.0, -0.0, 1.0, -1.0, 0.5, -0.5, 2.0, -2.0, INFINITY, -INFINITY, NAN, 5e-324, -5e-324,
                         2.2250738585072014e-308, -2.2250738585072014e-308, 1e-300, -1e-300, 1e300, -1e300,
                         709.782712893384, -708.3964185322641, -745.1332191019411, 1024.0, -1022.0, -1074.0,
                         -1075.0, 22.0, -22.0, 6.0, -6.0, 28.0, 0.84375, 1.25, 0.25, 0.99999999999999989,
                         -0.99999999999999989, 1e-10, -1e-10, 3.0, -3.0};
    for (double x : sp) chk(x);
    printf("f64 %s: %ld samples, %ld mismatches; %zu special values, %ld mismatches\n", f->name, n, rnd,
           sizeof(sp) / sizeof(sp[0]), bad);
    return rnd + bad != 0;
  }
  fprintf(stderr, "usage: libm_check erfinv_normal | erfinv_all <stride> | log <n> <seed> | f32 <fn> <stride> "
                  "<offset> | atan2 <n> <seed> | f64 <fn> <n> <seed>\n");
  return 2;
}
