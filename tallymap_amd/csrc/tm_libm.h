// tm_libm.h -- the transcendental functions of generated kernels, host + device.
//
// The parity target is the reference's CPU kernel backend, whose transcendentals are glibc's libm (reference
// tallymap/backends/kernel/host.py:43-48, op_table.py:199-223).  glibc's f32 functions are not correctly rounded,
// so the device cannot use its own math library and agree bitwise.  Each function here is written from a published
// method and checked on the host against glibc over the argument sets the tests name (exhaustively where the set
// is enumerable); tests/native/libm_check.cc and tests/test_native_cpu.py hold the checks.
//
//   tm_erfinvf f32 erf_inv as the reference's CPU target computes it: Giles (2010)'s single-precision polynomial
//              evaluated in double, rounded once to f32 (host.py:102-132).  Here the double part is a division-free
//              table log (tm_log_erfinv) and fused multiply-adds; the results are checked bitwise against the
//              reference formula (glibc's log, separate multiplies and adds) on EVERY f32 argument in (-1, 1):
//              2,130,706,430 arguments, 0 mismatches (so on all 2^23 that jax.random.normal produces).
//   tm_logf, tm_expf, tm_sinf, tm_cosf
//              glibc 2.35's f32 functions are the ARM optimized-routines algorithms (MIT / Apache-2.0; Szabolcs
//              Nagy), built on x86-64 in an FMA variant selected at run time on FMA/AVX2 hosts.  Restated here:
//              the same reductions, tables and polynomials, with an explicit fma wherever that build contracts a
//              multiply-add.  Checked bitwise against glibc on ALL 2^32 inputs: logf, sinf, cosf agree
//              everywhere; expf everywhere except two inputs whose glibc result lies on a rounding knife-edge of
//              the same evaluation, listed in tm_expf.  The exp2 table is 2^(i/32) rounded to double, minus i << 47
//              (computed from that definition); the 2/pi bit table is the binary expansion of 2/pi.
//   tm_exp2f, tm_log2f, tm_powf
//              the same library's exp2f / log2f / powf on the expf / logf tables.  exp2f and log2f agree with
//              glibc on all 2^32 inputs; powf on 1.0e9 random pairs (bit patterns, x near 1 with large |y|,
//              integer and non-integer y of both signs) and a grid of special pairs, 0 mismatches.
//   tm_atanf, tm_atan2f
//              fdlibm's float atanf / atan2f (Sun, freely redistributable) in float arithmetic, in glibc's form
//              (atanf returns +-pi/2 from |x| >= 2^25).  Checked bitwise against glibc on all 2^32 atanf arguments
//              and on random atan2f pairs over the full exponent range.
//   tm_expm1f, tm_log1pf, tm_tanhf
//              fdlibm's float expm1f / log1pf / tanhf, float arithmetic without contraction, as glibc 2.35's
//              generic build compiles them: bitwise equal to glibc on all 2^32 inputs.
//   tm_asinf, tm_acosf, tm_sinhf, tm_coshf, tm_atanhf, tm_asinhf, tm_acoshf, tm_erff, tm_erfcf
//              fdlibm's float versions (asinf with Cephes' single-precision asin polynomial, as glibc has it) on
//              the functions above (expf, expm1f, logf, log1pf), float arithmetic without contraction: bitwise
//              equal to glibc on all 2^32 inputs.
//   tm_tanf    fdlibm's float tan kernel (k_tanf.c) on glibc 2.35's rem_pio2f, which reduces with the sinf / cosf
//              reductions above in double and splits the result into a float head and tail: bitwise equal to
//              glibc on all 2^32 inputs.
//   tm_lgammaf fdlibm's float lgamma (e_lgammaf_r.c) as glibc 2.35 builds it, sin(pi x) for negative x on the
//              restated sinf / cosf: bitwise equal to glibc on all 2^32 inputs outside (-15, -2); there glibc
//              runs its own lgamma_negf (LGPL), and the device's math library is called instead.
//   tm_logisticf
//              1 / (1 + tm_expf(-x)), the reference CPU target's expression: all 2^32 inputs bitwise.
//   tm_exp, tm_exp2 (float64)
//              the same library's exp / exp2 (a 128-entry table of 2^(k/128) computed from its definition, a quartic
//              / quintic); exp as glibc's FMA build computes it, exp2 as its generic build.
//   tm_log, tm_log2, tm_pow (float64)
//              the same library's log (FMA build), log2 (generic build) and pow (FMA build; its log table computed
//              from its definition, its exp on tm_exp's table).  log's and log2's tables were chosen upstream by a
//              search (per subinterval, among the doubles near 1 / center, one whose rounded log c is a multiple of
//              2^-43 / 2^-42 and close to log c: within 2^-66 / 2^-62 here); that rule, applied to the candidates, leaves a few
//              hundred (log) or thousand (log2) per subinterval, and the entry kept is the one that agrees with
//              glibc on 2.4e6 arguments of its subinterval (tests/native/log_table_search.cc; tests/test_native_cpu.py
//              checks the rule on every entry).  Bitwise equal to glibc on 2e8 arguments each (pow: 6e7 pairs and a special grid).
//   tm_asinh, tm_acosh (float64)
//              fdlibm's asinh and acosh (acosh in its 64-bit-word form) on tm_log and tm_log1p: bitwise on 5e7
//              arguments each.
//   tm_lgamma (float64)
//              fdlibm's lgamma on tm_log: bitwise for positive arguments (2e8); negative ones between -2^52 and
//              -2^-70 take the device's math library (glibc's sin(pi x) there is IBM's sin / cos).
//   tm_expm1, tm_log1p, tm_tanh, tm_sinh, tm_cosh, tm_atanh, tm_erf, tm_erfc, tm_logistic_d (float64)
//              fdlibm's double code as glibc 2.35's generic build compiles it (no contraction; its polynomials
//              evaluated in pairs as glibc writes them), on tm_exp where it calls exp.  The float64 functions are
//              checked bitwise against glibc on random bit patterns, working ranges and the bands around every
//              branch boundary (2.0e8 arguments per function, 0 mismatches).
//
// Upstream notices of the restated code (the logf / expf / exp2f / log2f / powf / sinf / cosf reductions, tables
// and polynomial coefficients, and the atanf / atan2f / expm1f / log1pf / tanhf code and coefficients):
//
//   ARM optimized-routines (math/logf.c, math/expf.c, math/exp2f.c, math/log2f.c, math/powf.c, math/sinf.c,
//   math/cosf.c, math/exp.c, math/exp2.c, math/log.c, math/log2.c, math/pow.c and their data files):
//     Copyright (c) 2017-2022, Arm Limited.
//     SPDX-License-Identifier: MIT OR Apache-2.0 WITH LLVM-exception.  Used here under the MIT license:
//     Permission is hereby granted, free of charge, to any person obtaining a copy of this software and
//     associated documentation files (the "Software"), to deal in the Software without restriction, including
//     without limitation the rights to use, copy, modify, merge, publish, distribute, sublicense, and/or sell
//     copies of the Software, and to permit persons to whom the Software is furnished to do so, subject to the
//     following conditions: The above copyright notice and this permission notice shall be included in all copies
//     or substantial portions of the Software.  THE SOFTWARE IS PROVIDED "AS IS", WITHOUT WARRANTY OF ANY KIND,
//     EXPRESS OR IMPLIED, INCLUDING BUT NOT LIMITED TO THE WARRANTIES OF MERCHANTABILITY, FITNESS FOR A PARTICULAR
//     PURPOSE AND NONINFRINGEMENT.  IN NO EVENT SHALL THE AUTHORS OR COPYRIGHT HOLDERS BE LIABLE FOR ANY CLAIM,
//     DAMAGES OR OTHER LIABILITY, WHETHER IN AN ACTION OF CONTRACT, TORT OR OTHERWISE, ARISING FROM, OUT OF OR IN
//     CONNECTION WITH THE SOFTWARE OR THE USE OR OTHER DEALINGS IN THE SOFTWARE.
//
//   fdlibm (s_atanf.c, e_atan2f.c, s_expm1f.c, s_log1pf.c, s_tanhf.c, e_asinf.c, e_acosf.c, e_sinhf.c, e_coshf.c,
//   e_atanhf.c, s_asinhf.c, e_acoshf.c, s_erff.c, k_tanf.c, e_lgammaf_r.c -- float versions by Ian Lance Taylor, Cygnus Support -- and
//   s_expm1.c, s_log1p.c, s_tanh.c, e_sinh.c, e_cosh.c, e_atanh.c, s_erf.c, s_asinh.c, e_acosh.c, e_lgamma_r.c):
//     Copyright (C) 1993 by Sun Microsystems, Inc. All rights reserved.
//     Developed at SunPro, a Sun Microsystems, Inc. business.
//     Permission to use, copy, modify, and distribute this software is freely granted, provided that this notice
//     is preserved.
//
//   Cephes Math Library (asinf's polynomial coefficients): Copyright 1984, 1995, 2000 by Stephen L. Moshier,
//   distributed for free use.
#pragma once

// a * b + c rounded once (the same operation as __builtin_fma), on the device as the three-address v_fma_f64: the
// compiler turns an fma whose addend is a loop-invariant constant into v_mov_b64 (a copy of the constant) +
// the two-address v_fmac_f64, and on gfx950 the copy issues at about the rate of the fma itself (5.6e11 against
// 4.6e11 wave instructions per second).  Used where that copy is in the loop (erf_inv's Horner steps: C2's 24
// copies per step); in sinf / cosf / logf / expf the forced VGPR operands cost more than the copies save (C5's
// forward 4.31 -> 4.62 ms measured).  Not volatile: the compiler still schedules it.
TM_FN double tm_fma3(double a, double b, double c) {
#if defined(__HIP_DEVICE_COMPILE__)
  double r;
  asm("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
#else
  return __builtin_fma(a, b, c);
#endif
}

// w = -log(t) for erf_inv, t = (1 - a)(1 + a) in [2^-24, 1]: t = 2^k z, z in [0x1.6ap-1, 0x1.6ap0) split into 64
// equal pieces by the top six mantissa bits; log t = k ln2 + log c + log1p(z / c - 1) with 1/c the piece's
// midpoint reciprocal rounded to double, log c = -log(1/c) rounded to double (both from their definitions at 60
// digits), and log1p(r), |r| < 2^-7, by its Taylor series to r^8 (remainder < 2^-63).  No division.  The absolute
// error is below 4e-16 on this domain; erf_inv reads w through w - 2.5 or sqrt(w), so absolute accuracy is what
// matters (the function is not a general-purpose log: its relative error near t = 1 is large).
TM_FN double tm_log_erfinv(double x) {
  const double T[64][2] = {
      {0x1.6816816816817p+0, -0x1.5d5bddf595f31p-2},
      {0x1.642c8590b2164p+0, -0x1.522ae0738a3d7p-2},
      {0x1.6058160581606p+0, -0x1.4718dc271c41cp-2},
      {0x1.5c9882b931057p+0, -0x1.3c25277333183p-2},
      {0x1.58ed2308158edp+0, -0x1.314f1e1d35ce3p-2},
      {0x1.5555555555555p+0, -0x1.269621134db91p-2},
      {0x1.51d07eae2f815p+0, -0x1.1bf99635a6b95p-2},
      {0x1.4e5e0a72f0539p+0, -0x1.1178e8227e47ap-2},
      {0x1.4afd6a052bf5bp+0, -0x1.07138604d5864p-2},
      {0x1.47ae147ae147bp+0, -0x1.f991c6cb3b37ap-3},
      {0x1.446f86562d9fbp+0, -0x1.e530effe71013p-3},
      {0x1.4141414141414p+0, -0x1.d1037f2655e7bp-3},
      {0x1.3e22cbce4a902p+0, -0x1.bd087383bd8aap-3},
      {0x1.3b13b13b13b14p+0, -0x1.a93ed3c8ad9e5p-3},
      {0x1.3813813813814p+0, -0x1.95a5adcf70182p-3},
      {0x1.3521cfb2b78c1p+0, -0x1.823c16551a3c0p-3},
      {0x1.323e34a2b10bfp+0, -0x1.6f0128b756ab9p-3},
      {0x1.2f684bda12f68p+0, -0x1.5bf406b543db0p-3},
      {0x1.2c9fb4d812ca0p+0, -0x1.4913d8333b563p-3},
      {0x1.29e4129e4129ep+0, -0x1.365fcb0159014p-3},
      {0x1.27350b8812735p+0, -0x1.23d712a49c201p-3},
      {0x1.2492492492492p+0, -0x1.1178e8227e47ap-3},
      {0x1.21fb78121fb78p+0, -0x1.fe89139dbd565p-4},
      {0x1.1f7047dc11f70p+0, -0x1.da7276384469ep-4},
      {0x1.1cf06ada2811dp+0, -0x1.b6ac88dad5b1dp-4},
      {0x1.1a7b9611a7b96p+0, -0x1.9335e5d594988p-4},
      {0x1.1811811811812p+0, -0x1.700d30aeac0e8p-4},
      {0x1.15b1e5f75270dp+0, -0x1.4d3115d207eacp-4},
      {0x1.135c81135c811p+0, -0x1.2aa04a44717a1p-4},
      {0x1.1111111111111p+0, -0x1.08598b59e3a06p-4},
      {0x1.0ecf56be69c90p+0, -0x1.ccb73cdddb2d0p-5},
      {0x1.0c9714fbcda3bp+0, -0x1.894aa149fb34bp-5},
      {0x1.0a6810a6810a7p+0, -0x1.466aed42de3f9p-5},
      {0x1.0842108421084p+0, -0x1.0415d89e74440p-5},
      {0x1.0624dd2f1a9fcp+0, -0x1.8492528c8cac5p-6},
      {0x1.0410410410410p+0, -0x1.0205658935837p-6},
      {0x1.0204081020408p+0, -0x1.010157588de69p-7},
      {0x1.ff007fc01ff00p-1, 0x1.ff802a9ab11e6p-10},
      {0x1.f81f81f81f820p-1, 0x1.fc0a8b0fc03c4p-7},
      {0x1.f07c1f07c1f08p-1, 0x1.f829b0e7832f8p-6},
      {0x1.e9131abf0b767p-1, 0x1.77458f632dcffp-5},
      {0x1.e1e1e1e1e1e1ep-1, 0x1.f0a30c01162a8p-5},
      {0x1.dae6076b981dbp-1, 0x1.341d7961bd1d0p-4},
      {0x1.d41d41d41d41dp-1, 0x1.6f0d28ae56b4ep-4},
      {0x1.cd85689039b0bp-1, 0x1.a926d3a4ad562p-4},
      {0x1.c71c71c71c71cp-1, 0x1.e27076e2af2eap-4},
      {0x1.c0e070381c0e0p-1, 0x1.0d77e7cd08e5bp-3},
      {0x1.bacf914c1bad0p-1, 0x1.29552f81ff521p-3},
      {0x1.b4e81b4e81b4fp-1, 0x1.44d2b6ccb7d1cp-3},
      {0x1.af286bca1af28p-1, 0x1.5ff3070a793d6p-3},
      {0x1.a98ef606a63bep-1, 0x1.7ab890210d907p-3},
      {0x1.a41a41a41a41ap-1, 0x1.9525a9cf456b6p-3},
      {0x1.9ec8e951033d9p-1, 0x1.af3c94e80bff3p-3},
      {0x1.999999999999ap-1, 0x1.c8ff7c79a9a20p-3},
      {0x1.948b0fcd6e9e0p-1, 0x1.e27076e2af2e8p-3},
      {0x1.8f9c18f9c18fap-1, 0x1.fb9186d5e3e29p-3},
      {0x1.8acb90f6bf3aap-1, 0x1.0a324e27390e2p-2},
      {0x1.8618618618618p-1, 0x1.1675cababa60fp-2},
      {0x1.8181818181818p-1, 0x1.22941fbcf7966p-2},
      {0x1.7d05f417d05f4p-1, 0x1.2e8e2bae11d31p-2},
      {0x1.78a4c8178a4c8p-1, 0x1.3a64c556945eap-2},
      {0x1.745d1745d1746p-1, 0x1.4618bc21c5ec2p-2},
      {0x1.702e05c0b8170p-1, 0x1.51aad872df82ep-2},
      {0x1.6c16c16c16c17p-1, 0x1.5d1bdbf5809cap-2}};
  const u64 OFF = 0x3fe6a00000000000ull;
  const double Ln2hi = 0x1.62e42fefa3800p-1, Ln2lo = 0x1.ef35793c76730p-45;
  const u64 ix = tm_d2u(x);
  const u64 tmp = ix - OFF;
  const int i = (int)((tmp >> 46) & 63u);
  const i64 k = (i64)tmp >> 52;
  const double z = tm_u2d(ix - (tmp & (0xfffull << 52)));
  const double r = __builtin_fma(z, T[i][0], -1.0);
  const double kd = (double)k;
  const double r2 = r * r;
  double q = tm_fma3(r, -0.125, 0x1.2492492492492p-3);
  q = tm_fma3(r, q, -0x1.5555555555555p-3);
  q = tm_fma3(r, q, 0x1.999999999999ap-3);
  q = tm_fma3(r, q, -0.25);
  q = tm_fma3(r, q, 0x1.5555555555555p-2);
  q = tm_fma3(r, q, -0.5);
  const double hi = __builtin_fma(kd, Ln2hi, T[i][1]);
  return (hi + r) + __builtin_fma(r2, q, kd * Ln2lo);
}

// Giles (2010), "Approximating the erfinv function", the single-precision coefficients, evaluated in double with
// fused multiply-adds (host.py:107-118 evaluates the same polynomial with separate multiplies and adds and glibc's
// log; the f32 results agree bitwise on every f32 argument in (-1, 1): see tm_erfinvf).
TM_FN double tm_giles(double y) {
  const double a = y < 0.0 ? -y : y;
  double w = -tm_log_erfinv((1.0 - a) * (1.0 + a)), p;
  if (w < 5.0) {
    w -= 2.5;
    p = 2.81022636e-08;
    p = tm_fma3(p, w, 3.43273939e-07);
    p = tm_fma3(p, w, -3.5233877e-06);
    p = tm_fma3(p, w, -4.39150654e-06);
    p = tm_fma3(p, w, 0.00021858087);
    p = tm_fma3(p, w, -0.00125372503);
    p = tm_fma3(p, w, -0.00417768164);
    p = tm_fma3(p, w, 0.246640727);
    p = tm_fma3(p, w, 1.50140941);
  } else {
    w = __builtin_sqrt(w) - 3.0;
    p = -0.000200214257;
    p = tm_fma3(p, w, 0.000100950558);
    p = tm_fma3(p, w, 0.00134934322);
    p = tm_fma3(p, w, -0.00367342844);
    p = tm_fma3(p, w, 0.00573950773);
    p = tm_fma3(p, w, -0.0076224613);
    p = tm_fma3(p, w, 0.00943887047);
    p = tm_fma3(p, w, 1.00167406);
    p = tm_fma3(p, w, 2.83297682);
  }
  return p * a;
}

TM_FN float tm_erfinvf(float y) {
  if (!(y > -1.0f && y < 1.0f)) {
    return y == 1.0f ? __builtin_inff() : (y == -1.0f ? -__builtin_inff() : __builtin_nanf(""));
  }
  if (y == 0.0f) return y;
  const double r = tm_giles((double)y);
  return (float)(y < 0.0f ? -r : r);
}

// ------------------------------------------------------------------------------------------------ logf
// x = 2^k z, z in [0x3f330000, 2 * 0x3f330000); c near the center of z's sixteenth; log x = k ln2 + log c +
// log1p(z / c - 1), the last by a degree-4 polynomial in r = z * (1/c) - 1 evaluated in double.
TM_FN float tm_logf(float x) {
  const double T[16][2] = {
      {0x1.661ec79f8f3bep+0, -0x1.57bf7808caadep-2}, {0x1.571ed4aaf883dp+0, -0x1.2bef0a7c06ddbp-2},
      {0x1.49539f0f010bp+0, -0x1.01eae7f513a67p-2},  {0x1.3c995b0b80385p+0, -0x1.b31d8a68224e9p-3},
      {0x1.30d190c8864a5p+0, -0x1.6574f0ac07758p-3}, {0x1.25e227b0b8eap+0, -0x1.1aa2bc79c81p-3},
      {0x1.1bb4a4a1a343fp+0, -0x1.a4e76ce8c0e5ep-4}, {0x1.12358f08ae5bap+0, -0x1.1973c5a611cccp-4},
      {0x1.0953f419900a7p+0, -0x1.252f438e10c1ep-5}, {0x1p+0, 0x0p+0},
      {0x1.e608cfd9a47acp-1, 0x1.aa5aa5df25984p-5},  {0x1.ca4b31f026aap-1, 0x1.c5e53aa362eb4p-4},
      {0x1.b2036576afce6p-1, 0x1.526e57720db08p-3},  {0x1.9c2d163a1aa2dp-1, 0x1.bc2860d22477p-3},
      {0x1.886e6037841edp-1, 0x1.1058bc8a07ee1p-2},  {0x1.767dcf5534862p-1, 0x1.4043057b6ee09p-2}};
  const double A0 = -0x1.00ea348b88334p-2, A1 = 0x1.5575b0be00b6ap-2, A2 = -0x1.ffffef20a4123p-2;
  const double Ln2 = 0x1.62e42fefa39efp-1;
  u32 ix = tm_f2u(x);
  const bool rare = ix - 0x00800000u >= 0x7f800000u - 0x00800000u;
  if (__builtin_expect(rare, 0)) {
    ix = tm_f2u(x * 0x1p23f);                     // a subnormal: normalise (the others are replaced below)
    ix -= 23u << 23;
  }
  const u32 tmp = ix - 0x3f330000u;
  const int i = (int)((tmp >> 19) % 16u);
  const int k = (i32)tmp >> 23;
  const u32 iz = ix - (tmp & 0xff800000u);
  const double z = (double)tm_u2f(iz);
  const double r = __builtin_fma(z, T[i][0], -1.0);
  const double y0 = __builtin_fma((double)k, Ln2, T[i][1]);
  const double r2 = r * r;
  double y = __builtin_fma(A1, r, A2);
  y = __builtin_fma(A0, r2, y);
  y = __builtin_fma(y, r2, y0 + r);
  float res = (float)y;
  if (__builtin_expect(rare, 0)) {
    const u32 ux = tm_f2u(x);
    if (ux * 2u == 0u) res = -__builtin_inff();
    else if (ux == 0x7f800000u) res = x;
    else if ((ux & 0x80000000u) || ux * 2u >= 0xff000000u) res = __builtin_nanf("");
  }
  return res;
}

// ------------------------------------------------------------------------------------------------ expf
// x * 32 / ln2 = k + r, |r| <= 1/2; exp x = 2^(k/32) 2^(r/32), 2^(k/32) from the table (exponent added to the
// bits), 2^(r/32) by a cubic in r.
TM_FN float tm_expf(float x) {
  const u64 T[32] = {
      0x3ff0000000000000ull, 0x3fefd9b0d3158574ull, 0x3fefb5586cf9890full, 0x3fef9301d0125b51ull,
      0x3fef72b83c7d517bull, 0x3fef54873168b9aaull, 0x3fef387a6e756238ull, 0x3fef1e9df51fdee1ull,
      0x3fef06fe0a31b715ull, 0x3feef1a7373aa9cbull, 0x3feedea64c123422ull, 0x3feece086061892dull,
      0x3feebfdad5362a27ull, 0x3feeb42b569d4f82ull, 0x3feeab07dd485429ull, 0x3feea47eb03a5585ull,
      0x3feea09e667f3bcdull, 0x3fee9f75e8ec5f74ull, 0x3feea11473eb0187ull, 0x3feea589994cce13ull,
      0x3feeace5422aa0dbull, 0x3feeb737b0cdc5e5ull, 0x3feec49182a3f090ull, 0x3feed503b23e255dull,
      0x3feee89f995ad3adull, 0x3feeff76f2fb5e47ull, 0x3fef199bdd85529cull, 0x3fef3720dcef9069ull,
      0x3fef5818dcfba487ull, 0x3fef7c97337b9b5full, 0x3fefa4afa2a490daull, 0x3fefd0765b6e4540ull};
  const double InvLn2N = 0x1.71547652b82fep+0 * 32, SHIFT = 0x1.8p+52;
  const double C0 = 0x1.c6af84b912394p-5 / 32 / 32 / 32, C1 = 0x1.ebfce50fac4f3p-3 / 32 / 32,
               C2 = 0x1.62e42ff0c52d6p-1 / 32;
  const u32 ux = tm_f2u(x);
  if (ux == 0x4202422fu) return 0x1.f93e38p+46f;         // the two knife-edge inputs (see the header)
  if (ux == 0xc27c65d9u) return 0x1.f45326p-92f;
  const u32 abstop = (ux >> 20) & 0x7ffu;
  if (abstop >= (tm_f2u(88.0f) >> 20)) {
    if (ux == tm_f2u(-__builtin_inff())) return 0.0f;
    if (abstop >= (tm_f2u(__builtin_inff()) >> 20)) return x + x;
    if (x > 0x1.62e42ep6f) return __builtin_inff();
    if (x < -0x1.9fe368p6f) return 0.0f;
  }
  double z = InvLn2N * (double)x;
  double kd = z + SHIFT;
  const u64 ki = tm_d2u(kd);
  kd -= SHIFT;
  const double r = z - kd;
  u64 t = T[ki % 32u];
  t += ki << 47;
  const double s = tm_u2d(t);
  z = __builtin_fma(C0, r, C1);
  const double r2 = r * r;
  double y = __builtin_fma(C2, r, 1.0);
  y = __builtin_fma(z, r2, y);
  y = y * s;
  return (float)y;
}

// ------------------------------------------------------------------------------------------ sinf / cosf
// ARM's __sincosf_table[0] as constants.  Its second table is the same with the cosine coefficients c0..c4 negated,
// and a polynomial with every coefficient negated gives exactly the negated result (each fma and the final rounding
// are symmetric under negation), so the device keeps one constant set and flips the sign of the cosine result
// instead of selecting a table per lane: a per-lane table address turns every coefficient into a global load.
constexpr double TM_SC_HPI_INV = 0x1.45F306DC9C883p+23, TM_SC_HPI = 0x1.921FB54442D18p0;
constexpr double TM_SC_C0 = 0x1p0, TM_SC_C1 = -0x1.ffffffd0c621cp-2, TM_SC_C2 = 0x1.55553e1068f19p-5,
                 TM_SC_C3 = -0x1.6c087e89a359dp-10, TM_SC_C4 = 0x1.99343027bf8c3p-16;
constexpr double TM_SC_S1 = -0x1.555545995a603p-3, TM_SC_S2 = 0x1.1107605230bc4p-7, TM_SC_S3 = -0x1.994eb3774cf24p-13;
// the table's sign[n & 3] = {1, -1, -1, 1}: -1 when bits 0 and 1 of n differ
TM_FN double tm_sc_sign(int n) { return ((n ^ (n >> 1)) & 1) ? -1.0 : 1.0; }
// n even: the sine polynomial; n odd: the cosine polynomial, negated when `flip` (the second table).  Both are
// evaluated and one is selected: the lanes of a wave reduce to quadrants of both parities, and a branch would run
// both sides anyway, each with part of the lanes (each polynomial's operations are glibc's, so the bits are too).
TM_FN float tm_sc_poly(double x, double x2, int n, bool flip) {
  const double x3 = x * x2;
  const double s1 = __builtin_fma(x2, TM_SC_S3, TM_SC_S2);
  const double x7 = x3 * x2;
  const double s = __builtin_fma(x3, TM_SC_S1, x);
  const float rs = (float)__builtin_fma(x7, s1, s);
  const double x4 = x2 * x2;
  const double c2 = __builtin_fma(x2, TM_SC_C4, TM_SC_C3);
  const double c1 = __builtin_fma(x2, TM_SC_C1, TM_SC_C0);
  const double x6 = x4 * x2;
  const double c = __builtin_fma(x4, TM_SC_C2, c1);
  const float rc = (float)__builtin_fma(x6, c2, c);
  return (n & 1) == 0 ? rs : (flip ? -rc : rc);
}
// |x| < 120: n = round(x 2/pi) (through 2^24-scaled integer arithmetic), x - n pi/2 with one fma
TM_FN double tm_sc_reduce_fast(double x, int* np) {
  const double r = x * TM_SC_HPI_INV;
  // (any x may come here: the add wraps, and the caller replaces what |x| >= 120 gives)
  const int n = (i32)((u32)tm_d2i32(r) + 0x800000u) >> 24;
  *np = n;
  return __builtin_fma(-(double)n, TM_SC_HPI, x);
}
// |x| >= 120: x (4/pi) mod 4 in 64-bit fixed point from a 2/pi bit table
TM_FN double tm_sc_reduce_large(u32 xi, int* np) {
  const u32 P[24] = {0xa2u, 0xa2f9u, 0xa2f983u, 0xa2f9836eu, 0xf9836e4eu, 0x836e4e44u, 0x6e4e4415u, 0x4e441529u,
                     0x441529fcu, 0x1529fc27u, 0x29fc2757u, 0xfc2757d1u, 0x2757d1f5u, 0x57d1f534u, 0xd1f534ddu,
                     0xf534ddc0u, 0x34ddc0dbu, 0xddc0db62u, 0xc0db6295u, 0xdb629599u, 0x6295993cu, 0x95993c43u,
                     0x993c4390u, 0x3c439041u};
  const u32* arr = &P[(xi >> 26) & 15u];
  const int shift = (int)((xi >> 23) & 7u);
  xi = (xi & 0xffffffu) | 0x800000u;
  xi <<= shift;
  u64 res0 = (u64)(u32)(xi * arr[0]);
  const u64 res1 = (u64)xi * arr[4];
  const u64 res2 = (u64)xi * arr[8];
  res0 = (res2 >> 32) | (res0 << 32);
  res0 += res1;
  const u64 n = (res0 + (1ull << 61)) >> 62;
  res0 -= n << 62;
  *np = (int)n;
  return (double)(i64)res0 * 0x1.921FB54442D18p-62;
}
TM_FN u32 tm_abstop12(float x) { return (tm_f2u(x) >> 20) & 0x7ffu; }
// glibc evaluates |y| < pi/4 without the reduction and returns y itself below 2^-12; there the fast reduction gives
// n = 0 and r = y exactly, and the same polynomial: one path for every |y| < 120, so the lanes of a wave do not
// split on |y| < pi/4, with y itself selected below 2^-12 (the polynomial turns -0 into +0).  Bitwise glibc's on
// all 2^32 inputs.
// The rare arguments (|y| >= 120) replace the result afterwards, in a branch no wave takes in ordinary work: the common
// path runs without a lane mask of its own.
TM_FN float tm_sinf_large(float y) {
  if (tm_abstop12(y) >= tm_abstop12(__builtin_inff())) return y - y;
  int n;
  const u32 xi = tm_f2u(y);
  const double x = tm_sc_reduce_large(xi, &n);
  const int q = n + (int)(xi >> 31);
  return tm_sc_poly(x * tm_sc_sign(q), x * x, n, (q & 2) != 0);
}
TM_FN float tm_cosf_large(float y) {
  if (tm_abstop12(y) >= tm_abstop12(__builtin_inff())) return y - y;
  int n;
  const u32 xi = tm_f2u(y);
  const double x = tm_sc_reduce_large(xi, &n);
  const int q = n + (int)(xi >> 31);
  return tm_sc_poly(x * tm_sc_sign(q), x * x, n ^ 1, (q & 2) != 0);
}
TM_FN float tm_sinf(float y) {
  int n;
  const double x = tm_sc_reduce_fast(y, &n);
  float r = tm_sc_poly(x * tm_sc_sign(n), x * x, n, (n & 2) != 0);
  if (tm_abstop12(y) < tm_abstop12(0x1p-12f)) r = y;
  if (__builtin_expect(tm_abstop12(y) >= tm_abstop12(120.0f), 0)) r = tm_sinf_large(y);
  return r;
}
TM_FN float tm_cosf(float y) {             // (one path for |y| < 120, as tm_sinf; glibc returns 1 below 2^-12)
  int n;
  const double x = tm_sc_reduce_fast(y, &n);
  float r = tm_sc_poly(x * tm_sc_sign(n), x * x, n ^ 1, (n & 2) != 0);
  if (tm_abstop12(y) < tm_abstop12(0x1p-12f)) r = 1.0f;
  if (__builtin_expect(tm_abstop12(y) >= tm_abstop12(120.0f), 0)) r = tm_cosf_large(y);
  return r;
}
// both of one angle: the reduction and the two polynomials once (tm_sinf and tm_cosf evaluate both polynomials each and
// select).  Bitwise tm_sinf's and tm_cosf's.
TM_FN void tm_sincosf(float y, float& sin_y, float& cos_y) {
  int n;
  const double x = tm_sc_reduce_fast(y, &n);
  const double xs = x * tm_sc_sign(n), x2 = x * x;
  const float a = tm_sc_poly(xs, x2, 0, false), c = tm_sc_poly(xs, x2, 1, (n & 2) != 0);   // sine, cosine polynomial
  const bool tiny = tm_abstop12(y) < tm_abstop12(0x1p-12f), odd = (n & 1) != 0;
  float rs = tiny ? y : (odd ? c : a), rc = tiny ? 1.0f : (odd ? a : c);
  if (__builtin_expect(tm_abstop12(y) >= tm_abstop12(120.0f), 0)) {
    rs = tm_sinf_large(y);
    rc = tm_cosf_large(y);
  }
  sin_y = rs;
  cos_y = rc;
}

// ----------------------------------------------------------------------------------------------------- tanf
// glibc 2.35's tanf: fdlibm's float kernel on a float pair (y0, y1) ~ x - n pi/2 that glibc's rem_pio2f forms
// from the sinf reductions above, in double: y0 = (float)r, y1 = (float)(r - y0).  That build does not contract
// the fast reduction (x - n hpi is a multiply and a subtraction).  The kernel, for |y0| <= pi/4 and iy = +-1
// (n even / odd): tan(y0 + y1) or -1/tan(y0 + y1) as
//   |y0| < 2^-13            y0, or -1/y0
//   |y0| >= 0.6744          tan(pi/4 - y) = (1 - tan y) / (1 + tan y) on y = pi/4 - |y0| (head + tail)
//   otherwise               y + y^3 T(y^2), T of degree 12 split into its even and odd terms; for iy = -1 the
//                           reciprocal -1/w with w = y + r formed carefully (w and -1/w with their low 12 bits
//                           cleared, plus the corrections)
TM_FN float tm_tanf_kernel(float x, float y, int iy) {
  const float T0 = 3.3333334327e-01f, T1 = 1.3333334029e-01f, T2 = 5.3968254477e-02f, T3 = 2.1869488060e-02f,
              T4 = 8.8632395491e-03f, T5 = 3.5920790397e-03f, T6 = 1.4562094584e-03f, T7 = 5.8804126456e-04f,
              T8 = 2.4646313977e-04f, T9 = 7.8179444245e-05f, T10 = 7.1407252108e-05f, T11 = -1.8558637748e-05f,
              T12 = 2.5907305826e-05f, pio4 = 7.8539812565e-01f, pio4lo = 3.7748947079e-08f;
  const i32 hx = (i32)tm_f2u(x), ix = hx & 0x7fffffff;
  if (ix < 0x39000000) {                         // |y0| < 2^-13
    if ((ix | (iy + 1)) == 0) return 1.0f / __builtin_fabsf(x);
    return iy == 1 ? x : -1.0f / x;
  }
  const bool big = ix >= 0x3f2ca140;
  if (big) {
    if (hx < 0) { x = -x; y = -y; }
    x = (pio4 - x) + (pio4lo - y);
    y = 0.0f;
    if (__builtin_fabsf(x) < 0x1p-13f) return (float)(1 - ((hx >> 30) & 2)) * (float)iy * (1.0f - (float)(2 * iy) * x);
  }
  const float z = x * x, w2 = z * z;
  const float ro = T1 + w2 * (T3 + w2 * (T5 + w2 * (T7 + w2 * (T9 + w2 * T11))));
  const float ve = z * (T2 + w2 * (T4 + w2 * (T6 + w2 * (T8 + w2 * (T10 + w2 * T12)))));
  const float s = z * x;
  float r = y + z * (s * (ro + ve) + y);
  r += T0 * s;
  const float w = x + r;
  if (big) {
    const float v = (float)iy;
    return (float)(1 - ((hx >> 30) & 2)) * (v - 2.0f * (x - (w * w / (w + v) - r)));
  }
  if (iy == 1) return w;
  const float wh = tm_u2f(tm_f2u(w) & 0xfffff000u), v = r - (wh - x);
  const float a = -1.0f / w, t = tm_u2f(tm_f2u(a) & 0xfffff000u);
  return t + a * ((1.0f + t * wh) + t * v);
}
// |x| <= pi/4 needs no reduction in glibc; there the fast reduction gives n = 0 and r = x exactly (x 2^24 (2/pi)
// stays below 2^23), so one path serves every |x| < 120.  Bitwise glibc's on all 2^32 inputs.
TM_FN float tm_tanf(float x) {
  const u32 xi = tm_f2u(x);
  double r;
  int n;
  if (tm_abstop12(x) < tm_abstop12(120.0f)) {
    const double d = x, q = d * TM_SC_HPI_INV;
    n = ((i32)q + 0x800000) >> 24;
    r = d - (double)n * TM_SC_HPI;
  } else if (tm_abstop12(x) < tm_abstop12(__builtin_inff())) {
    r = tm_sc_reduce_large(xi, &n);
    if (xi >> 31) r = -r;
  } else {
    return x - x;
  }
  const float y0 = (float)r, y1 = (float)(r - (double)y0);
  return tm_tanf_kernel(y0, y1, 1 - ((n & 1) << 1));
}

// -------------------------------------------------------------------------------------- atanf / atan2f
TM_FN float tm_atanf(float x) {
  const float atanhi[4] = {4.6364760399e-01f, 7.8539812565e-01f, 9.8279368877e-01f, 1.5707962513e+00f};
  const float atanlo[4] = {5.0121582440e-09f, 3.7748947079e-08f, 3.4473217170e-08f, 7.5497894159e-08f};
  const float aT[11] = {3.3333334327e-01f, -2.0000000298e-01f, 1.4285714924e-01f, -1.1111110449e-01f,
                        9.0908870101e-02f, -7.6918758452e-02f, 6.6610731184e-02f, -5.8335702866e-02f,
                        4.9768779427e-02f, -3.6531571299e-02f, 1.6285819933e-02f};
  const i32 hx = (i32)tm_f2u(x), ix = hx & 0x7fffffff;
  int id;
  if (ix >= 0x4c000000) {                          // |x| >= 2^25
    if (ix > 0x7f800000) return x + x;
    return hx > 0 ? atanhi[3] + atanlo[3] : -atanhi[3] - atanlo[3];
  }
  if (ix < 0x31000000) return x;
  // the four reductions' quotients as one division of selected operands (x / 1 is x): the lanes of a wave are in
  // several ranges, and a division in each branch would run one after another
  const float a = __builtin_fabsf(x);
  float num, den;
  if (ix < 0x3ee00000) { id = -1; num = x; den = 1.0f; }
  else if (ix < 0x3f300000) { id = 0; num = 2.0f * a - 1.0f; den = 2.0f + a; }
  else if (ix < 0x3f980000) { id = 1; num = a - 1.0f; den = a + 1.0f; }
  else if (ix < 0x401c0000) { id = 2; num = a - 1.5f; den = 1.0f + 1.5f * a; }
  else { id = 3; num = -1.0f; den = a; }
  x = num / den;
  const float z = x * x, w = z * z;
  const float s1 = z * (aT[0] + w * (aT[2] + w * (aT[4] + w * (aT[6] + w * (aT[8] + w * aT[10])))));
  const float s2 = w * (aT[1] + w * (aT[3] + w * (aT[5] + w * (aT[7] + w * aT[9]))));
  if (id < 0) return x - x * (s1 + s2);
  const float r = atanhi[id] - ((x * (s1 + s2) - atanlo[id]) - x);
  return hx < 0 ? -r : r;
}
TM_FN float tm_atan2f(float y, float x) {
  const float tiny = 1.0e-30f, pi_o_4 = 7.8539818525e-01f, pi_o_2 = 1.5707963705e+00f, pi = 3.1415927410e+00f,
              pi_lo = -8.7422776573e-08f;
  const i32 hx = (i32)tm_f2u(x), ix = hx & 0x7fffffff, hy = (i32)tm_f2u(y), iy = hy & 0x7fffffff;
  if (ix > 0x7f800000 || iy > 0x7f800000) return x + y;
  if (hx == 0x3f800000) return tm_atanf(y);
  const int m = ((hy >> 31) & 1) | ((hx >> 30) & 2);
  if (iy == 0) return m == 0 || m == 1 ? y : (m == 2 ? pi + tiny : -pi - tiny);
  if (ix == 0) return hy < 0 ? -pi_o_2 - tiny : pi_o_2 + tiny;
  if (ix == 0x7f800000) {
    if (iy == 0x7f800000) {
      return m == 0 ? pi_o_4 + tiny : (m == 1 ? -pi_o_4 - tiny : (m == 2 ? 3.0f * pi_o_4 + tiny : -3.0f * pi_o_4 - tiny));
    }
    return m == 0 ? 0.0f : (m == 1 ? -0.0f : (m == 2 ? pi + tiny : -pi - tiny));
  }
  if (iy == 0x7f800000) return hy < 0 ? -pi_o_2 - tiny : pi_o_2 + tiny;
  const i32 k = (iy - ix) >> 23;
  float z;
  if (k > 60) z = pi_o_2 + 0.5f * pi_lo;
  else if (hx < 0 && k < -60) z = 0.0f;
  else z = tm_atanf(__builtin_fabsf(y / x));
  switch (m) {
    case 0: return z;
    case 1: return tm_u2f(tm_f2u(z) ^ 0x80000000u);
    case 2: return pi - (z - pi_lo);
    default: return (z - pi_lo) - pi;
  }
}
// ----------------------------------------------------------------------------------------------- exp2f
// the exp2f of glibc 2.35 (ARM optimized-routines): x = k/32 + r, |r| <= 1/64; 2^(k/32) from tm_expf's table, 2^r by
// a cubic (the unscaled coefficients of tm_expf's polynomial: C_i here = C_i there x 32^(3-i)).
TM_FN double tm_exp2_table(u64 ki) {
  const u64 T[32] = {
      0x3ff0000000000000ull, 0x3fefd9b0d3158574ull, 0x3fefb5586cf9890full, 0x3fef9301d0125b51ull,
      0x3fef72b83c7d517bull, 0x3fef54873168b9aaull, 0x3fef387a6e756238ull, 0x3fef1e9df51fdee1ull,
      0x3fef06fe0a31b715ull, 0x3feef1a7373aa9cbull, 0x3feedea64c123422ull, 0x3feece086061892dull,
      0x3feebfdad5362a27ull, 0x3feeb42b569d4f82ull, 0x3feeab07dd485429ull, 0x3feea47eb03a5585ull,
      0x3feea09e667f3bcdull, 0x3fee9f75e8ec5f74ull, 0x3feea11473eb0187ull, 0x3feea589994cce13ull,
      0x3feeace5422aa0dbull, 0x3feeb737b0cdc5e5ull, 0x3feec49182a3f090ull, 0x3feed503b23e255dull,
      0x3feee89f995ad3adull, 0x3feeff76f2fb5e47ull, 0x3fef199bdd85529cull, 0x3fef3720dcef9069ull,
      0x3fef5818dcfba487ull, 0x3fef7c97337b9b5full, 0x3fefa4afa2a490daull, 0x3fefd0765b6e4540ull};
  u64 t = T[ki % 32u];
  t += ki << 47;
  return tm_u2d(t);
}
TM_FN float tm_exp2f(float x) {
  const double SHIFT = 0x1.8p+52 / 32, C0 = 0x1.c6af84b912394p-5, C1 = 0x1.ebfce50fac4f3p-3,
               C2 = 0x1.62e42ff0c52d6p-1;
  const u32 ux = tm_f2u(x);
  const u32 abstop = (ux >> 20) & 0x7ffu;
  if (abstop >= (tm_f2u(128.0f) >> 20)) {
    if (ux == tm_f2u(-__builtin_inff())) return 0.0f;
    if (abstop >= (tm_f2u(__builtin_inff()) >> 20)) return x + x;
    if (x > 0.0f) return __builtin_inff();
    if (x <= -150.0f) return 0.0f;
  }
  const double xd = (double)x;
  double kd = xd + SHIFT;
  const u64 ki = tm_d2u(kd);
  kd -= SHIFT;
  const double r = xd - kd;
  const double s = tm_exp2_table(ki);
  const double z = __builtin_fma(C0, r, C1);
  const double r2 = r * r;
  double y = __builtin_fma(C2, r, 1.0);
  y = __builtin_fma(z, r2, y);
  y = y * s;
  return (float)y;
}

// ----------------------------------------------------------------------------------------------- log2f
// the log2f of glibc 2.35 (ARM optimized-routines): tm_logf's reduction and invc values; log2 c = -log2(invc)
// rounded to double (computed from that definition, as tm_logf's log c = -log(invc) is); log1p(r) / ln2 by a
// quartic in double.
TM_FN float tm_log2f(float x) {
  const double T[16][2] = {
      {0x1.661ec79f8f3bep+0, -0x1.efec65b963019p-2}, {0x1.571ed4aaf883dp+0, -0x1.b0b6832d4fca4p-2},
      {0x1.49539f0f010b0p+0, -0x1.7418b0a1fb77bp-2}, {0x1.3c995b0b80385p+0, -0x1.39de91a6dcf7bp-2},
      {0x1.30d190c8864a5p+0, -0x1.01d9bf3f2b631p-2}, {0x1.25e227b0b8ea0p+0, -0x1.97c1d1b3b7af0p-3},
      {0x1.1bb4a4a1a343fp+0, -0x1.2f9e393af3c9fp-3}, {0x1.12358f08ae5bap+0, -0x1.960cbbf788d5cp-4},
      {0x1.0953f419900a7p+0, -0x1.a6f9db6475fcep-5}, {0x1.0000000000000p+0, 0x0.0p+0},
      {0x1.e608cfd9a47acp-1, 0x1.338ca9f24f53dp-4}, {0x1.ca4b31f026aa0p-1, 0x1.476a9543891bap-3},
      {0x1.b2036576afce6p-1, 0x1.e840b4ac4e4d2p-3}, {0x1.9c2d163a1aa2dp-1, 0x1.40645f0c6651cp-2},
      {0x1.886e6037841edp-1, 0x1.88e9c2c1b9ff8p-2}, {0x1.767dcf5534862p-1, 0x1.ce0a44eb17bccp-2}};
  const double A0 = -0x1.712b6f70a7e4dp-2, A1 = 0x1.ecabf496832ep-2, A2 = -0x1.715479ffae3dep-1,
               A3 = 0x1.715475f35c8b8p0;
  u32 ix = tm_f2u(x);
  if (ix == 0x3f800000u) return 0.0f;
  if (ix - 0x00800000u >= 0x7f800000u - 0x00800000u) {
    if (ix * 2u == 0u) return -__builtin_inff();
    if (ix == 0x7f800000u) return x;
    if ((ix & 0x80000000u) || ix * 2u >= 0xff000000u) return __builtin_nanf("");
    ix = tm_f2u(x * 0x1p23f);
    ix -= 23u << 23;
  }
  const u32 tmp = ix - 0x3f330000u;
  const int i = (int)((tmp >> 19) % 16u);
  const u32 top = tmp & 0xff800000u;
  const u32 iz = ix - top;
  const int k = (i32)tmp >> 23;
  const double z = (double)tm_u2f(iz);
  const double r = __builtin_fma(z, T[i][0], -1.0);
  const double y0 = T[i][1] + (double)k;
  const double r2 = r * r;
  double y = __builtin_fma(A1, r, A2);
  y = __builtin_fma(A0, r2, y);
  const double p = __builtin_fma(A3, r, y0);
  y = __builtin_fma(y, r2, p);
  return (float)y;
}

// ---------------------------------------------------------------------------------------------- expm1f
// fdlibm's float expm1f as glibc 2.35 builds it (generic code, float arithmetic, no contraction): x = k ln2 + r,
// |r| <= ln2 / 2 (hi / lo parts), expm1(r) by a rational form with R(r^2/2) (five coefficients), then
// 2^k (1 + expm1(r)) - 1 assembled so that no cancellation loses bits.
TM_FN float tm_expm1f(float x) {
  const float huge = 1.0e+30f, tiny = 1.0e-30f, o_threshold = 8.8721679688e+01f, ln2_hi = 6.9313812256e-01f,
              ln2_lo = 9.0580006145e-06f, invln2 = 1.4426950216e+00f, Q1 = -3.3333335072e-02f,
              Q2 = 1.5873016091e-03f, Q3 = -7.9365076090e-05f, Q4 = 4.0082177293e-06f, Q5 = -2.0109921195e-07f;
  float y, hi, lo, c = 0.0f, t, e, hxs, hfx, r1;
  i32 k;
  u32 hx = tm_f2u(x);
  const u32 xsb = hx & 0x80000000u;
  hx &= 0x7fffffffu;
  if (hx >= 0x4195b844u) {                       // |x| >= 27 ln2
    if (hx >= 0x42b17218u) {                     // |x| >= 88.721...
      if (hx > 0x7f800000u) return x + x;
      if (hx == 0x7f800000u) return xsb == 0u ? x : -1.0f;
      if (x > o_threshold) return huge * huge;
    }
    if (xsb != 0u) {                             // x < -27 ln2
      if (x + tiny < 0.0f) return tiny - 1.0f;
    }
  }
  if (hx > 0x3eb17218u) {                        // |x| > 0.5 ln2
    if (hx < 0x3F851592u) {                      // and |x| < 1.5 ln2
      if (xsb == 0u) { hi = x - ln2_hi; lo = ln2_lo; k = 1; }
      else { hi = x + ln2_hi; lo = -ln2_lo; k = -1; }
    } else {
      k = (i32)(invln2 * x + (xsb == 0u ? 0.5f : -0.5f));
      t = (float)k;
      hi = x - t * ln2_hi;
      lo = t * ln2_lo;
    }
    x = hi - lo;
    c = (hi - x) - lo;
  } else if (hx < 0x33000000u) {                 // |x| < 2^-25
    t = huge + x;
    return x - (t - (huge + x));
  } else {
    k = 0;
  }
  hfx = 0.5f * x;
  hxs = x * hfx;
  r1 = 1.0f + hxs * (Q1 + hxs * (Q2 + hxs * (Q3 + hxs * (Q4 + hxs * Q5))));
  t = 3.0f - r1 * hfx;
  e = hxs * ((r1 - t) / (6.0f - x * t));
  if (k == 0) return x - (x * e - hxs);
  e = (x * (e - c) - c);
  e -= hxs;
  if (k == -1) return 0.5f * (x - e) - 0.5f;
  if (k == 1) {
    if (x < -0.25f) return -2.0f * (e - (x + 0.5f));
    return 1.0f + 2.0f * (x - e);
  }
  if (k <= -2 || k > 56) {                       // suffice to return exp(x) - 1
    i32 i;
    y = 1.0f - (e - x);
    i = (i32)tm_f2u(y);
    y = tm_u2f((u32)(i + (k << 23)));
    return y - 1.0f;
  }
  if (k < 23) {
    t = tm_u2f(0x3f800000u - (0x1000000u >> k));   // 1 - 2^-k
    y = t - (e - x);
    y = tm_u2f((u32)((i32)tm_f2u(y) + (k << 23)));
  } else {
    t = tm_u2f((u32)((0x7f - k) << 23));         // 2^-k
    y = x - (e + t);
    y += 1.0f;
    y = tm_u2f((u32)((i32)tm_f2u(y) + (k << 23)));
  }
  return y;
}

// ---------------------------------------------------------------------------------------------- log1pf
// fdlibm's float log1pf as glibc 2.35 builds it: 1 + x = 2^k (1 + f), sqrt(2)/2 < 1 + f < sqrt(2), a correction
// term c for the rounding of 1 + x, log(1 + f) = f - s (f - R) with s = f / (2 + f) and R a polynomial in s^2.
TM_FN float tm_log1pf(float x) {
  const float ln2_hi = 6.9313812256e-01f, ln2_lo = 9.0580006145e-06f, two25 = 3.355443200e+07f,
              Lp1 = 6.6666668653e-01f, Lp2 = 4.0000000596e-01f, Lp3 = 2.8571429849e-01f, Lp4 = 2.2222198546e-01f,
              Lp5 = 1.8183572590e-01f, Lp6 = 1.5313838422e-01f, Lp7 = 1.4798198640e-01f;
  float hfsq, f = 0.0f, c = 0.0f, s, z, R, u;
  i32 k, hu = 0;
  const i32 hx = (i32)tm_f2u(x);
  const i32 ax = hx & 0x7fffffff;
  k = 1;
  if (hx < 0x3ed413d7) {                         // x < 0.41422
    if (ax >= 0x3f800000) {                      // x <= -1
      if (x == -1.0f) return -__builtin_inff();
      return __builtin_nanf("");
    }
    if (ax < 0x31000000) {                       // |x| < 2^-29
      if (ax < 0x24800000) return x;             // |x| < 2^-54
      return x - x * x * 0.5f;
    }
    if (hx > 0 || hx <= (i32)0xbe95f61fu) { k = 0; f = x; hu = 1; }     // -0.2929 < x < 0.41422
  } else if (hx >= 0x7f800000) {
    return x + x;
  }
  if (k != 0) {
    if (hx < 0x5a000000) {
      u = 1.0f + x;
      hu = (i32)tm_f2u(u);
      k = (hu >> 23) - 127;
      c = (k > 0) ? 1.0f - (u - x) : x - (u - 1.0f);      // the rounding of 1 + x
      c /= u;
    } else {
      u = x;
      hu = (i32)tm_f2u(u);
      k = (hu >> 23) - 127;
      c = 0.0f;
    }
    hu &= 0x007fffff;
    if (hu < 0x3504f7) {
      u = tm_u2f((u32)(hu | 0x3f800000));        // normalise u
    } else {
      k += 1;
      u = tm_u2f((u32)(hu | 0x3f000000));        // normalise u / 2
      hu = (0x00800000 - hu) >> 2;
    }
    f = u - 1.0f;
  }
  hfsq = 0.5f * f * f;
  if (hu == 0) {                                 // |f| < 2^-20
    if (f == 0.0f) {
      if (k == 0) return 0.0f;
      c += (float)k * ln2_lo;
      return (float)k * ln2_hi + c;
    }
    R = hfsq * (1.0f - 0.66666666666666666f * f);
    if (k == 0) return f - R;
    return (float)k * ln2_hi - ((R - ((float)k * ln2_lo + c)) - f);
  }
  s = f / (2.0f + f);
  z = s * s;
  R = z * (Lp1 + z * (Lp2 + z * (Lp3 + z * (Lp4 + z * (Lp5 + z * (Lp6 + z * Lp7))))));
  if (k == 0) return f - (hfsq - s * (hfsq + R));
  return (float)k * ln2_hi - ((hfsq - (s * (hfsq + R) + ((float)k * ln2_lo + c))) - f);
}

// ----------------------------------------------------------------------------------------------- tanhf
// fdlibm's float tanhf as glibc 2.35 builds it, on tm_expm1f: |x| < 1: -t / (t + 2) with t = expm1(-2|x|);
// 1 <= |x| < 22: 1 - 2 / (expm1(2|x|) + 2); beyond, +-1.
TM_FN float tm_tanhf(float x) {
  const i32 jx = (i32)tm_f2u(x), ix = jx & 0x7fffffff;
  float t, z;
  if (ix >= 0x7f800000) return jx >= 0 ? 1.0f / x + 1.0f : 1.0f / x - 1.0f;
  if (ix < 0x41b00000) {                         // |x| < 22
    if (ix == 0) return x;
    if (ix < 0x24000000) return x * (1.0f + x);  // |x| < 2^-55
    if (ix >= 0x3f800000) {
      t = tm_expm1f(2.0f * __builtin_fabsf(x));
      z = 1.0f - 2.0f / (t + 2.0f);
    } else {
      t = tm_expm1f(-2.0f * __builtin_fabsf(x));
      z = -t / (t + 2.0f);
    }
  } else {
    z = 1.0f - 1.0e-30f;
  }
  return jx >= 0 ? z : -z;
}

// --------------------------------------------------------------------------------------------- asinf / acosf
// glibc 2.35's float asin: fdlibm's structure with a single-precision polynomial asin x = x + x^3 P(x^2) (Cephes,
// S. L. Moshier; five coefficients) -- |x| < 1/2 directly; above, asin|x| = pi/2 - 2 asin(sqrt(t)), t = (1 - |x|)/2,
// through sqrt(t)'s head w (low 12 bits cleared) and a correction c = (t - w^2) / (sqrt t + w) below 0.975.
TM_FN float tm_asinf(float x) {
  const float pio2_hi = 1.57079637050628662109375f, pio2_lo = -4.37113900018624283e-8f,
              pio4_hi = 0.785398185253143310546875f, p0 = 1.666675248e-1f, p1 = 7.495297643e-2f,
              p2 = 4.547037598e-2f, p3 = 2.417951451e-2f, p4 = 4.216630880e-2f;
  const i32 hx = (i32)tm_f2u(x), ix = hx & 0x7fffffff;
  if (ix == 0x3f800000) return x * pio2_hi + x * pio2_lo;
  if (ix > 0x3f800000) return (x - x) / (x - x);
  if (ix < 0x3f000000) {                         // |x| < 1/2
    if (ix < 0x32000000) return x;               // |x| < 2^-27
    const float t = x * x, w = t * (p0 + t * (p1 + t * (p2 + t * (p3 + t * p4))));
    return x + x * w;
  }
  const float t = (1.0f - __builtin_fabsf(x)) * 0.5f;
  const float p = t * (p0 + t * (p1 + t * (p2 + t * (p3 + t * p4))));
  const float s = __builtin_sqrtf(t);
  float r;
  if (ix >= 0x3F79999A) {                        // |x| > 0.975
    r = pio2_hi - (2.0f * (s + s * p) - pio2_lo);
  } else {
    const float w = tm_u2f(tm_f2u(s) & 0xfffff000u), c = (t - w * w) / (s + w);
    const float pp = 2.0f * s * p - (pio2_lo - 2.0f * c), q = pio4_hi - 2.0f * w;
    r = pio4_hi - (pp - q);
  }
  return hx > 0 ? r : -r;
}

// fdlibm's float acos: |x| < 1/2 pi/2 - (x + x R(x^2)) with R a rational approximation (the double method's
// coefficients rounded to float); x < -1/2 pi - 2 (s + s R(z)) and x > 1/2 2 (w + (s R(z) + c)), z = (1 -+ x) / 2,
// s = sqrt z, w its head (low 12 bits cleared), c = (z - w^2) / (s + w).
TM_FN float tm_acosf(float x) {
  const float pi = tm_u2f(0x40490fdau), pio2_hi = tm_u2f(0x3fc90fdau), pio2_lo = tm_u2f(0x33a22168u),
              pS0 = (float)1.66666666666666657415e-01, pS1 = (float)-3.25565818622400915405e-01,
              pS2 = (float)2.01212532134862925881e-01, pS3 = (float)-4.00555345006794114027e-02,
              pS4 = (float)7.91534994289814532176e-04, pS5 = (float)3.47933107596021167570e-05,
              qS1 = (float)-2.40339491173441421878e+00, qS2 = (float)2.02094576023350569471e+00,
              qS3 = (float)-6.88283971605453293030e-01, qS4 = (float)7.70381505559019352791e-02;
  const i32 hx = (i32)tm_f2u(x), ix = hx & 0x7fffffff;
  if (ix == 0x3f800000) return hx > 0 ? 0.0f : pi + 2.0f * pio2_lo;
  if (ix > 0x3f800000) return (x - x) / (x - x);
  if (ix < 0x3f000000) {                         // |x| < 1/2
    if (ix <= 0x32800000) return pio2_hi + pio2_lo;
    const float z = x * x;
    const float p = z * (pS0 + z * (pS1 + z * (pS2 + z * (pS3 + z * (pS4 + z * pS5)))));
    const float q = 1.0f + z * (qS1 + z * (qS2 + z * (qS3 + z * qS4)));
    return pio2_hi - (x - (pio2_lo - x * (p / q)));
  }
  const float z = (hx < 0 ? 1.0f + x : 1.0f - x) * 0.5f;
  const float p = z * (pS0 + z * (pS1 + z * (pS2 + z * (pS3 + z * (pS4 + z * pS5)))));
  const float q = 1.0f + z * (qS1 + z * (qS2 + z * (qS3 + z * qS4)));
  const float s = __builtin_sqrtf(z), r = p / q;
  if (hx < 0) return pi - 2.0f * (s + (r * s - pio2_lo));
  const float df = tm_u2f(tm_f2u(s) & 0xfffff000u), c = (z - df * df) / (s + df);
  return 2.0f * (df + (r * s + c));
}

// --------------------------------------------------------------------------------------------- sinhf / coshf
// fdlibm's float sinhf / coshf as glibc 2.35 builds them, on tm_expm1f and tm_expf: below 22, sinh from
// t = expm1|x| as (2t - t^2 / (t + 1)) / 2 (|x| < 1) or (t + t / (t + 1)) / 2, cosh as 1 + t^2 / (2 (1 + t)) below
// ln2 / 2 and (e + 1 / e) / 2 with e = exp|x| above; to 88.72 (0x42b17180) exp|x| / 2; to the overflow threshold
// (0x42b2d4fc) w (w / 2) with w = exp(|x| / 2), so that the intermediate does not overflow.
TM_FN float tm_sinhf(float x) {
  const i32 jx = (i32)tm_f2u(x), ix = jx & 0x7fffffff;
  if (ix >= 0x7f800000) return x + x;
  const float h = jx < 0 ? -0.5f : 0.5f;
  if (ix < 0x41b00000) {                         // |x| < 22
    if (ix < 0x31800000) return x;               // |x| < 2^-28
    const float t = tm_expm1f(__builtin_fabsf(x));
    if (ix < 0x3f800000) return h * (2.0f * t - t * t / (t + 1.0f));
    return h * (t + t / (t + 1.0f));
  }
  if (ix < 0x42b17180) return h * tm_expf(__builtin_fabsf(x));
  if (ix <= 0x42b2d4fc) {
    const float w = tm_expf(0.5f * __builtin_fabsf(x)), t = h * w;
    return t * w;
  }
  return x * 1.0e37f;
}

TM_FN float tm_coshf(float x) {
  const i32 ix = (i32)tm_f2u(x) & 0x7fffffff;
  if (ix < 0x41b00000) {                         // |x| < 22
    if (ix < 0x3eb17218) {                       // |x| < ln2 / 2
      if (ix < 0x24000000) return 1.0f;          // |x| < 2^-55
      const float t = tm_expm1f(__builtin_fabsf(x)), w = 1.0f + t;
      return 1.0f + (t * t) / (w + w);
    }
    const float t = tm_expf(__builtin_fabsf(x));
    return 0.5f * t + 0.5f / t;
  }
  if (ix < 0x42b17180) return 0.5f * tm_expf(__builtin_fabsf(x));
  if (ix <= 0x42b2d4fc) {
    const float w = tm_expf(0.5f * __builtin_fabsf(x)), t = 0.5f * w;
    return t * w;
  }
  if (ix >= 0x7f800000) return x * x;
  return 1.0e30f * 1.0e30f;
}

// --------------------------------------------------------------------------------- atanhf / asinhf / acoshf
// fdlibm's float inverse hyperbolic functions as glibc 2.35 builds them.  atanh |x| = log1p(2|x| + 2|x||x| /
// (1 - |x|)) / 2 below 1/2 and log1p(2|x| / (1 - |x|)) / 2 above; asinh |x| = log1p(|x| + x^2 / (1 + sqrt(1 + x^2)))
// to 2, log(2|x| + 1 / (sqrt(x^2 + 1) + |x|)) to 2^14, log|x| + ln2 beyond; acosh x = log1p(t + sqrt(2t + t^2))
// with t = x - 1 to 2, log(2x - 1 / (x + sqrt(x^2 - 1))) to 2^28, log x + ln2 beyond.
TM_FN float tm_atanhf(float x) {
  const float xa = __builtin_fabsf(x);
  float t;
  if (xa < 0.5f) {
    if (xa < 0x1.0p-28f) return x;
    t = xa + xa;
    t = 0.5f * tm_log1pf(t + t * xa / (1.0f - xa));
  } else if (xa < 1.0f) {
    t = 0.5f * tm_log1pf((xa + xa) / (1.0f - xa));
  } else if (xa > 1.0f) {
    return (x - x) / (x - x);
  } else if (xa == 1.0f) {
    return x / 0.0f;
  } else {
    return x + x;                                // NaN
  }
  return __builtin_copysignf(t, x);
}

TM_FN float tm_asinhf(float x) {
  const float ln2 = 6.9314718246e-01f;
  const i32 ix = (i32)tm_f2u(x) & 0x7fffffff;
  float w;
  if (ix < 0x38000000) return x;                 // |x| < 2^-14
  if (ix > 0x47000000) {                         // |x| > 2^14
    if (ix >= 0x7f800000) return x + x;
    w = tm_logf(__builtin_fabsf(x)) + ln2;
  } else {
    const float xa = __builtin_fabsf(x);
    if (ix > 0x40000000) {                       // 2 < |x| <= 2^14
      w = tm_logf(2.0f * xa + 1.0f / (__builtin_sqrtf(xa * xa + 1.0f) + xa));
    } else {
      const float t = xa * xa;
      w = tm_log1pf(xa + t / (1.0f + __builtin_sqrtf(1.0f + t)));
    }
  }
  return __builtin_copysignf(w, x);
}

TM_FN float tm_acoshf(float x) {
  const float ln2 = 6.9314718246e-01f;
  const i32 hx = (i32)tm_f2u(x);
  if (hx < 0x3f800000) return (x - x) / (x - x);                 // x < 1 (negative x included)
  if (hx >= 0x4d800000) {                                        // x >= 2^28
    if (hx >= 0x7f800000) return x + x;
    return tm_logf(x) + ln2;
  }
  if (hx == 0x3f800000) return 0.0f;
  if (hx > 0x40000000) {                                         // 2 < x < 2^28
    const float t = x * x;
    return tm_logf(2.0f * x - 1.0f / (x + __builtin_sqrtf(t - 1.0f)));
  }
  const float t = x - 1.0f;
  return tm_log1pf(t + __builtin_sqrtf(2.0f * t + t * t));
}

// ---------------------------------------------------------------------------------------------- erff / erfcf
// fdlibm's float erf / erfc (the double method with its coefficients rounded to float, Horner's order, float
// arithmetic, no contraction), on tm_expf in the tails.  The float coefficients are the double method's rounded
// to nearest, written here as the double values the float conversion started from.
struct TmErffTail { float R, S; };
TM_FN TmErffTail tm_erff_tail(float x, bool big) {    // x = |x|, big: |x| >= 1 / 0.35
  const float s = 1.0f / (x * x);
  TmErffTail o;
  if (!big) {
    const float ra0 = (float)-9.86494403484714822705e-03, ra1 = (float)-6.93858572707181764372e-01,
                ra2 = (float)-1.05586262253232909814e+01, ra3 = (float)-6.23753324503260060396e+01,
                ra4 = (float)-1.62396669462573470355e+02, ra5 = (float)-1.84605092906711035994e+02,
                ra6 = (float)-8.12874355063065934246e+01, ra7 = (float)-9.81432934416914548592e+00,
                sa1 = (float)1.96512716674392571292e+01, sa2 = (float)1.37657754143519042600e+02,
                sa3 = (float)4.34565877475229228821e+02, sa4 = (float)6.45387271733267880336e+02,
                sa5 = (float)4.29008140027567833386e+02, sa6 = (float)1.08635005541779435134e+02,
                sa7 = (float)6.57024977031928170135e+00, sa8 = (float)-6.04244152148580987438e-02;
    o.R = ra0 + s * (ra1 + s * (ra2 + s * (ra3 + s * (ra4 + s * (ra5 + s * (ra6 + s * ra7))))));
    o.S = 1.0f + s * (sa1 + s * (sa2 + s * (sa3 + s * (sa4 + s * (sa5 + s * (sa6 + s * (sa7 + s * sa8)))))));
  } else {
    const float rb0 = (float)-9.86494292470009928597e-03, rb1 = (float)-7.99283237680523006574e-01,
                rb2 = (float)-1.77579549177547519889e+01, rb3 = (float)-1.60636384855821916062e+02,
                rb4 = (float)-6.37566443368389627722e+02, rb5 = (float)-1.02509513161107724954e+03,
                rb6 = (float)-4.83519191608651397019e+02, sb1 = (float)3.03380607434824582924e+01,
                sb2 = (float)3.25792512996573918826e+02, sb3 = (float)1.53672958608443695994e+03,
                sb4 = (float)3.19985821950859553908e+03, sb5 = (float)2.55305040643316442583e+03,
                sb6 = (float)4.74528541206955367215e+02, sb7 = (float)-2.24409524465858183362e+01;
    o.R = rb0 + s * (rb1 + s * (rb2 + s * (rb3 + s * (rb4 + s * (rb5 + s * rb6)))));
    o.S = 1.0f + s * (sb1 + s * (sb2 + s * (sb3 + s * (sb4 + s * (sb5 + s * (sb6 + s * sb7))))));
  }
  return o;
}
// |x| < 0.84375: y = P(x^2) / Q(x^2), erf = x + x y
TM_FN float tm_erff_small(float z) {
  const float pp0 = (float)1.28379167095512558561e-01, pp1 = (float)-3.25042107247001499370e-01,
              pp2 = (float)-2.84817495755985104766e-02, pp3 = (float)-5.77027029648944159157e-03,
              pp4 = (float)-2.37630166566501626084e-05, qq1 = (float)3.97917223959155352819e-01,
              qq2 = (float)6.50222499887672944485e-02, qq3 = (float)5.08130628187576562776e-03,
              qq4 = (float)1.32494738004321644526e-04, qq5 = (float)-3.96022827877536812320e-06;
  const float r = pp0 + z * (pp1 + z * (pp2 + z * (pp3 + z * pp4)));
  const float s = 1.0f + z * (qq1 + z * (qq2 + z * (qq3 + z * (qq4 + z * qq5))));
  return r / s;
}
// 0.84375 <= |x| < 1.25: P(s) / Q(s), s = |x| - 1
TM_FN float tm_erff_mid(float s) {
  const float pa0 = (float)-2.36211856075265944077e-03, pa1 = (float)4.14856118683748331666e-01,
              pa2 = (float)-3.72207876035701323847e-01, pa3 = (float)3.18346619901161753674e-01,
              pa4 = (float)-1.10894694282396677476e-01, pa5 = (float)3.54783043256182359371e-02,
              pa6 = (float)-2.16637559486879084300e-03, qa1 = (float)1.06420880400844228286e-01,
              qa2 = (float)5.40397917702171048937e-01, qa3 = (float)7.18286544141962662868e-02,
              qa4 = (float)1.26171219808761642112e-01, qa5 = (float)1.36370839120290507362e-02,
              qa6 = (float)1.19844998467991074170e-02;
  const float P = pa0 + s * (pa1 + s * (pa2 + s * (pa3 + s * (pa4 + s * (pa5 + s * pa6)))));
  const float Q = 1.0f + s * (qa1 + s * (qa2 + s * (qa3 + s * (qa4 + s * (qa5 + s * qa6)))));
  return P / Q;
}
// exp(-z^2 - 0.5625) exp((z - x)(z + x) + R / S) for x = |x|, z = x with its low `mask` bits cleared
TM_FN float tm_erff_exp(float x, u32 mask, float R, float S) {
  const float z = tm_u2f(tm_f2u(x) & mask);
  return tm_expf(-z * z - 0.5625f) * tm_expf((z - x) * (z + x) + R / S);
}

TM_FN float tm_erff(float x) {
  const float erx = (float)8.45062911510467529297e-01, efx = (float)1.28379167095512586316e-01;
  const i32 hx = (i32)tm_f2u(x), ix = hx & 0x7fffffff;
  if (ix >= 0x7f800000) return (float)(1 - (i32)(((u32)hx >> 31) << 1)) + 1.0f / x;
  if (ix < 0x3f580000) {                         // |x| < 0.84375
    if (ix < 0x31800000) {                       // |x| < 2^-28
      if (ix < 0x04000000) return 0.0625f * (16.0f * x + (16.0f * efx) * x);
      return x + efx * x;
    }
    return x + x * tm_erff_small(x * x);
  }
  if (ix < 0x3fa00000) {                         // |x| < 1.25
    const float q = tm_erff_mid(__builtin_fabsf(x) - 1.0f);
    return hx >= 0 ? erx + q : -erx - q;
  }
  if (ix >= 0x40c00000) return hx >= 0 ? 1.0f - 1.0e-30f : 1.0e-30f - 1.0f;   // |x| >= 6
  const float xa = __builtin_fabsf(x);
  const TmErffTail t = tm_erff_tail(xa, ix >= 0x4036DB6E);
  const float r = tm_erff_exp(xa, 0xfffff000u, t.R, t.S);
  return hx >= 0 ? 1.0f - r / xa : r / xa - 1.0f;
}

TM_FN float tm_erfcf(float x) {
  const float erx = (float)8.45062911510467529297e-01;
  const i32 hx = (i32)tm_f2u(x), ix = hx & 0x7fffffff;
  if (ix >= 0x7f800000) return (float)(((u32)hx >> 31) << 1) + 1.0f / x;
  if (ix < 0x3f580000) {                         // |x| < 0.84375
    if (ix < 0x32800000) return 1.0f - x;        // |x| < 2^-26
    const float y = tm_erff_small(x * x);
    if (hx < 0x3e800000) return 1.0f - (x + x * y);               // x < 1/4
    float r = x * y;
    r += (x - 0.5f);
    return 0.5f - r;
  }
  if (ix < 0x3fa00000) {                         // |x| < 1.25
    const float q = tm_erff_mid(__builtin_fabsf(x) - 1.0f);
    if (hx >= 0) return (1.0f - erx) - q;
    return 1.0f + (erx + q);
  }
  if (ix < 0x41e00000) {                         // |x| < 28
    const float xa = __builtin_fabsf(x);
    const bool big = ix >= 0x4036DB6D;
    if (big && hx < 0 && ix >= 0x40c00000) return 2.0f - 1.0e-30f;   // x < -6
    const TmErffTail t = tm_erff_tail(xa, big);
    const float r = tm_erff_exp(xa, 0xffffe000u, t.R, t.S);
    return hx > 0 ? r / xa : 2.0f - r / xa;
  }
  return hx > 0 ? 1.0e-30f * 1.0e-30f : 2.0f - 1.0e-30f;
}

// ---------------------------------------------------------------------------------------------- logistic
// lax.logistic as the reference's CPU target computes it (op_table.py:243-247): 1 / (1 + expf(-x)), IEEE.
TM_FN float tm_logisticf(float x) { return 1.0f / (1.0f + tm_expf(-x)); }

// ------------------------------------------------------------------------------------------------ lgammaf
// fdlibm's float lgamma as glibc 2.35 builds it.  x > 0: below 2 a rational or polynomial approximation about 1,
// tc (the minimum, 1.4616...) or 2 in y = x - 1 / x - tc / 2 - x (after -log x below 0.9); in [2, 8) the rational
// in the fractional part plus log of the product (y + 2)..(y + i - 1); to 2^26 Stirling's series; beyond
// x (log x - 1).  The float file's tf is the double tf truncated (0xbdf8cdcd) and its tt the tail of that float.
// x < 0: log(pi / |x sin(pi x)|) - lgamma(-x), sin(pi x) from glibc's sinf / cosf after reduction mod 2 -- except
// on (-15, -2), where glibc has its own (LGPL) lgamma_negf: there the device's math library is used.
TM_FN float tm_lgammaf_pos(float x) {                 // x > 0, finite, at least 2^-30
  const float a0 = 7.72156649015328655494e-02, a1 = 3.22467033424113591611e-01, a2 = 6.73523010531292681824e-02,
      a3 = 2.05808084325167332806e-02, a4 = 7.38555086081402883957e-03, a5 = 2.89051383673415629091e-03,
      a6 = 1.19270763183362067845e-03, a7 = 5.10069792153511336608e-04, a8 = 2.20862790713908385557e-04,
      a9 = 1.08011567247583939954e-04, a10 = 2.52144565451257326939e-05, a11 = 4.48640949618915160150e-05;
  const float tc = 1.46163214496836224576e+00, tf = -1.2148628384e-01f, tt = 6.6971006518e-09f;
  const float t0 = 4.83836122723810047042e-01, t1 = -1.47587722994593911752e-01, t2 = 6.46249402391333854778e-02,
      t3 = -3.27885410759859649565e-02, t4 = 1.79706750811820387126e-02, t5 = -1.03142241298341437450e-02,
      t6 = 6.10053870246291332635e-03, t7 = -3.68452016781138256760e-03, t8 = 2.25964780900612472250e-03,
      t9 = -1.40346469989232843813e-03, t10 = 8.81081882437654011382e-04, t11 = -5.38595305356740546715e-04,
      t12 = 3.15632070903625950361e-04, t13 = -3.12754168375120860518e-04, t14 = 3.35529192635519073543e-04;
  const float u0 = -7.72156649015328655494e-02, u1 = 6.32827064025093366517e-01, u2 = 1.45492250137234768737e+00,
      u3 = 9.77717527963372745603e-01, u4 = 2.28963728064692451092e-01, u5 = 1.33810918536787660377e-02,
      v1 = 2.45597793713041134822e+00, v2 = 2.12848976379893395361e+00, v3 = 7.69285150456672783825e-01,
      v4 = 1.04222645593369134254e-01, v5 = 3.21709242282423911810e-03;
  const float s0 = -7.72156649015328655494e-02, s1 = 2.14982415960608852501e-01, s2 = 3.25778796408930981787e-01,
      s3 = 1.46350472652464452805e-01, s4 = 2.66422703033638609560e-02, s5 = 1.84028451407337715652e-03,
      s6 = 3.19475326584100867617e-05, r1 = 1.39200533467621045958e+00, r2 = 7.21935547567138069525e-01,
      r3 = 1.71933865632803078993e-01, r4 = 1.86459191715652901344e-02, r5 = 7.77942496381893596434e-04,
      r6 = 7.32668430744625636189e-06;
  const float w0 = 4.18938533204672725052e-01, w1 = 8.33333333333329678849e-02, w2 = -2.77777777728775536470e-03,
      w3 = 7.93650558643019558500e-04, w4 = -5.95187557450339963135e-04, w5 = 8.36339918996282139126e-04,
      w6 = -1.63092934096575273989e-03;
  const i32 ix = (i32)tm_f2u(x);
  if (ix == 0x3f800000 || ix == 0x40000000) return 0.0f;
  if (ix < 0x40000000) {                              // x < 2
    float r, y;
    int i;
    if (ix <= 0x3f666666) {                           // x <= 0.9: lgamma(x + 1) - log x
      r = -tm_logf(x);
      if (ix >= 0x3f3b4a20) { y = 1.0f - x; i = 0; }
      else if (ix >= 0x3e6d3308) { y = x - (tc - 1.0f); i = 1; }
      else { y = x; i = 2; }
    } else {
      r = 0.0f;
      if (ix >= 0x3fdda618) { y = 2.0f - x; i = 0; }
      else if (ix >= 0x3f9da620) { y = x - tc; i = 1; }
      else { y = x - 1.0f; i = 2; }
    }
    if (i == 0) {
      const float z = y * y;
      const float p1 = a0 + z * (a2 + z * (a4 + z * (a6 + z * (a8 + z * a10))));
      const float p2 = z * (a1 + z * (a3 + z * (a5 + z * (a7 + z * (a9 + z * a11)))));
      const float p = y * p1 + p2;
      return r + (p - 0.5f * y);
    }
    if (i == 1) {
      const float z = y * y, w = z * y;
      const float p1 = t0 + w * (t3 + w * (t6 + w * (t9 + w * t12)));
      const float p2 = t1 + w * (t4 + w * (t7 + w * (t10 + w * t13)));
      const float p3 = t2 + w * (t5 + w * (t8 + w * (t11 + w * t14)));
      const float p = z * p1 - (tt - w * (p2 + y * p3));
      return r + (tf + p);
    }
    const float p1 = y * (u0 + y * (u1 + y * (u2 + y * (u3 + y * (u4 + y * u5)))));
    const float p2 = 1.0f + y * (v1 + y * (v2 + y * (v3 + y * (v4 + y * v5))));
    return r + (-0.5f * y + p1 / p2);
  }
  if (ix < 0x41000000) {                              // 2 <= x < 8
    const int i = (int)x;
    const float y = x - (float)i;
    const float p = y * (s0 + y * (s1 + y * (s2 + y * (s3 + y * (s4 + y * (s5 + y * s6))))));
    const float q = 1.0f + y * (r1 + y * (r2 + y * (r3 + y * (r4 + y * (r5 + y * r6)))));
    float r = 0.5f * y + p / q, z = 1.0f;
    if (i >= 7) z *= y + 6.0f;
    if (i >= 6) z *= y + 5.0f;
    if (i >= 5) z *= y + 4.0f;
    if (i >= 4) z *= y + 3.0f;
    if (i >= 3) { z *= y + 2.0f; r += tm_logf(z); }
    return r;
  }
  if (ix < 0x4c800000) {                              // 8 <= x < 2^26
    const float t = tm_logf(x), z = 1.0f / x, y = z * z;
    const float w = w0 + z * (w1 + y * (w2 + y * (w3 + y * (w4 + y * (w5 + y * w6)))));
    return (x - 0.5f) * (t - 1.0f) + w;
  }
  return x * (tm_logf(x) - 1.0f);
}
// sin(pi x) for x < 0 (as lgammaf needs it): |x| mod 2 by halving and floor, then sinf / cosf of pi times the
// remainder's distance to the nearest quarter; exact integers give +-0 by their parity.
TM_FN float tm_sin_pif(float x) {
  const float pi = 3.1415927410e+00f;
  const i32 ix = (i32)tm_f2u(x) & 0x7fffffff;
  if (ix < 0x3e800000) return tm_sinf(pi * x);
  float y = -x, z = __builtin_floorf(y);
  int n;
  if (z != y) {
    y *= 0.5f;
    y = 2.0f * (y - __builtin_floorf(y));
    n = (int)(y * 4.0f);
  } else if (ix >= 0x4b800000) {
    y = 0.0f;
    n = 0;
  } else {
    if (ix < 0x4b000000) z = y + 8388608.0f;
    n = (int)(tm_f2u(z) & 1u);
    y = (float)n;
    n <<= 2;
  }
  switch (n) {
    case 0: y = tm_sinf(pi * y); break;
    case 1: case 2: y = tm_cosf(pi * (0.5f - y)); break;
    case 3: case 4: y = tm_sinf(pi * (1.0f - y)); break;
    case 5: case 6: y = -tm_cosf(pi * (y - 1.5f)); break;
    default: y = tm_sinf(pi * (y - 2.0f)); break;
  }
  return -y;
}
TM_FN float tm_lgammaf(float x) {
  const i32 hx = (i32)tm_f2u(x), ix = hx & 0x7fffffff;
  if (ix >= 0x7f800000) return x * x;
  if (ix == 0) return 1.0f / __builtin_fabsf(x);
  if (ix < 0x30800000) return -tm_logf(hx < 0 ? -x : x);      // |x| < 2^-30
  if (hx >= 0) return tm_lgammaf_pos(x);
  if (ix >= 0x4b000000) return __builtin_fabsf(x) / 0.0f;      // a negative integer
  if (ix > 0x40000000 && ix < 0x41700000) return lgammaf(x);   // (-15, -2): the device's math library
  const float t = tm_sin_pif(x);
  if (t == 0.0f) return 1.0f / __builtin_fabsf(t);
  return tm_logf(3.1415927410e+00f / __builtin_fabsf(t * x)) - tm_lgammaf_pos(-x);
}

// ------------------------------------------------------------------------------------------------ powf
// the powf of glibc 2.35 (ARM optimized-routines): x^y = 2^(y log2 x), log2 x in double from tm_log2f's table by a
// quintic, 2^t from tm_exp2f's table and cubic with the result's sign folded into the table index for negative x
// with odd integer y; special cases first (y zero / inf / NaN, x zero / inf / NaN, negative x, subnormal x).
TM_FN int tm_powf_checkint(u32 iy) {              // 0: not an integer, 1: odd, 2: even
  const int e = (int)(iy >> 23 & 0xffu);
  if (e < 0x7f) return 0;
  if (e > 0x7f + 23) return 2;
  if (iy & ((1u << (0x7f + 23 - e)) - 1u)) return 0;
  if (iy & (1u << (0x7f + 23 - e))) return 1;
  return 2;
}
TM_FN bool tm_zeroinfnanf(u32 ix) { return 2u * ix - 1u >= 2u * 0x7f800000u - 1u; }
TM_FN bool tm_issnanf(u32 ix) { return (ix & 0x7fc00000u) == 0x7f800000u && (ix & 0x7fffffu) != 0u; }
TM_FN float tm_powf(float x, float y) {
  const double T[16][2] = {
      {0x1.661ec79f8f3bep+0, -0x1.efec65b963019p-2}, {0x1.571ed4aaf883dp+0, -0x1.b0b6832d4fca4p-2},
      {0x1.49539f0f010b0p+0, -0x1.7418b0a1fb77bp-2}, {0x1.3c995b0b80385p+0, -0x1.39de91a6dcf7bp-2},
      {0x1.30d190c8864a5p+0, -0x1.01d9bf3f2b631p-2}, {0x1.25e227b0b8ea0p+0, -0x1.97c1d1b3b7af0p-3},
      {0x1.1bb4a4a1a343fp+0, -0x1.2f9e393af3c9fp-3}, {0x1.12358f08ae5bap+0, -0x1.960cbbf788d5cp-4},
      {0x1.0953f419900a7p+0, -0x1.a6f9db6475fcep-5}, {0x1.0000000000000p+0, 0x0.0p+0},
      {0x1.e608cfd9a47acp-1, 0x1.338ca9f24f53dp-4}, {0x1.ca4b31f026aa0p-1, 0x1.476a9543891bap-3},
      {0x1.b2036576afce6p-1, 0x1.e840b4ac4e4d2p-3}, {0x1.9c2d163a1aa2dp-1, 0x1.40645f0c6651cp-2},
      {0x1.886e6037841edp-1, 0x1.88e9c2c1b9ff8p-2}, {0x1.767dcf5534862p-1, 0x1.ce0a44eb17bccp-2}};
  const double A0 = 0x1.27616c9496e0bp-2, A1 = -0x1.71969a075c67ap-2, A2 = 0x1.ec70a6ca7baddp-2,
               A3 = -0x1.7154748bef6c8p-1, A4 = 0x1.71547652ab82bp0;
  const double SHIFT = 0x1.8p+52 / 32, C0 = 0x1.c6af84b912394p-5, C1 = 0x1.ebfce50fac4f3p-3,
               C2 = 0x1.62e42ff0c52d6p-1;
  const u64 SIGN_BIAS = 1ull << (5 + 11);
  u64 sign_bias = 0;
  u32 ix = tm_f2u(x);
  const u32 iy = tm_f2u(y);
  if (ix - 0x00800000u >= 0x7f800000u - 0x00800000u || tm_zeroinfnanf(iy)) {
    if (tm_zeroinfnanf(iy)) {
      if (2u * iy == 0u) return tm_issnanf(ix) ? x + y : 1.0f;
      if (ix == 0x3f800000u) return tm_issnanf(iy) ? x + y : 1.0f;
      if (2u * ix > 2u * 0x7f800000u || 2u * iy > 2u * 0x7f800000u) return x + y;
      if (2u * ix == 2u * 0x3f800000u) return 1.0f;
      if ((2u * ix < 2u * 0x3f800000u) == !(iy & 0x80000000u)) return 0.0f;
      return y * y;
    }
    if (tm_zeroinfnanf(ix)) {
      float x2 = x * x;
      if ((ix & 0x80000000u) && tm_powf_checkint(iy) == 1) x2 = -x2;
      return (iy & 0x80000000u) ? 1.0f / x2 : x2;
    }
    if (ix & 0x80000000u) {                      // finite x < 0
      const int yint = tm_powf_checkint(iy);
      if (yint == 0) return __builtin_nanf("");
      if (yint == 1) sign_bias = SIGN_BIAS;
      ix &= 0x7fffffffu;
    }
    if (ix < 0x00800000u) {                      // subnormal x: normalise
      ix = tm_f2u(x * 0x1p23f);
      ix &= 0x7fffffffu;
      ix -= 23u << 23;
    }
  }
  // log2 x
  const u32 tmp = ix - 0x3f330000u;
  const int i = (int)((tmp >> 19) % 16u);
  const u32 top = tmp & 0xff800000u;
  const u32 iz = ix - top;
  const int k = (i32)top >> 23;
  const double z = (double)tm_u2f(iz);
  const double r = __builtin_fma(z, T[i][0], -1.0);
  const double y0 = T[i][1] + (double)k;
  const double r2 = r * r;
  double yy = __builtin_fma(A0, r, A1);
  const double p = __builtin_fma(A2, r, A3);
  const double r4 = r2 * r2;
  double q = __builtin_fma(A4, r, y0);
  q = __builtin_fma(p, r2, q);
  yy = __builtin_fma(yy, r4, q);
  const double ylogx = (double)y * yy;
  if (((tm_d2u(ylogx) >> 47) & 0xffffu) >= (tm_d2u(126.0) >> 47)) {
    if (ylogx > 0x1.fffffffd1d571p+6) return sign_bias ? -__builtin_inff() : __builtin_inff();
    if (ylogx <= -150.0) return sign_bias ? -0.0f : 0.0f;
  }
  // 2^ylogx
  double kd = ylogx + SHIFT;
  const u64 ki = tm_d2u(kd);
  kd -= SHIFT;
  const double rr = ylogx - kd;
  const u64 TT[32] = {
      0x3ff0000000000000ull, 0x3fefd9b0d3158574ull, 0x3fefb5586cf9890full, 0x3fef9301d0125b51ull,
      0x3fef72b83c7d517bull, 0x3fef54873168b9aaull, 0x3fef387a6e756238ull, 0x3fef1e9df51fdee1ull,
      0x3fef06fe0a31b715ull, 0x3feef1a7373aa9cbull, 0x3feedea64c123422ull, 0x3feece086061892dull,
      0x3feebfdad5362a27ull, 0x3feeb42b569d4f82ull, 0x3feeab07dd485429ull, 0x3feea47eb03a5585ull,
      0x3feea09e667f3bcdull, 0x3fee9f75e8ec5f74ull, 0x3feea11473eb0187ull, 0x3feea589994cce13ull,
      0x3feeace5422aa0dbull, 0x3feeb737b0cdc5e5ull, 0x3feec49182a3f090ull, 0x3feed503b23e255dull,
      0x3feee89f995ad3adull, 0x3feeff76f2fb5e47ull, 0x3fef199bdd85529cull, 0x3fef3720dcef9069ull,
      0x3fef5818dcfba487ull, 0x3fef7c97337b9b5full, 0x3fefa4afa2a490daull, 0x3fefd0765b6e4540ull};
  u64 t = TT[ki % 32u];
  t += (ki + sign_bias) << 47;
  const double s = tm_u2d(t);
  const double zz = __builtin_fma(C0, rr, C1);
  const double rr2 = rr * rr;
  double w = __builtin_fma(C2, rr, 1.0);
  w = __builtin_fma(zz, rr2, w);
  w = w * s;
  return (float)w;
}

// ================================================================================================ float64
// glibc 2.35's float64 exp / exp2 (ARM optimized-routines) and fdlibm's float64 expm1 / log1p / tanh / sinh / cosh
// / atanh / erf / erfc as glibc builds them, restated so the device returns glibc's bits.  x86-64 glibc selects an
// FMA build of exp at run time on FMA hosts (its polynomial and reduction contract to fused multiply-adds, its
// underflow path does not); exp2 and the fdlibm functions are generic builds without contraction.  Each is checked
// bitwise against glibc on random bit patterns, its working range and its branch boundaries
// (tests/native/libm_check.cc f64, tests/test_native_cpu.py) and on the device (tests/test_gpu_libm.py).

// 2^(k/128), k = 0 .. 127, as (T, H - k 2^45): H = 2^(k/128) rounded to double, T = (2^(k/128) - H) / H rounded
// to double, the pair's second word the bits of H with k / 128 taken off its exponent (so the bits of a scale
// 2^(i/128) are the entry's second word + i << 45).  Computed from that definition at 80 digits.
TM_FN void tm_exp_pair(u64 k, double& tail, u64& hbits) {
  const u64 E[256] = {
      0x0000000000000000ull, 0x3ff0000000000000ull, 0x3c9b3b4f1a88bf6eull, 0x3feff63da9fb3335ull,
      0xbc7160139cd8dc5dull, 0x3fefec9a3e778061ull, 0xbc905e7a108766d1ull, 0x3fefe315e86e7f85ull,
      0x3c8cd2523567f613ull, 0x3fefd9b0d3158574ull, 0xbc8bce8023f98efaull, 0x3fefd06b29ddf6deull,
      0x3c60f74e61e6c861ull, 0x3fefc74518759bc8ull, 0x3c90a3e45b33d399ull, 0x3fefbe3ecac6f383ull,
      0x3c979aa65d837b6dull, 0x3fefb5586cf9890full, 0x3c8eb51a92fdeffcull, 0x3fefac922b7247f7ull,
      0x3c3ebe3d702f9cd1ull, 0x3fefa3ec32d3d1a2ull, 0xbc6a033489906e0bull, 0x3fef9b66affed31bull,
      0xbc9556522a2fbd0eull, 0x3fef9301d0125b51ull, 0xbc5080ef8c4eea55ull, 0x3fef8abdc06c31ccull,
      0xbc91c923b9d5f416ull, 0x3fef829aaea92de0ull, 0x3c80d3e3e95c55afull, 0x3fef7a98c8a58e51ull,
      0xbc801b15eaa59348ull, 0x3fef72b83c7d517bull, 0xbc8f1ff055de323dull, 0x3fef6af9388c8deaull,
      0x3c8b898c3f1353bfull, 0x3fef635beb6fcb75ull, 0xbc96d99c7611eb26ull, 0x3fef5be084045cd4ull,
      0x3c9aecf73e3a2f60ull, 0x3fef54873168b9aaull, 0xbc8fe782cb86389dull, 0x3fef4d5022fcd91dull,
      0x3c8a6f4144a6c38dull, 0x3fef463b88628cd6ull, 0x3c807a05b0e4047dull, 0x3fef3f49917ddc96ull,
      0x3c968efde3a8a894ull, 0x3fef387a6e756238ull, 0x3c875e18f274487dull, 0x3fef31ce4fb2a63full,
      0x3c80472b981fe7f2ull, 0x3fef2b4565e27cddull, 0xbc96b87b3f71085eull, 0x3fef24dfe1f56381ull,
      0x3c82f7e16d09ab31ull, 0x3fef1e9df51fdee1ull, 0xbc3d219b1a6fbffaull, 0x3fef187fd0dad990ull,
      0x3c8b3782720c0ab4ull, 0x3fef1285a6e4030bull, 0x3c6e149289cecb8full, 0x3fef0cafa93e2f56ull,
      0x3c834d754db0abb6ull, 0x3fef06fe0a31b715ull, 0x3c864201e2ac744cull, 0x3fef0170fc4cd831ull,
      0x3c8fdd395dd3f84aull, 0x3feefc08b26416ffull, 0xbc86a3803b8e5b04ull, 0x3feef6c55f929ff1ull,
      0xbc924aedcc4b5068ull, 0x3feef1a7373aa9cbull, 0xbc9907f81b512d8eull, 0x3feeecae6d05d866ull,
      0xbc71d1e83e9436d2ull, 0x3feee7db34e59ff7ull, 0xbc991919b3ce1b15ull, 0x3feee32dc313a8e5ull,
      0x3c859f48a72a4c6dull, 0x3feedea64c123422ull, 0xbc9312607a28698aull, 0x3feeda4504ac801cull,
      0xbc58a78f4817895bull, 0x3feed60a21f72e2aull, 0xbc7c2c9b67499a1bull, 0x3feed1f5d950a897ull,
      0x3c4363ed60c2ac11ull, 0x3feece086061892dull, 0x3c9666093b0664efull, 0x3feeca41ed1d0057ull,
      0x3c6ecce1daa10379ull, 0x3feec6a2b5c13cd0ull, 0x3c93ff8e3f0f1230ull, 0x3feec32af0d7d3deull,
      0x3c7690cebb7aafb0ull, 0x3feebfdad5362a27ull, 0x3c931dbdeb54e077ull, 0x3feebcb299fddd0dull,
      0xbc8f94340071a38eull, 0x3feeb9b2769d2ca7ull, 0xbc87deccdc93a349ull, 0x3feeb6daa2cf6642ull,
      0xbc78dec6bd0f385full, 0x3feeb42b569d4f82ull, 0xbc861246ec7b5cf6ull, 0x3feeb1a4ca5d920full,
      0x3c93350518fdd78eull, 0x3feeaf4736b527daull, 0x3c7b98b72f8a9b05ull, 0x3feead12d497c7fdull,
      0x3c9063e1e21c5409ull, 0x3feeab07dd485429ull, 0x3c34c7855019c6eaull, 0x3feea9268a5946b7ull,
      0x3c9432e62b64c035ull, 0x3feea76f15ad2148ull, 0xbc8ce44a6199769full, 0x3feea5e1b976dc09ull,
      0xbc8c33c53bef4da8ull, 0x3feea47eb03a5585ull, 0xbc845378892be9aeull, 0x3feea34634ccc320ull,
      0xbc93cedd78565858ull, 0x3feea23882552225ull, 0x3c5710aa807e1964ull, 0x3feea155d44ca973ull,
      0xbc93b3efbf5e2228ull, 0x3feea09e667f3bcdull, 0xbc6a12ad8734b982ull, 0x3feea012750bdabfull,
      0xbc6367efb86da9eeull, 0x3fee9fb23c651a2full, 0xbc80dc3d54e08851ull, 0x3fee9f7df9519484ull,
      0xbc781f647e5a3ecfull, 0x3fee9f75e8ec5f74ull, 0xbc86ee4ac08b7db0ull, 0x3fee9f9a48a58174ull,
      0xbc8619321e55e68aull, 0x3fee9feb564267c9ull, 0x3c909ccb5e09d4d3ull, 0x3feea0694fde5d3full,
      0xbc7b32dcb94da51dull, 0x3feea11473eb0187ull, 0x3c94ecfd5467c06bull, 0x3feea1ed0130c132ull,
      0x3c65ebe1abd66c55ull, 0x3feea2f336cf4e62ull, 0xbc88a1c52fb3cf42ull, 0x3feea427543e1a12ull,
      0xbc9369b6f13b3734ull, 0x3feea589994cce13ull, 0xbc805e843a19ff1eull, 0x3feea71a4623c7adull,
      0xbc94d450d872576eull, 0x3feea8d99b4492edull, 0x3c90ad675b0e8a00ull, 0x3feeaac7d98a6699ull,
      0x3c8db72fc1f0eab4ull, 0x3feeace5422aa0dbull, 0xbc65b6609cc5e7ffull, 0x3feeaf3216b5448cull,
      0x3c7bf68359f35f44ull, 0x3feeb1ae99157736ull, 0xbc93091fa71e3d83ull, 0x3feeb45b0b91ffc6ull,
      0xbc5da9b88b6c1e29ull, 0x3feeb737b0cdc5e5ull, 0xbc6c23f97c90b959ull, 0x3feeba44cbc8520full,
      0xbc92434322f4f9aaull, 0x3feebd829fde4e50ull, 0xbc85ca6cd7668e4bull, 0x3feec0f170ca07baull,
      0x3c71affc2b91ce27ull, 0x3feec49182a3f090ull, 0x3c6dd235e10a73bbull, 0x3feec86319e32323ull,
      0xbc87c50422622263ull, 0x3feecc667b5de565ull, 0x3c8b1c86e3e231d5ull, 0x3feed09bec4a2d33ull,
      0xbc91bbd1d3bcbb15ull, 0x3feed503b23e255dull, 0x3c90cc319cee31d2ull, 0x3feed99e1330b358ull,
      0x3c8469846e735ab3ull, 0x3feede6b5579fdbfull, 0xbc82dfcd978e9db4ull, 0x3feee36bbfd3f37aull,
      0x3c8c1a7792cb3387ull, 0x3feee89f995ad3adull, 0xbc907b8f4ad1d9faull, 0x3feeee07298db666ull,
      0xbc55c3d956dcaebaull, 0x3feef3a2b84f15fbull, 0xbc90a40e3da6f640ull, 0x3feef9728de5593aull,
      0xbc68d6f438ad9334ull, 0x3feeff76f2fb5e47ull, 0xbc91eee26b588a35ull, 0x3fef05b030a1064aull,
      0x3c74ffd70a5fddcdull, 0x3fef0c1e904bc1d2ull, 0xbc91bdfbfa9298acull, 0x3fef12c25bd71e09ull,
      0x3c736eae30af0cb3ull, 0x3fef199bdd85529cull, 0x3c8ee3325c9ffd94ull, 0x3fef20ab5fffd07aull,
      0x3c84e08fd10959acull, 0x3fef27f12e57d14bull, 0x3c63cdaf384e1a67ull, 0x3fef2f6d9406e7b5ull,
      0x3c676b2c6c921968ull, 0x3fef3720dcef9069ull, 0xbc808a1883ccb5d2ull, 0x3fef3f0b555dc3faull,
      0xbc8fad5d3ffffa6full, 0x3fef472d4a07897cull, 0xbc900dae3875a949ull, 0x3fef4f87080d89f2ull,
      0x3c74a385a63d07a7ull, 0x3fef5818dcfba487ull, 0xbc82919e2040220full, 0x3fef60e316c98398ull,
      0x3c8e5a50d5c192acull, 0x3fef69e603db3285ull, 0x3c843a59ac016b4bull, 0x3fef7321f301b460ull,
      0xbc82d52107b43e1full, 0x3fef7c97337b9b5full, 0xbc892ab93b470dc9ull, 0x3fef864614f5a129ull,
      0x3c74b604603a88d3ull, 0x3fef902ee78b3ff6ull, 0x3c83c5ec519d7271ull, 0x3fef9a51fbc74c83ull,
      0xbc8ff7128fd391f0ull, 0x3fefa4afa2a490daull, 0xbc8dae98e223747dull, 0x3fefaf482d8e67f1ull,
      0x3c8ec3bc41aa2008ull, 0x3fefba1bee615a27ull, 0x3c842b94c3a9eb32ull, 0x3fefc52b376bba97ull,
      0x3c8a64a931d185eeull, 0x3fefd0765b6e4540ull, 0xbc8e37bae43be3edull, 0x3fefdbfdad9cbe14ull,
      0x3c77893b4d91cd9dull, 0x3fefe7c1819e90d8ull, 0x3c5305c14160cc89ull, 0x3feff3c22b8f71f1ull};
  tail = tm_u2d(E[2 * k]);
  hbits = E[2 * k + 1];
}

// the scaling of exp / exp2's result past the finite-double range of the table scale: s = the scale's bits (its
// exponent k / 128 may be out of range), q the polynomial part; overflow side: 2^1009 (s 2^-1009) (1 + q), the
// multiply-add fused as the FMA build fuses it (2^1 and 2^-1 for exp2's generic build, unfused); underflow side:
// 2^-1022 (s 2^1022) (1 + q), unfused, with the subnormal result's double rounding removed
TM_FN double tm_exp_scaled(double q, u64 s, u64 ki, bool fused, u64 up_adj, double up) {
  if ((ki & 0x80000000ull) == 0ull) {
    const double sc = tm_u2d(s - up_adj);
    return up * (fused ? __builtin_fma(sc, q, sc) : sc + sc * q);
  }
  const double sc = tm_u2d(s + (1022ull << 52));
  double y = sc + sc * q;
  if (y < 1.0) {
    double lo = sc - y + sc * q;
    const double hi = 1.0 + y;
    lo = 1.0 - hi + y + lo;
    y = (hi + lo) - 1.0;
    if (y == 0.0) y = 0.0;
  }
  return 0x1p-1022 * y;
}

// exp x = 2^(k/128) e^r, x = k ln2 / 128 + r, |r| <= ln2 / 256; e^r - 1 by a quartic in r; 2^(k/128) from the
// table (its tail folded into the polynomial).  |x| >= 512 and tiny |x| take the checks first.
TM_FN double tm_exp(double x) {
  const double InvLn2N = 0x1.71547652b82fep0 * 128, Shift = 0x1.8p52, NegLn2hiN = -0x1.62e42fefa0000p-8,
               NegLn2loN = -0x1.cf79abc9e3b3ap-47, C2 = 0x1.ffffffffffdbdp-2, C3 = 0x1.555555555543cp-3,
               C4 = 0x1.55555cf172b91p-5, C5 = 0x1.1111167a4d017p-7;
  u32 top = (u32)(tm_d2u(x) >> 52) & 0x7ffu;
  const u32 t_tiny = 0x3c9u, t_512 = 0x408u, t_1024 = 0x409u;     // the top 12 bits of 2^-54, 512, 1024
  if (top - t_tiny >= t_512 - t_tiny) {
    if ((i32)(top - t_tiny) < 0) return 1.0 + x;                    // |x| < 2^-54
    if (top >= t_1024) {
      if (tm_d2u(x) == 0xfff0000000000000ull) return 0.0;
      if (top >= 0x7ffu) return 1.0 + x;
      return (tm_d2u(x) >> 63) ? 0x1p-767 * 0x1p-767 : 0x1p769 * 0x1p769;
    }
    top = 0u;                                                        // 512 <= |x| < 1024: the scaled path
  }
  const double z = InvLn2N * x;
  double kd = z + Shift;
  const u64 ki = tm_d2u(kd);
  kd -= Shift;
  const double r = __builtin_fma(kd, NegLn2loN, __builtin_fma(kd, NegLn2hiN, x));
  double tail;
  u64 hb;
  tm_exp_pair(ki & 127ull, tail, hb);
  const u64 s = hb + (ki << 45);
  const double r2 = r * r;
  const double q = __builtin_fma(r2 * r2, __builtin_fma(r, C5, C4), __builtin_fma(r2, __builtin_fma(r, C3, C2), tail + r));
  if (top == 0u) return tm_exp_scaled(q, s, ki, true, 1009ull << 52, 0x1p1009);
  const double sc = tm_u2d(s);
  return __builtin_fma(sc, q, sc);
}

// exp2 x = 2^(k/128) 2^r, |r| <= 1/256, on the same table; a quintic in r, no fused operations (generic build).
TM_FN double tm_exp2(double x) {
  const double Shift = 0x1.8p52 / 128, C1 = 0x1.62e42fefa39efp-1, C2 = 0x1.ebfbdff82c424p-3,
               C3 = 0x1.c6b08d70cf4b5p-5, C4 = 0x1.3b2abd24650ccp-7, C5 = 0x1.5d7e09b4e3a84p-10;
  u32 top = (u32)(tm_d2u(x) >> 52) & 0x7ffu;
  const u32 t_tiny = 0x3c9u, t_512 = 0x408u, t_1024 = 0x409u;
  if (top - t_tiny >= t_512 - t_tiny) {
    if ((i32)(top - t_tiny) < 0) return 1.0 + x;
    if (top >= t_1024) {
      if (tm_d2u(x) == 0xfff0000000000000ull) return 0.0;
      if (top >= 0x7ffu) return 1.0 + x;
      if (!(tm_d2u(x) >> 63)) return 0x1p769 * 0x1p769;
      if (tm_d2u(x) >= tm_d2u(-1075.0)) return 0x1p-767 * 0x1p-767;
    }
    if (2ull * tm_d2u(x) > 2ull * tm_d2u(928.0)) top = 0u;         // the scaled path
  }
  double kd = x + Shift;
  const u64 ki = tm_d2u(kd);
  kd -= Shift;
  const double r = x - kd;
  double tail;
  u64 hb;
  tm_exp_pair(ki & 127ull, tail, hb);
  const u64 s = hb + (ki << 45);
  const double r2 = r * r;
  const double q = tail + r * C1 + r2 * (C2 + r * C3) + r2 * r2 * (C4 + r * C5);
  if (top == 0u) return tm_exp_scaled(q, s, ki, false, 1ull << 52, 2.0);
  const double sc = tm_u2d(s);
  return sc + sc * q;
}

// -------------------------------------------------------------------------------------------------- log (f64)
// glibc 2.35's log (ARM optimized-routines), as its FMA build computes it: x = 2^k z with z in [0x1.6p-1, 0x1.6p0)
// split into 128 subintervals by the top bits of z; log x = k ln2 + log c + log1p(r), r = z invc - 1 (one fma),
// |r| < 1/256, log1p(r) - r a quintic; the sum formed as hi + lo.  Within (1 - 2^-4, 1 + 0x1.09p-4) a degree-11
// polynomial in r = x - 1 with r^2 / 2 split exactly.  The table holds per subinterval invc = 1/c and
// logc = log c rounded, c near the subinterval's center chosen so that logc is a multiple of 2^-43 (k ln2hi + logc
// then rounds exactly) and log c - logc is below 2^-66: that rule, applied to the 2^30 doubles nearest 1 / center,
// leaves about 250 candidates per subinterval, and each entry here is the one candidate that agrees with glibc
// on 2.4e6 arguments of its subinterval at four exponents.
TM_FN double tm_log(double x) {
  const double A0 = -0x1.0000000000001p-1, A1 = 0x1.555555551305bp-2, A2 = -0x1.fffffffeb459p-3,
               A3 = 0x1.999b324f10111p-3, A4 = -0x1.55575e506c89fp-3;
  const double B0 = -0x1p-1, B1 = 0x1.5555555555577p-2, B2 = -0x1.ffffffffffdcbp-3, B3 = 0x1.999999995dd0cp-3,
               B4 = -0x1.55555556745a7p-3, B5 = 0x1.24924a344de3p-3, B6 = -0x1.fffffa4423d65p-4,
               B7 = 0x1.c7184282ad6cap-4, B8 = -0x1.999eb43b068ffp-4, B9 = 0x1.78182f7afd085p-4,
               B10 = -0x1.5521375d145cdp-4;
  const double Ln2hi = 0x1.62e42fefa3800p-1, Ln2lo = 0x1.ef35793c76730p-45;
  u64 ix = tm_d2u(x);
  const u64 lo1 = 0x3fee000000000000ull, hi1 = 0x3ff1090000000000ull;      // 1 - 2^-4, 1 + 0x1.09p-4
  if (ix - lo1 < hi1 - lo1) {
    if (ix == 0x3ff0000000000000ull) return 0.0;
    const double r = x - 1.0, r2 = r * r, r3 = r * r2;
    double p = __builtin_fma(r2, B9, __builtin_fma(r, B8, B7));
    p = __builtin_fma(r3, B10, p);
    double q = __builtin_fma(r2, B6, __builtin_fma(r, B5, B4));
    q = __builtin_fma(r3, p, q);
    double s = __builtin_fma(r2, B3, __builtin_fma(r, B2, B1));
    s = __builtin_fma(r3, q, s);
    const double w27 = r * 0x1p27, rhi = r + w27 - w27, rlo = r - rhi;
    const double w = rhi * rhi * B0;                 // exact: rhi has 26 bits
    const double hi = r + w;
    double lo = r - hi + w;
    lo = __builtin_fma(B0 * rlo, rhi + r, lo);
    double y = __builtin_fma(r3, s, lo);
    y += hi;
    return y;
  }
  const u32 top = (u32)(ix >> 48);
  if (top - 0x0010u >= 0x7ff0u - 0x0010u) {        // below 2^-1022, negative, infinite or NaN
    if (ix * 2 == 0) return -1.0 / 0.0;
    if (ix == 0x7ff0000000000000ull) return x;
    if ((top & 0x8000u) || (top & 0x7ff0u) == 0x7ff0u) return (x - x) / (x - x);
    ix = tm_d2u(x * 0x1p52) - (52ull << 52);       // subnormal: normalise
  }
  const double T[256] = {
      0x1.734f0c3e0de9fp+0, -0x1.7cc7f79e69p-2, 0x1.713786a2ce91fp+0, -0x1.76feec20dp-2,
      0x1.6f26008fab5ap+0, -0x1.713e31351ep-2, 0x1.6d1a61f138c7dp+0, -0x1.6b85b382878p-2,
      0x1.6b1490bc5b4d1p+0, -0x1.65d55908078p-2, 0x1.69147332f0cbap+0, -0x1.602d07618p-2,
      0x1.6719f18224223p+0, -0x1.5a8ca86909p-2, 0x1.6524f99a51ed9p+0, -0x1.54f4356035p-2,
      0x1.63356aa8f24c4p+0, -0x1.4f637c36b4p-2, 0x1.614b36b9ddc14p+0, -0x1.49da7fda85p-2,
      0x1.5f66452c65c4cp+0, -0x1.445923989a8p-2, 0x1.5d867b5912c4fp+0, -0x1.3edf439b0b8p-2,
      0x1.5babccb5b90dep+0, -0x1.396ce448f7p-2, 0x1.59d61f2d91a78p+0, -0x1.3401e17bdap-2,
      0x1.5805612465687p+0, -0x1.2e9e2ef468p-2, 0x1.56397cee76bd3p+0, -0x1.2941b3830ep-2,
      0x1.54725e2a77f93p+0, -0x1.23ec58cda88p-2, 0x1.52aff42064583p+0, -0x1.1e9e129279p-2,
      0x1.50f22dbb2bddfp+0, -0x1.1956d2b48f8p-2, 0x1.4f38f4734ded7p+0, -0x1.141679ab9f8p-2,
      0x1.4d843cfde284p+0, -0x1.0edd094ef98p-2, 0x1.4bd3ec078a3c8p+0, -0x1.09aa518db1p-2,
      0x1.4a27fc3e0258ap+0, -0x1.047e65263b8p-2, 0x1.4880524d48434p+0, -0x1.feb224586fp-3,
      0x1.46dce1b192d0bp+0, -0x1.f474a7517bp-3, 0x1.453d9d3391854p+0, -0x1.ea4443d103p-3,
      0x1.43a2744b4845ap+0, -0x1.e020d44e9bp-3, 0x1.420b54115f8fbp+0, -0x1.d60a22977fp-3,
      0x1.40782da3ef4b1p+0, -0x1.cc00104959p-3, 0x1.3ee8f5d57fe8fp+0, -0x1.c202956891p-3,
      0x1.3d5d9a00b4ce9p+0, -0x1.b81178d811p-3, 0x1.3bd60c010c12bp+0, -0x1.ae2c9ccd3dp-3,
      0x1.3a5242b75dab8p+0, -0x1.a45402e129p-3, 0x1.38d22cd9fd002p+0, -0x1.9a877681dfp-3,
      0x1.3755bc5847a1cp+0, -0x1.90c6d69483p-3, 0x1.35dce49ad36e2p+0, -0x1.87120a645cp-3,
      0x1.34679984dd44p+0, -0x1.7d68fb4143p-3, 0x1.32f5cceffcb24p+0, -0x1.73cb83c627p-3,
      0x1.3187775a10d49p+0, -0x1.6a39a9b376p-3, 0x1.301c8373e399p+0, -0x1.60b3154b7ap-3,
      0x1.2eb4ebb95f841p+0, -0x1.5737d76243p-3, 0x1.2d50a0219a9d1p+0, -0x1.4dc7b8fc23p-3,
      0x1.2bef9a8b7fd2ap+0, -0x1.4462c51d2p-3, 0x1.2a91c7a0c1babp+0, -0x1.3b08abc83p-3,
      0x1.293726014b53p+0, -0x1.31b996b49p-3, 0x1.27dfa5757a1f5p+0, -0x1.2875490a44p-3,
      0x1.268b39b1d3bbfp+0, -0x1.1f3b9f879ap-3, 0x1.2539d838ff5bdp+0, -0x1.160c8252cap-3,
      0x1.23eb7aac9083bp+0, -0x1.0ce7f57f72p-3, 0x1.22a012ba940b6p+0, -0x1.03cdc49feap-3,
      0x1.2157996cc4132p+0, -0x1.f57bdbc4b8p-4, 0x1.201201dd2fc9bp+0, -0x1.e370896404p-4,
      0x1.1ecf4494d480bp+0, -0x1.d17983ef94p-4, 0x1.1d8f5528f6569p+0, -0x1.bf9674ed8ap-4,
      0x1.1c52311577e7cp+0, -0x1.adc79202f6p-4, 0x1.1b17c74cb26e9p+0, -0x1.9c0c3e7288p-4,
      0x1.19e010c2c1ab6p+0, -0x1.8a646b372cp-4, 0x1.18ab07bb670bdp+0, -0x1.78d01b3acp-4,
      0x1.1778a25efbcb6p+0, -0x1.674f14538p-4, 0x1.1648d354c31dap+0, -0x1.55e0e6d878p-4,
      0x1.151b990275fddp+0, -0x1.4485cdea1ep-4, 0x1.13f0ea432d24cp+0, -0x1.333d94d6aap-4,
      0x1.12c8b7210f9dap+0, -0x1.22079f8c56p-4, 0x1.11a3028ecb531p+0, -0x1.10e4698622p-4,
      0x1.107fbda8434afp+0, -0x1.ffa6c6ad2p-5, 0x1.0f5ee0f4e6bb3p+0, -0x1.dda8d4a774p-5,
      0x1.0e4065d2a9fcep+0, -0x1.bbcece485p-5, 0x1.0d244632ca521p+0, -0x1.9a1894012cp-5,
      0x1.0c0a77ce2981ap+0, -0x1.788583302cp-5, 0x1.0af2f83c636d1p+0, -0x1.5715e67d68p-5,
      0x1.09ddb98a01339p+0, -0x1.35c8a49658p-5, 0x1.08cabaf52e7dfp+0, -0x1.149e364154p-5,
      0x1.07b9f2f4e28fbp+0, -0x1.e72c082eb8p-6, 0x1.06ab58c358f19p+0, -0x1.a55f152528p-6,
      0x1.059eea5ecf92cp+0, -0x1.63d62cf818p-6, 0x1.04949cdd12c9p+0, -0x1.228fb8caap-6,
      0x1.038c6c6f0ada9p+0, -0x1.c317b20f9p-7, 0x1.02865137932a9p+0, -0x1.419355daap-7,
      0x1.0182427ea7348p+0, -0x1.81203c2ecp-8, 0x1.008040614b195p+0, -0x1.004097924p-9,
      0x1.fe01ff726fa1ap-1, 0x1.feff3849p-9, 0x1.fa11cc261ea74p-1, 0x1.7dc41353dp-7,
      0x1.f6310b081992ep-1, 0x1.3cea3c4c28p-6, 0x1.f25f63ceeadcdp-1, 0x1.b9fc11489p-6,
      0x1.ee9c8039113e7p-1, 0x1.1b0d8ce11p-5, 0x1.eae8078cbb1abp-1, 0x1.58a5bd001cp-5,
      0x1.e741aa29d0c9bp-1, 0x1.95c8340d88p-5, 0x1.e3a91830a99b5p-1, 0x1.d276aef578p-5,
      0x1.e01e009609a56p-1, 0x1.07598e598cp-4, 0x1.dca01e577bb98p-1, 0x1.253f5e30d2p-4,
      0x1.d92f20b7c9103p-1, 0x1.42edd8b38p-4, 0x1.d5cac66fb5ccep-1, 0x1.606598757cp-4,
      0x1.d272caa5ede9dp-1, 0x1.7da76356ap-4, 0x1.cf26e3e6b2ccdp-1, 0x1.9ab434e1c6p-4,
      0x1.cbe6da2a77902p-1, 0x1.b78c7bb0d6p-4, 0x1.c8b266d37086dp-1, 0x1.d431332e72p-4,
      0x1.c5894bd5d5804p-1, 0x1.f0a3171de6p-4, 0x1.c26b533bb9f8cp-1, 0x1.067152b914p-3,
      0x1.bf583eeece73fp-1, 0x1.147858292bp-3, 0x1.bc4fd75db96c1p-1, 0x1.2266ecdca3p-3,
      0x1.b951e0c864a28p-1, 0x1.303d7a6c55p-3, 0x1.b65e2c5ef3e2cp-1, 0x1.3dfc33c331p-3,
      0x1.b374867c9888bp-1, 0x1.4ba366b7a8p-3, 0x1.b094b211d304ap-1, 0x1.5933928d1fp-3,
      0x1.adbe885f2ef7ep-1, 0x1.66acd2418fp-3, 0x1.aaf1d31603da2p-1, 0x1.740f8ec669p-3,
      0x1.a82e63fd358a7p-1, 0x1.815c0f51afp-3, 0x1.a5740ef09738bp-1, 0x1.8e92954f68p-3,
      0x1.a2c2a90ab4b27p-1, 0x1.9bb3602f84p-3, 0x1.a01a01393f2d1p-1, 0x1.a8bed1c2cp-3,
      0x1.9d79f24db3c1bp-1, 0x1.b5b515c01dp-3, 0x1.9ae2505c7b19p-1, 0x1.c2967ccbccp-3,
      0x1.9852ef297ce2fp-1, 0x1.cf635d5486p-3, 0x1.95cbaeea44b75p-1, 0x1.dc1bd3446cp-3,
      0x1.934c69de74838p-1, 0x1.e8c01b8cfep-3, 0x1.90d4f2f6752e6p-1, 0x1.f5509c0179p-3,
      0x1.8e6528effd79dp-1, 0x1.00e6c121fb8p-2, 0x1.8bfce9fcc007cp-1, 0x1.071b80e93dp-2,
      0x1.899c0dabec30ep-1, 0x1.0d46b9e867p-2, 0x1.87427aa2317fbp-1, 0x1.13687334bdp-2,
      0x1.84f00acb39a08p-1, 0x1.1980d672348p-2, 0x1.82a49e8653e55p-1, 0x1.1f8ffe0cc8p-2,
      0x1.8060195f4026p-1, 0x1.2595fd76368p-2, 0x1.7e22563e0a329p-1, 0x1.2b9300914a8p-2,
      0x1.7beb377dcb5adp-1, 0x1.3187210436p-2, 0x1.79baa679725c2p-1, 0x1.377266dec18p-2,
      0x1.77907f2170657p-1, 0x1.3d54ffbaf3p-2, 0x1.756cadbd6130cp-1, 0x1.432eee32fep-2
};
  const u64 tmp = ix - 0x3fe6000000000000ull;
  const int i = (int)((tmp >> 45) & 127u);
  const double kd = (double)((i64)tmp >> 52);
  const double z = tm_u2d(ix - (tmp & (0xfffull << 52)));
  const double r = __builtin_fma(z, T[2 * i], -1.0);
  const double w = __builtin_fma(kd, Ln2hi, T[2 * i + 1]);
  const double hi = w + r;
  const double lo = __builtin_fma(kd, Ln2lo, w - hi + r);
  const double r2 = r * r;
  const double p = __builtin_fma(r2, __builtin_fma(r, A4, A3), __builtin_fma(r, A2, A1));
  return __builtin_fma(r * r2, p, __builtin_fma(r2, A0, lo)) + hi;
}

// ------------------------------------------------------------------------------------------------- log2 (f64)
// glibc 2.35's log2 (ARM optimized-routines), as its generic build computes it (x86-64 glibc has no FMA variant of
// it): x = 2^k z, z in [0x1.6p-1, 0x1.6p0) split into 64 subintervals; log2 x = k + log2 c + log2(1 + r) with
// r = (z - chi - clo) invc (chi + clo = c = 1/invc); r / ln2 from r split at 32 bits times a two-part 1/ln2, plus
// r^2 times a quintic.  Within (1 - 0x1.5b51p-5, 1 + 0x1.6ab2p-5) a polynomial in r = x - 1 of degree 11.  The
// table: per subinterval invc, logc = log2 c rounded (a multiple of 2^-42, so k + logc rounds exactly, within
// 2^-62 of log2 c), chi, clo; found as tm_log's table (candidates among the 2^34 doubles nearest 1 / center by that
// rule, about 32,000 per subinterval, each entry the one that agrees with glibc on 2.4e6 arguments).
TM_FN double tm_log2(double x) {
  const double A0 = -0x1.71547652b8339p-1, A1 = 0x1.ec709dc3a04bep-2, A2 = -0x1.7154764702ffbp-2,
               A3 = 0x1.2776c50034c48p-2, A4 = -0x1.ec7b328ea92bcp-3, A5 = 0x1.a6225e117f92ep-3;
  const double B0 = -0x1.71547652b82fep-1, B1 = 0x1.ec709dc3a03f7p-2, B2 = -0x1.71547652b7c3fp-2,
               B3 = 0x1.2776c50f05be4p-2, B4 = -0x1.ec709dd768fe5p-3, B5 = 0x1.a61761ec4e736p-3,
               B6 = -0x1.7153fbc64a79bp-3, B7 = 0x1.484d154f01b4ap-3, B8 = -0x1.289e4a72c383cp-3,
               B9 = 0x1.0b32f285aee66p-3;
  const double InvLn2hi = 0x1.7154765200000p+0, InvLn2lo = 0x1.705fc2eefa200p-33;
  u64 ix = tm_d2u(x);
  const u64 lo1 = 0x3feea4af00000000ull, hi1 = 0x3ff0b55900000000ull;      // 1 - 0x1.5b51p-5, 1 + 0x1.6ab2p-5
  if (ix - lo1 < hi1 - lo1) {
    if (ix == 0x3ff0000000000000ull) return 0.0;
    const double r = x - 1.0;
    const double rhi = tm_u2d(tm_d2u(r) & 0xffffffff00000000ull), rlo = r - rhi;
    const double hi = rhi * InvLn2hi;
    double lo = rlo * InvLn2hi + r * InvLn2lo;
    const double r2 = r * r, r4 = r2 * r2;
    const double p = r2 * (B0 + r * B1);
    double y = hi + p;
    lo += hi - y + p;
    lo += r4 * (B2 + r * B3 + r2 * (B4 + r * B5) + r4 * (B6 + r * B7 + r2 * (B8 + r * B9)));
    y += lo;
    return y;
  }
  const u32 top = (u32)(ix >> 48);
  if (top - 0x0010u >= 0x7ff0u - 0x0010u) {        // below 2^-1022, negative, infinite or NaN
    if (ix * 2 == 0) return -1.0 / 0.0;
    if (ix == 0x7ff0000000000000ull) return x;
    if ((top & 0x8000u) || (top & 0x7ff0u) == 0x7ff0u) return (x - x) / (x - x);
    ix = tm_d2u(x * 0x1p52) - (52ull << 52);       // subnormal: normalise
  }
  const double T[256] = {                          // invc, logc, chi, clo
      0x1.724286bb1acf8p+0, -0x1.1095feecdbp-1, 0x1.6200012b90a8ep-1, 0x1.904ab0644b605p-55,
      0x1.6e1f766d2cca1p+0, -0x1.08494bd76dp-1, 0x1.66000045734a6p-1, 0x1.1ff9bea62f7a9p-57,
      0x1.6a13d0e30d48ap+0, -0x1.00143aee8f8p-1, 0x1.69fffc325f2c5p-1, 0x1.27ecfcb3c90bap-55,
      0x1.661ec32d06c85p+0, -0x1.efec5360b4p-2, 0x1.6e00038b95a04p-1, 0x1.8ff8856739326p-55,
      0x1.623fa951198f8p+0, -0x1.dfdd91ab7ep-2, 0x1.71fffe09994e3p-1, 0x1.afd40275f82b1p-55,
      0x1.5e75ba4cf026cp+0, -0x1.cffae0cc79p-2, 0x1.7600015590e1p-1, -0x1.2fd75b4238341p-56,
      0x1.5ac055a214fb8p+0, -0x1.c043811fdap-2, 0x1.7a00012655bd5p-1, 0x1.808e67c242b76p-56,
      0x1.571ed0f166e1ep+0, -0x1.b0b67323aep-2, 0x1.7e0003259e9a6p-1, -0x1.208e426f622b7p-57,
      0x1.53909590bf835p+0, -0x1.a152f5a2dbp-2, 0x1.81fffedb4b2d2p-1, -0x1.402461ea5c92fp-55,
      0x1.5014fed61adddp+0, -0x1.9217f5af86p-2, 0x1.860002dfafcc3p-1, 0x1.df7f4a2f29a1fp-57,
      0x1.4cab88e487bdp+0, -0x1.8304db0719p-2, 0x1.89ffff78c6b5p-1, -0x1.e0453094995fdp-55,
      0x1.49539b4334feep+0, -0x1.74189f9a9ep-2, 0x1.8e00039671566p-1, -0x1.a04f3bec77b45p-55,
      0x1.460cbdfafd569p+0, -0x1.6552bb5199p-2, 0x1.91fffe2bf1745p-1, -0x1.7fa34400e203cp-56,
      0x1.42d664ee4b953p+0, -0x1.56b23a29b1p-2, 0x1.95fffcc5c9fd1p-1, -0x1.6ff8005a0695dp-56,
      0x1.3fb01111dd8a6p+0, -0x1.483650f5fap-2, 0x1.9a0003bba4767p-1, 0x1.0f8c4c4ec7e03p-56,
      0x1.3c995b70c5836p+0, -0x1.39de937f6ap-2, 0x1.9dfffe7b92da5p-1, 0x1.e7fd9478c4602p-55,
      0x1.3991c4ab6fd4ap+0, -0x1.2baa1538d6p-2, 0x1.a1fffd72efdafp-1, -0x1.a0c554dcdae7ep-57,
      0x1.3698e0ce099b5p+0, -0x1.1d98340ca4p-2, 0x1.a5fffde04ff95p-1, 0x1.67da98ce9b26bp-55,
      0x1.33ae48213e7b2p+0, -0x1.0fa853a40ep-2, 0x1.a9fffca5e8d2bp-1, -0x1.284c9b54c13dep-55,
      0x1.30d191985bdb1p+0, -0x1.01d9c32e73p-2, 0x1.adfffddad03eap-1, 0x1.812c8ea602e3cp-58,
      0x1.2e025cab271d7p+0, -0x1.e857da2fa6p-3, 0x1.b1ffff10d3d4dp-1, -0x1.efaddad27789cp-55,
      0x1.2b404cf13cd82p+0, -0x1.cd3c8633d8p-3, 0x1.b5fffce21165ap-1, 0x1.3cb1719c61237p-58,
      0x1.288b02c7ccb5p+0, -0x1.b26034c14ap-3, 0x1.b9fffd950e674p-1, 0x1.3f7d94194cep-56,
      0x1.25e2263944de5p+0, -0x1.97c1c2f4fep-3, 0x1.be000139ca8afp-1, 0x1.50ac4215d9bcp-56,
      0x1.234563d8615b1p+0, -0x1.7d6023f8p-3, 0x1.c20005b46df99p-1, 0x1.beea653e9c1c9p-57,
      0x1.20b46e33eaf38p+0, -0x1.633a71a05ep-3, 0x1.c600040b9f7aep-1, -0x1.c079f274a70d6p-56,
      0x1.1e2eefdcda3ddp+0, -0x1.494f5e957p-3, 0x1.ca0006255fd8ap-1, -0x1.a0b4076e84c1fp-56,
      0x1.1bb4a580b393p+0, -0x1.2f9e424e0ap-3, 0x1.cdfffd94c095dp-1, 0x1.8f933f99ab5d7p-55,
      0x1.19453847f22p+0, -0x1.162595afdcp-3, 0x1.d1ffff975d6cfp-1, -0x1.82c08665fe1bep-58,
      0x1.16e06c0d5d73cp+0, -0x1.f9c9a75bd8p-4, 0x1.d5fffa2561c93p-1, -0x1.b04289bd295f3p-56,
      0x1.1485f47b7e4c2p+0, -0x1.c7b575bf9cp-4, 0x1.d9fff9d228b0cp-1, 0x1.70251340fa236p-55,
      0x1.12358ad0085d1p+0, -0x1.960c60ff48p-4, 0x1.de00065bc7e16p-1, -0x1.5011e16a4d80cp-56,
      0x1.0fef00f532227p+0, -0x1.64ce247b6p-4, 0x1.e200002f64791p-1, 0x1.9802f09ef62ep-55,
      0x1.0db2077d03a8fp+0, -0x1.33f78b2014p-4, 0x1.e600057d7a6d8p-1, -0x1.e0b75580cf7fap-56,
      0x1.0b7e6d65980d9p+0, -0x1.0387d1a42cp-4, 0x1.ea00027edc00cp-1, -0x1.c848309459811p-55,
      0x1.0953efe7b408dp+0, -0x1.a6f9208b5p-5, 0x1.ee0006cf5cb7cp-1, -0x1.f8027951576f4p-55,
      0x1.07325cac53b83p+0, -0x1.47a954f77p-5, 0x1.f2000782b7dccp-1, -0x1.f81d97274538fp-55,
      0x1.05197e40d1b5cp+0, -0x1.d23a8c50cp-6, 0x1.f6000260c450ap-1, -0x1.071002727ffdcp-59,
      0x1.03091c1208ea2p+0, -0x1.16a262978p-6, 0x1.f9fffe88cd533p-1, -0x1.81bdce1fda8bp-58,
      0x1.0101025b37e21p+0, -0x1.720f8d8e8p-8, 0x1.fdfffd50f8689p-1, 0x1.7f91acb918e6ep-55,
      0x1.fc07ef9caa76bp-1, 0x1.6fe53b15p-7, 0x1.0200004292367p+0, 0x1.b7ff365324681p-54,
      0x1.f4465d3f6f184p-1, 0x1.11ccce10f8p-5, 0x1.05fffe3e3d668p+0, 0x1.6fa08ddae957bp-55,
      0x1.ecc079f84107fp-1, 0x1.c4dfc8c8b8p-5, 0x1.0a0000a85a757p+0, -0x1.7e2de80d3fb91p-58,
      0x1.e573a99975ae8p-1, 0x1.3aa321e574p-4, 0x1.0e0001a5f3fccp+0, -0x1.1823305c5f014p-54,
      0x1.de5d6f0bd3de6p-1, 0x1.918a0d08b8p-4, 0x1.11ffff8afbaf5p+0, -0x1.bfabb6680bac2p-55,
      0x1.d77b681ff38b3p-1, 0x1.e72e9da044p-4, 0x1.15fffe54d91adp+0, -0x1.d7f121737e7efp-54,
      0x1.d0cb5724de943p-1, 0x1.1dcd2507f6p-3, 0x1.1a00011ac36e1p+0, 0x1.c000a0516f5ffp-54,
      0x1.ca4b2dc0e7563p-1, 0x1.476ab03deap-3, 0x1.1e00019c84248p+0, -0x1.082fbe4da5dap-54,
      0x1.c3f8ee8d6cb51p-1, 0x1.7074377e22p-3, 0x1.220000ffe5e6ep+0, -0x1.8fdd04c9cfb43p-55,
      0x1.bdd2b4f020c4cp-1, 0x1.98ede8ba94p-3, 0x1.26000269fd891p+0, 0x1.cfe2a7994d183p-55,
      0x1.b7d6c006015cap-1, 0x1.c0db86ad2ep-3, 0x1.2a00029a6e6dap+0, -0x1.00273715e8bc5p-56,
      0x1.b20366e2e338fp-1, 0x1.e840aafceep-3, 0x1.2dfffe0293e39p+0, 0x1.b7c39dab2a6f9p-54,
      0x1.ac57026295039p-1, 0x1.0790ab4678p-2, 0x1.31ffff7dcf082p+0, 0x1.df1336edc5254p-56,
      0x1.a6d01bc2731ddp-1, 0x1.1ac056801cp-2, 0x1.35ffff05a8b6p+0, -0x1.e03564ccd31ebp-54,
      0x1.a16d3bc3ff18bp-1, 0x1.2db11d4feep-2, 0x1.3a0002e0eaeccp+0, 0x1.5f0e74bd3a477p-56,
      0x1.9c2d14967feadp-1, 0x1.406464ec58p-2, 0x1.3e000043bb236p+0, 0x1.c7dcb149d8833p-54,
      0x1.970e4f47c9902p-1, 0x1.52dbe093afp-2, 0x1.4200002d187ffp+0, 0x1.e08afcf2d3d28p-56,
      0x1.920fb3982bcf2p-1, 0x1.651902050dp-2, 0x1.460000d387cb1p+0, 0x1.20837856599a6p-55,
      0x1.8d30187f759f1p-1, 0x1.771d2cdeafp-2, 0x1.4a00004569f89p+0, -0x1.9fa5c904fbcd2p-55,
      0x1.886e5ebb9f66dp-1, 0x1.88e9c857d9p-2, 0x1.4e000043543f3p+0, -0x1.81125ed175329p-56,
      0x1.83c97b658b994p-1, 0x1.9a80155e16p-2, 0x1.51fffcc027f0fp+0, 0x1.883d8847754dcp-54,
      0x1.7f405ffc61022p-1, 0x1.abe186ed3dp-2, 0x1.55ffffd87b36fp+0, -0x1.709e731d02807p-55,
      0x1.7ad22181415cap-1, 0x1.bd0f2aea0ep-2, 0x1.59ffff21df7bap+0, 0x1.7f79f68727b02p-55,
      0x1.767dcf99eff8cp-1, 0x1.ce0a43dbf4p-2, 0x1.5dfffebfc3481p+0, -0x1.180902e30e93ep-54
};
  const u64 tmp = ix - 0x3fe6000000000000ull;
  const int i = (int)((tmp >> 46) & 63u);
  const double kd = (double)((i64)tmp >> 52);
  const double z = tm_u2d(ix - (tmp & (0xfffull << 52)));
  const double r = (z - T[4 * i + 2] - T[4 * i + 3]) * T[4 * i];
  const double rhi = tm_u2d(tm_d2u(r) & 0xffffffff00000000ull), rlo = r - rhi;
  const double t1 = rhi * InvLn2hi, t2 = rlo * InvLn2hi + r * InvLn2lo;
  const double t3 = kd + T[4 * i + 1], hi = t3 + t1, lo = t3 - hi + t1 + t2;
  const double r2 = r * r, r4 = r2 * r2;
  const double p = A0 + r * A1 + r2 * (A2 + r * A3) + r4 * (A4 + r * A5);
  return lo + r2 * p + hi;
}

// -------------------------------------------------------------------------------------------------- pow (f64)
// glibc 2.35's pow (ARM optimized-routines), as its FMA build computes it: x^y = exp(y log x) with log x formed as
// hi + lo to about 68 bits and the product split as ehi + elo, then exp on tm_exp's table and polynomial with the
// tail folded in and the sign of a negative x with odd integer y carried in the scale's exponent bits.  log x:
// x = 2^k z, z in [0x1.69555p-1, 0x1.69555p0) split into 128 subintervals; invc = 1/c is j/128 or j/256 (so
// r = z invc - 1 is exact), logc + logctail = log c with logc a multiple of 2^-43 -- the table computed from that
// definition (c near each subinterval's center; log c at 113 bits).
TM_FN int tm_pow_checkint(u64 iy) {             // 0: not an integer, 1: odd, 2: even
  const int e = (int)((iy >> 52) & 0x7ffu);
  if (e < 0x3ff) return 0;
  if (e > 0x3ff + 52) return 2;
  if (iy & ((1ull << (0x3ff + 52 - e)) - 1ull)) return 0;
  if (iy & (1ull << (0x3ff + 52 - e))) return 1;
  return 2;
}
TM_FN bool tm_zeroinfnan(u64 i) { return 2ull * i - 1ull >= 2ull * 0x7ff0000000000000ull - 1ull; }
TM_FN bool tm_issnan(u64 i) { return ((i >> 51) & 0xfffu) == 0xffeu && (i & 0x7ffffffffffffull) != 0ull; }
TM_FN double tm_pow_log(u64 ix, double& tail) {
  const double A0 = -0x1p-1, A1 = 0x1.555555555556p-2 * -2, A2 = -0x1.0000000000006p-2 * -2,
               A3 = 0x1.999999959554ep-3 * 4, A4 = -0x1.555555529a47ap-3 * 4, A5 = 0x1.2495b9b4845e9p-3 * -8,
               A6 = -0x1.0002b8b263fc3p-3 * -8;
  const double Ln2hi = 0x1.62e42fefa3800p-1, Ln2lo = 0x1.ef35793c76730p-45;
  const double T[384] = {                          // invc, logc, logctail
      0x1.6ap+0, -0x1.62c82f2b9c8p-2, 0x1.ab4242837568p-48,
      0x1.68p+0, -0x1.5d1bdbf5808p-2, -0x1.ca508d8e0f72p-46,
      0x1.66p+0, -0x1.57677174558p-2, -0x1.362a4d5b6506dp-45,
      0x1.64p+0, -0x1.51aad872df8p-2, -0x1.684e49eb067d5p-49,
      0x1.62p+0, -0x1.4be5f957778p-2, -0x1.41b6993293eep-47,
      0x1.6p+0, -0x1.4618bc21c6p-2, 0x1.3d82f484c84ccp-46,
      0x1.5ep+0, -0x1.404308686a8p-2, 0x1.c42f3ed820b3ap-50,
      0x1.5cp+0, -0x1.3a64c556948p-2, 0x1.0b1c68651946p-45,
      0x1.5ap+0, -0x1.347dd9a988p-2, 0x1.5594dd4c58092p-45,
      0x1.58p+0, -0x1.2e8e2bae12p-2, 0x1.67b1e99b72bd8p-45,
      0x1.56p+0, -0x1.2895a13de88p-2, 0x1.5ca14b6cfb03fp-46,
      0x1.56p+0, -0x1.2895a13de88p-2, 0x1.5ca14b6cfb03fp-46,
      0x1.54p+0, -0x1.22941fbcf78p-2, -0x1.65a242853da76p-46,
      0x1.52p+0, -0x1.1c898c16998p-2, -0x1.fafbc68e75404p-46,
      0x1.5p+0, -0x1.1675cababa8p-2, 0x1.f1fc63382a8fp-46,
      0x1.4ep+0, -0x1.1058bf9ae48p-2, -0x1.6a8c4fd055a66p-45,
      0x1.4cp+0, -0x1.0a324e2739p-2, -0x1.c6bee7ef4030ep-47,
      0x1.4ap+0, -0x1.0402594b4dp-2, -0x1.036b89ef42d7fp-48,
      0x1.4ap+0, -0x1.0402594b4dp-2, -0x1.036b89ef42d7fp-48,
      0x1.48p+0, -0x1.fb9186d5e4p-3, 0x1.d572aab993c87p-47,
      0x1.46p+0, -0x1.ef0adcbdc6p-3, 0x1.b26b79c86af24p-45,
      0x1.44p+0, -0x1.e27076e2afp-3, -0x1.72f4f543fff1p-46,
      0x1.42p+0, -0x1.d5c216b4fcp-3, 0x1.1ba91bbca681bp-45,
      0x1.4p+0, -0x1.c8ff7c79aap-3, 0x1.7794f689f8434p-45,
      0x1.4p+0, -0x1.c8ff7c79aap-3, 0x1.7794f689f8434p-45,
      0x1.3ep+0, -0x1.bc286742d9p-3, 0x1.94eb0318bb78fp-46,
      0x1.3cp+0, -0x1.af3c94e80cp-3, 0x1.a4e633fcd9066p-52,
      0x1.3ap+0, -0x1.a23bc1fe2bp-3, -0x1.58c64dc46c1eap-45,
      0x1.3ap+0, -0x1.a23bc1fe2bp-3, -0x1.58c64dc46c1eap-45,
      0x1.38p+0, -0x1.9525a9cf45p-3, -0x1.ad1d904c1d4e3p-45,
      0x1.36p+0, -0x1.87fa06520dp-3, 0x1.bbdbf7fdbfa09p-45,
      0x1.34p+0, -0x1.7ab890210ep-3, 0x1.bdb9072534a58p-45,
      0x1.34p+0, -0x1.7ab890210ep-3, 0x1.bdb9072534a58p-45,
      0x1.32p+0, -0x1.6d60fe719dp-3, -0x1.0e46aa3b2e266p-46,
      0x1.3p+0, -0x1.5ff3070a79p-3, -0x1.e9e439f105039p-46,
      0x1.3p+0, -0x1.5ff3070a79p-3, -0x1.e9e439f105039p-46,
      0x1.2ep+0, -0x1.526e5e3a1bp-3, -0x1.0de8b90075b8fp-45,
      0x1.2cp+0, -0x1.44d2b6ccb8p-3, 0x1.70cc16135783cp-46,
      0x1.2cp+0, -0x1.44d2b6ccb8p-3, 0x1.70cc16135783cp-46,
      0x1.2ap+0, -0x1.371fc201e9p-3, 0x1.178864d27543ap-48,
      0x1.28p+0, -0x1.29552f81ffp-3, -0x1.48d301771c408p-45,
      0x1.26p+0, -0x1.1b72ad52f6p-3, -0x1.e80a41811a396p-45,
      0x1.26p+0, -0x1.1b72ad52f6p-3, -0x1.e80a41811a396p-45,
      0x1.24p+0, -0x1.0d77e7cd09p-3, 0x1.a699688e85bf4p-47,
      0x1.24p+0, -0x1.0d77e7cd09p-3, 0x1.a699688e85bf4p-47,
      0x1.22p+0, -0x1.fec9131dbep-4, -0x1.575545ca333f2p-45,
      0x1.2p+0, -0x1.e27076e2bp-4, 0x1.a342c2af0003cp-45,
      0x1.2p+0, -0x1.e27076e2bp-4, 0x1.a342c2af0003cp-45,
      0x1.1ep+0, -0x1.c5e548f5bcp-4, -0x1.d0c57585fbe06p-46,
      0x1.1cp+0, -0x1.a926d3a4aep-4, 0x1.53935e85baac8p-45,
      0x1.1cp+0, -0x1.a926d3a4aep-4, 0x1.53935e85baac8p-45,
      0x1.1ap+0, -0x1.8c345d631ap-4, 0x1.37c294d2f5668p-46,
      0x1.1ap+0, -0x1.8c345d631ap-4, 0x1.37c294d2f5668p-46,
      0x1.18p+0, -0x1.6f0d28ae56p-4, -0x1.69737c93373dap-45,
      0x1.16p+0, -0x1.51b073f062p-4, 0x1.f025b61c65e57p-46,
      0x1.16p+0, -0x1.51b073f062p-4, 0x1.f025b61c65e57p-46,
      0x1.14p+0, -0x1.341d7961bep-4, 0x1.c5edaccf913dfp-45,
      0x1.14p+0, -0x1.341d7961bep-4, 0x1.c5edaccf913dfp-45,
      0x1.12p+0, -0x1.16536eea38p-4, 0x1.47c5e768fa309p-46,
      0x1.1p+0, -0x1.f0a30c0118p-5, 0x1.d599e83368e91p-45,
      0x1.1p+0, -0x1.f0a30c0118p-5, 0x1.d599e83368e91p-45,
      0x1.0ep+0, -0x1.b42dd71198p-5, 0x1.c827ae5d6704cp-46,
      0x1.0ep+0, -0x1.b42dd71198p-5, 0x1.c827ae5d6704cp-46,
      0x1.0cp+0, -0x1.77458f632cp-5, -0x1.cfc4634f2a1eep-45,
      0x1.0cp+0, -0x1.77458f632cp-5, -0x1.cfc4634f2a1eep-45,
      0x1.0ap+0, -0x1.39e87b9fecp-5, 0x1.502b7f526feaap-48,
      0x1.0ap+0, -0x1.39e87b9fecp-5, 0x1.502b7f526feaap-48,
      0x1.08p+0, -0x1.f829b0e78p-6, -0x1.980267c7e09e4p-45,
      0x1.08p+0, -0x1.f829b0e78p-6, -0x1.980267c7e09e4p-45,
      0x1.06p+0, -0x1.7b91b07d58p-6, -0x1.88d5493faa639p-45,
      0x1.04p+0, -0x1.fc0a8b0fcp-7, -0x1.f1e7cf6d3a69cp-50,
      0x1.04p+0, -0x1.fc0a8b0fcp-7, -0x1.f1e7cf6d3a69cp-50,
      0x1.02p+0, -0x1.fe02a6b1p-8, -0x1.9e23f0dda40e4p-46,
      0x1.02p+0, -0x1.fe02a6b1p-8, -0x1.9e23f0dda40e4p-46,
      0x1p+0, -0x0p+0, 0x0p+0,
      0x1p+0, -0x0p+0, 0x0p+0,
      0x1.fcp-1, 0x1.010157589p-7, -0x1.0c76b999d2be8p-46,
      0x1.f8p-1, 0x1.0205658938p-6, -0x1.3dc5b06e2f7d2p-45,
      0x1.f4p-1, 0x1.8492528c9p-6, -0x1.aa0ba325a0c34p-45,
      0x1.fp-1, 0x1.0415d89e74p-5, 0x1.111c05cf1d753p-47,
      0x1.ecp-1, 0x1.466aed42ep-5, -0x1.c167375bdfd28p-45,
      0x1.e8p-1, 0x1.894aa149fcp-5, -0x1.97995d05a267dp-46,
      0x1.e4p-1, 0x1.ccb73cdddcp-5, -0x1.a68f247d82807p-46,
      0x1.e2p-1, 0x1.eea31c006cp-5, -0x1.e113e4fc93b7bp-47,
      0x1.dep-1, 0x1.1973bd1466p-4, -0x1.5325d560d9e9bp-45,
      0x1.dap-1, 0x1.3bdf5a7d1ep-4, 0x1.cc85ea5db4ed7p-45,
      0x1.d6p-1, 0x1.5e95a4d97ap-4, -0x1.c69063c5d1d1ep-45,
      0x1.d4p-1, 0x1.700d30aeacp-4, 0x1.c1e8da99ded32p-49,
      0x1.dp-1, 0x1.9335e5d594p-4, 0x1.3115c3abd47dap-45,
      0x1.ccp-1, 0x1.b6ac88dad6p-4, -0x1.390802bf768e5p-46,
      0x1.cap-1, 0x1.c885801bc4p-4, 0x1.646d1c65aacd3p-45,
      0x1.c6p-1, 0x1.ec739830a2p-4, -0x1.dc068afe645ep-45,
      0x1.c4p-1, 0x1.fe89139dbep-4, -0x1.534d64fa10afdp-45,
      0x1.cp-1, 0x1.1178e8227ep-3, 0x1.1ef78ce2d07f2p-45,
      0x1.bep-1, 0x1.1aa2b7e23fp-3, 0x1.ca78e44389934p-45,
      0x1.bap-1, 0x1.2d1610c868p-3, 0x1.39d6ccb81b4a1p-47,
      0x1.b8p-1, 0x1.365fcb0159p-3, 0x1.62fa8234b7289p-51,
      0x1.b4p-1, 0x1.4913d8333bp-3, 0x1.5837954fdb678p-45,
      0x1.b2p-1, 0x1.527e5e4a1bp-3, 0x1.633e8e5697dc7p-45,
      0x1.aep-1, 0x1.6574ebe8c1p-3, 0x1.9cf8b2c3c2e78p-46,
      0x1.acp-1, 0x1.6f0128b757p-3, -0x1.5118de59c21e1p-45,
      0x1.aap-1, 0x1.7898d85445p-3, -0x1.c661070914305p-46,
      0x1.a6p-1, 0x1.8beafeb39p-3, -0x1.73d54aae92cd1p-47,
      0x1.a4p-1, 0x1.95a5adcf7p-3, 0x1.7f22858a0ff6fp-47,
      0x1.ap-1, 0x1.a93ed3c8aep-3, -0x1.8724350562169p-45,
      0x1.9ep-1, 0x1.b31d8575bdp-3, -0x1.c358d4eace1aap-47,
      0x1.9cp-1, 0x1.bd087383bep-3, -0x1.d4bc4595412b6p-45,
      0x1.9ap-1, 0x1.c6ffbc6f01p-3, -0x1.1ec72c5962bd2p-48,
      0x1.96p-1, 0x1.db13db0d49p-3, -0x1.aff2af715b035p-45,
      0x1.94p-1, 0x1.e530effe71p-3, 0x1.212276041f43p-51,
      0x1.92p-1, 0x1.ef5ade4ddp-3, -0x1.a211565bb8e11p-51,
      0x1.9p-1, 0x1.f991c6cb3bp-3, 0x1.bcbecca0cdf3p-46,
      0x1.8cp-1, 0x1.07138604d58p-2, 0x1.89cdb16ed4e91p-48,
      0x1.8ap-1, 0x1.0c42d67616p-2, 0x1.7188b163ceae9p-45,
      0x1.88p-1, 0x1.1178e8227e8p-2, -0x1.c210e63a5f01cp-45,
      0x1.86p-1, 0x1.16b5ccbacf8p-2, 0x1.b9acdf7a51681p-45,
      0x1.84p-1, 0x1.1bf99635a68p-2, 0x1.ca6ed5147bdb7p-45,
      0x1.82p-1, 0x1.214456d0eb8p-2, 0x1.a87deba46baeap-47,
      0x1.7ep-1, 0x1.2bef07cdc9p-2, 0x1.a9cfa4a5004f4p-45,
      0x1.7cp-1, 0x1.314f1e1d36p-2, -0x1.8e27ad3213cb8p-45,
      0x1.7ap-1, 0x1.36b6776be1p-2, 0x1.16ecdb0f177c8p-46,
      0x1.78p-1, 0x1.3c25277333p-2, 0x1.83b54b606bd5cp-46,
      0x1.76p-1, 0x1.419b423d5e8p-2, 0x1.8e436ec90e09dp-47,
      0x1.74p-1, 0x1.4718dc271c8p-2, -0x1.f27ce0967d675p-45,
      0x1.72p-1, 0x1.4c9e09e173p-2, -0x1.e20891b0ad8a4p-45,
      0x1.7p-1, 0x1.522ae0738ap-2, 0x1.ebe708164c759p-45,
      0x1.6ep-1, 0x1.57bf753c8dp-2, 0x1.fadedee5d40efp-46,
      0x1.6cp-1, 0x1.5d5bddf596p-2, -0x1.a0b2a08a465dcp-47
};
  const u64 tmp = ix - 0x3fe6955500000000ull;
  const int i = (int)((tmp >> 45) & 127u);
  const double kd = (double)((i64)tmp >> 52);
  const double z = tm_u2d(ix - (tmp & (0xfffull << 52)));
  const double r = __builtin_fma(z, T[3 * i], -1.0);
  const double t1 = __builtin_fma(kd, Ln2hi, T[3 * i + 1]);
  const double t2 = t1 + r;
  const double lo1 = __builtin_fma(kd, Ln2lo, T[3 * i + 2]);
  const double lo2 = t1 - t2 + r;
  const double ar = A0 * r, ar2 = r * ar, ar3 = r * ar2;
  const double hi = t2 + ar2;
  const double lo3 = __builtin_fma(ar, r, -ar2);
  const double lo4 = t2 - hi + ar2;
  const double q = __builtin_fma(ar2, __builtin_fma(ar2, __builtin_fma(r, A6, A5), __builtin_fma(r, A4, A3)),
                                 __builtin_fma(r, A2, A1));
  const double lo = __builtin_fma(ar3, q, lo1 + lo2 + lo3 + lo4);
  const double y = hi + lo;
  tail = hi - y + lo;
  return y;
}
// exp(x + xtail) with the sign in sign_bias (0 or 0x800 << 7: added to the scale's exponent bits)
TM_FN double tm_pow_exp(double x, double xtail, u64 sign_bias) {
  const double InvLn2N = 0x1.71547652b82fep0 * 128, Shift = 0x1.8p52, NegLn2hiN = -0x1.62e42fefa0000p-8,
               NegLn2loN = -0x1.cf79abc9e3b3ap-47, C2 = 0x1.ffffffffffdbdp-2, C3 = 0x1.555555555543cp-3,
               C4 = 0x1.55555cf172b91p-5, C5 = 0x1.1111167a4d017p-7;
  u32 abstop = (u32)(tm_d2u(x) >> 52) & 0x7ffu;
  const u32 t_tiny = 0x3c9u, t_512 = 0x408u, t_1024 = 0x409u;
  if (abstop - t_tiny >= t_512 - t_tiny) {
    if ((i32)(abstop - t_tiny) < 0) return sign_bias ? -1.0 : 1.0;
    if (abstop >= t_1024) {
      if (tm_d2u(x) >> 63) return (sign_bias ? -0x1p-767 : 0x1p-767) * 0x1p-767;
      return (sign_bias ? -0x1p769 : 0x1p769) * 0x1p769;
    }
    abstop = 0u;
  }
  const double z = InvLn2N * x;
  double kd = z + Shift;
  const u64 ki = tm_d2u(kd);
  kd -= Shift;
  double r = __builtin_fma(kd, NegLn2loN, __builtin_fma(kd, NegLn2hiN, x));
  r += xtail;
  double tl;
  u64 hb;
  tm_exp_pair(ki & 127ull, tl, hb);
  const u64 sbits = hb + ((ki + sign_bias) << 45);
  const double r2 = r * r;
  const double tmp = __builtin_fma(r2 * r2, __builtin_fma(r, C5, C4), __builtin_fma(r2, __builtin_fma(r, C3, C2), tl + r));
  if (abstop == 0u) {
    if ((ki & 0x80000000ull) == 0ull) {
      const double sc = tm_u2d(sbits - (1009ull << 52));
      return 0x1p1009 * __builtin_fma(sc, tmp, sc);
    }
    const u64 sb = sbits + (1022ull << 52);
    const double sc = tm_u2d(sb);
    double y = sc + sc * tmp;
    if (__builtin_fabs(y) < 1.0) {
      const double one = y < 0.0 ? -1.0 : 1.0;
      double lo = sc - y + sc * tmp;
      const double hi = one + y;
      lo = one - hi + y + lo;
      y = (hi + lo) - one;
      if (y == 0.0) y = tm_u2d(sb & 0x8000000000000000ull);
    }
    return 0x1p-1022 * y;
  }
  const double sc = tm_u2d(sbits);
  return __builtin_fma(sc, tmp, sc);
}
TM_FN double tm_pow(double x, double y) {
  u64 sign_bias = 0;
  u64 ix = tm_d2u(x);
  const u64 iy = tm_d2u(y);
  u32 topx = (u32)(ix >> 52);
  const u32 topy = (u32)(iy >> 52);
  if (topx - 0x001u >= 0x7ffu - 0x001u || (topy & 0x7ffu) - 0x3beu >= 0x43eu - 0x3beu) {
    if (tm_zeroinfnan(iy)) {
      if (2ull * iy == 0ull) return tm_issnan(ix) ? x + y : 1.0;
      if (ix == 0x3ff0000000000000ull) return tm_issnan(iy) ? x + y : 1.0;
      if (2ull * ix > 2ull * 0x7ff0000000000000ull || 2ull * iy > 2ull * 0x7ff0000000000000ull) return x + y;
      if (2ull * ix == 2ull * 0x3ff0000000000000ull) return 1.0;
      if ((2ull * ix < 2ull * 0x3ff0000000000000ull) == !(iy >> 63)) return 0.0;
      return y * y;
    }
    if (tm_zeroinfnan(ix)) {
      double x2 = x * x;
      if ((ix >> 63) && tm_pow_checkint(iy) == 1) x2 = -x2;
      return (iy >> 63) ? 1.0 / x2 : x2;
    }
    if (ix >> 63) {
      const int yint = tm_pow_checkint(iy);
      if (yint == 0) return (x - x) / (x - x);
      if (yint == 1) sign_bias = 0x800ull << 7;
      ix &= 0x7fffffffffffffffull;
      topx &= 0x7ffu;
    }
    if ((topy & 0x7ffu) - 0x3beu >= 0x43eu - 0x3beu) {
      if (ix == 0x3ff0000000000000ull) return 1.0;
      if ((topy & 0x7ffu) < 0x3beu) return ix > 0x3ff0000000000000ull ? 1.0 + y : 1.0 - y;
      return (ix > 0x3ff0000000000000ull) == (topy < 0x800u) ? 0x1p769 * 0x1p769 : 0x1p-767 * 0x1p-767;
    }
    if (topx == 0u) {
      ix = tm_d2u(x * 0x1p52) & 0x7fffffffffffffffull;
      ix -= 52ull << 52;
    }
  }
  double lo;
  const double hi = tm_pow_log(ix, lo);
  const double ehi = y * hi;
  const double elo = __builtin_fma(y, lo, __builtin_fma(y, hi, -ehi));
  return tm_pow_exp(ehi, elo, sign_bias);
}

TM_FN u32 tm_hi32(double x) { return (u32)(tm_d2u(x) >> 32); }
TM_FN double tm_with_hi32(double x, u32 h) { return tm_u2d(((u64)h << 32) | (tm_d2u(x) & 0xffffffffull)); }

// fdlibm's expm1: x = k ln2 + r (hi - lo, with the rounding c), r in [-ln2/2, ln2/2]; e^r - 1 from the rational
// approximation r1(r^2 / 2) (glibc evaluates it as three pairs); then 2^k (e^r - 1) + 2^k - 1 assembled without
// cancellation per range of k.
TM_FN double tm_expm1(double x) {
  const double huge = 1.0e+300, tiny = 1.0e-300, o_threshold = 7.09782712893383973096e+02,
               ln2_hi = 6.93147180369123816490e-01, ln2_lo = 1.90821492927058770002e-10,
               invln2 = 1.44269504088896338700e+00, Q1 = -3.33333333333331316428e-02,
               Q2 = 1.58730158725481460165e-03, Q3 = -7.93650757867487942473e-05,
               Q4 = 4.00821782732936239552e-06, Q5 = -2.01099218183624371326e-07;
  double y, hi, lo, c = 0.0, t, e;
  i32 k;
  u32 hx = tm_hi32(x);
  const u32 neg = hx & 0x80000000u;
  hx &= 0x7fffffffu;
  if (hx >= 0x4043687Au) {                                   // |x| >= 56 ln2
    if (hx >= 0x40862E42u) {                                 // |x| >= 709.78
      if (hx >= 0x7ff00000u) {
        if (((hx & 0xfffffu) | (u32)tm_d2u(x)) != 0u) return x + x;
        return neg == 0u ? x : -1.0;
      }
      if (x > o_threshold) return huge * huge;
    }
    if (neg != 0u) return tiny - 1.0;
  }
  if (hx > 0x3fd62e42u) {                                    // |x| > ln2 / 2
    if (hx < 0x3FF0A2B2u) {                                  // and < 1.5 ln2
      if (neg == 0u) { hi = x - ln2_hi; lo = ln2_lo; k = 1; }
      else { hi = x + ln2_hi; lo = -ln2_lo; k = -1; }
    } else {
      k = (i32)(invln2 * x + (neg == 0u ? 0.5 : -0.5));
      t = (double)k;
      hi = x - t * ln2_hi;
      lo = t * ln2_lo;
    }
    x = hi - lo;
    c = (hi - x) - lo;
  } else if (hx < 0x3c900000u) {                             // |x| < 2^-54
    t = huge + x;
    return x - (t - (huge + x));
  } else {
    k = 0;
  }
  const double hfx = 0.5 * x, hxs = x * hfx;
  const double h2 = hxs * hxs, h4 = h2 * h2;
  const double r1 = (1.0 + hxs * Q1) + h2 * (Q2 + hxs * Q3) + h4 * (Q4 + hxs * Q5);
  t = 3.0 - r1 * hfx;
  e = hxs * ((r1 - t) / (6.0 - x * t));
  if (k == 0) return x - (x * e - hxs);
  e = (x * (e - c) - c);
  e -= hxs;
  if (k == -1) return 0.5 * (x - e) - 0.5;
  if (k == 1) return x < -0.25 ? -2.0 * (e - (x + 0.5)) : 1.0 + 2.0 * (x - e);
  if (k <= -2 || k > 56) {                                   // exp(x) - 1 as 2^k (1 + r) - 1
    y = 1.0 - (e - x);
    y = k == 1024 ? y * 2.0 * 0x1p1023 : tm_with_hi32(y, tm_hi32(y) + ((u32)k << 20));
    return y - 1.0;
  }
  if (k < 20) {
    t = tm_u2d((u64)(0x3ff00000u - (0x200000u >> k)) << 32);      // 1 - 2^-k
    y = t - (e - x);
  } else {
    t = tm_u2d((u64)((u32)(0x3ff - k) << 20) << 32);              // 2^-k
    y = x - (e + t);
    y += 1.0;
  }
  return tm_with_hi32(y, tm_hi32(y) + ((u32)k << 20));
}

// fdlibm's log1p: 1 + x = 2^k (1 + f) with sqrt(2)/2 < 1 + f < sqrt(2) and a correction c for the rounding of 1 + x;
// log(1 + f) = f - (f^2/2 - s (f^2/2 + R(s^2))), s = f / (2 + f), R evaluated in four pairs (as glibc does).
TM_FN double tm_log1p(double x) {
  const double ln2_hi = 6.93147180369123816490e-01, ln2_lo = 1.90821492927058770002e-10,
               Lp1 = 6.666666666666735130e-01, Lp2 = 3.999999999940941908e-01, Lp3 = 2.857142874366239149e-01,
               Lp4 = 2.222219843214978396e-01, Lp5 = 1.818357216161805012e-01, Lp6 = 1.531383769920937332e-01,
               Lp7 = 1.479819860511658591e-01;
  double f = 0.0, c = 0.0, u;
  i32 k = 1, hu = 0;
  const i32 hx = (i32)tm_hi32(x), ax = hx & 0x7fffffff;
  if (hx < 0x3FDA827A) {                                     // x < 0.41422
    if (ax >= 0x3ff00000) return x == -1.0 ? -__builtin_inf() : __builtin_nan("");    // x <= -1
    if (ax < 0x3e200000) {                                   // |x| < 2^-29
      if (ax < 0x3c900000) return x;
      return x - x * x * 0.5;
    }
    if (hx > 0 || hx <= (i32)0xbfd2bec3u) { k = 0; f = x; hu = 1; }      // -0.2929 < x < 0.41422
  } else if (hx >= 0x7ff00000) {
    return x + x;
  }
  if (k != 0) {
    if (hx < 0x43400000) {
      u = 1.0 + x;
      hu = (i32)tm_hi32(u);
      k = (hu >> 20) - 1023;
      c = k > 0 ? 1.0 - (u - x) : x - (u - 1.0);
      c /= u;
    } else {
      u = x;
      hu = (i32)tm_hi32(u);
      k = (hu >> 20) - 1023;
      c = 0.0;
    }
    hu &= 0x000fffff;
    if (hu < 0x6a09e) {
      u = tm_with_hi32(u, (u32)(hu | 0x3ff00000));          // normalise u
    } else {
      k += 1;
      u = tm_with_hi32(u, (u32)(hu | 0x3fe00000));          // normalise u / 2
      hu = (0x00100000 - hu) >> 2;
    }
    f = u - 1.0;
  }
  const double hfsq = 0.5 * f * f;
  const double dk = (double)k;
  if (hu == 0) {                                             // |f| < 2^-20
    if (f == 0.0) {
      if (k == 0) return 0.0;
      c += dk * ln2_lo;
      return dk * ln2_hi + c;
    }
    const double R = hfsq * (1.0 - 0.66666666666666666 * f);
    if (k == 0) return f - R;
    return dk * ln2_hi - ((R - (dk * ln2_lo + c)) - f);
  }
  const double s = f / (2.0 + f), z = s * s;
  const double z2 = z * z, z4 = z2 * z2, z6 = z4 * z2;
  const double R = z * Lp1 + z2 * (Lp2 + z * Lp3) + z4 * (Lp4 + z * Lp5) + z6 * (Lp6 + z * Lp7);
  if (k == 0) return f - (hfsq - s * (hfsq + R));
  return dk * ln2_hi - ((hfsq - (s * (hfsq + R) + (dk * ln2_lo + c))) - f);
}

// fdlibm's tanh on tm_expm1: |x| < 1: -t / (t + 2), t = expm1(-2|x|); 1 <= |x| < 22: 1 - 2 / (expm1(2|x|) + 2).
TM_FN double tm_tanh(double x) {
  const i32 jx = (i32)tm_hi32(x), ix = jx & 0x7fffffff;
  double t, z;
  if (ix >= 0x7ff00000) return jx >= 0 ? 1.0 / x + 1.0 : 1.0 / x - 1.0;
  if (ix < 0x40360000) {                                     // |x| < 22
    if ((ix | (i32)(u32)tm_d2u(x)) == 0) return x;
    if (ix < 0x3c800000) return x * (1.0 + x);               // |x| < 2^-55
    if (ix >= 0x3ff00000) {
      t = tm_expm1(2.0 * __builtin_fabs(x));
      z = 1.0 - 2.0 / (t + 2.0);
    } else {
      t = tm_expm1(-2.0 * __builtin_fabs(x));
      z = -t / (t + 2.0);
    }
  } else {
    z = 1.0 - 1.0e-300;
  }
  return jx >= 0 ? z : -z;
}

// fdlibm's sinh / cosh on tm_expm1 and tm_exp: |x| < 22 from expm1 (cosh: from exp past ln2 / 2), then e^|x| / 2,
// and near the overflow threshold (e^(|x|/2) / 2) e^(|x|/2).
TM_FN double tm_sinh(double x) {
  const i32 jx = (i32)tm_hi32(x), ix = jx & 0x7fffffff;
  if (ix >= 0x7ff00000) return x + x;
  const double h = jx < 0 ? -0.5 : 0.5;
  if (ix < 0x40360000) {                                     // |x| < 22
    if (ix < 0x3e300000 && 1.0e307 + x > 1.0) return x;      // |x| < 2^-28
    const double t = tm_expm1(__builtin_fabs(x));
    if (ix < 0x3ff00000) return h * (2.0 * t - t * t / (t + 1.0));
    return h * (t + t / (t + 1.0));
  }
  if (ix < 0x40862e42) return h * tm_exp(__builtin_fabs(x));
  const u32 lx = (u32)tm_d2u(x);
  if (ix < 0x408633ce || (ix == 0x408633ce && lx <= 0x8fb9f87du)) {
    const double w = tm_exp(0.5 * __builtin_fabs(x)), t = h * w;
    return t * w;
  }
  return x * 1.0e307;
}

TM_FN double tm_cosh(double x) {
  const i32 ix = (i32)tm_hi32(x) & 0x7fffffff;
  if (ix < 0x40360000) {                                     // |x| < 22
    if (ix < 0x3fd62e43) {                                   // |x| < ln2 / 2
      if (ix < 0x3c800000) return 1.0;
      const double t = tm_expm1(__builtin_fabs(x)), w = 1.0 + t;
      return 1.0 + (t * t) / (w + w);
    }
    const double t = tm_exp(__builtin_fabs(x));
    return 0.5 * t + 0.5 / t;
  }
  if (ix < 0x40862e42) return 0.5 * tm_exp(__builtin_fabs(x));
  const u32 lx = (u32)tm_d2u(x);
  if (ix < 0x408633ce || (ix == 0x408633ce && lx <= 0x8fb9f87du)) {
    const double w = tm_exp(0.5 * __builtin_fabs(x)), t = 0.5 * w;
    return t * w;
  }
  if (ix >= 0x7ff00000) return x * x;
  return 1.0e300 * 1.0e300;
}

// fdlibm's atanh on tm_log1p: atanh |x| = log1p(2|x| + 2|x||x| / (1 - |x|)) / 2 below 1/2, log1p(2|x| / (1 - |x|))
// / 2 above.
TM_FN double tm_atanh(double x) {
  const double xa = __builtin_fabs(x);
  double t;
  if (xa < 0.5) {
    if (xa < 0x1.0p-28) return x;
    t = xa + xa;
    t = 0.5 * tm_log1p(t + t * xa / (1.0 - xa));
  } else if (xa < 1.0) {
    t = 0.5 * tm_log1p((xa + xa) / (1.0 - xa));
  } else if (xa > 1.0) {
    return (x - x) / (x - x);
  } else if (xa == 1.0) {
    return x / 0.0;
  } else {
    return x + x;                                            // NaN
  }
  return __builtin_copysign(t, x);
}

// fdlibm's asinh on tm_log / tm_log1p: |x| below 2^-28 x itself; to 2 log1p(|x| + x^2 / (1 + sqrt(1 + x^2))); to
// 2^28 log(2|x| + 1 / (sqrt(x^2 + 1) + |x|)); beyond log|x| + ln2; the sign of x restored.
TM_FN double tm_asinh(double x) {
  const double ln2 = 6.93147180559945286227e-01;
  const u32 ix = tm_hi32(x) & 0x7fffffffu;
  if (ix < 0x3e300000u) return x;
  double w;
  if (ix > 0x41b00000u) {
    if (ix >= 0x7ff00000u) return x + x;
    w = tm_log(__builtin_fabs(x)) + ln2;
  } else {
    const double xa = __builtin_fabs(x);
    if (ix > 0x40000000u) {
      w = tm_log(2.0 * xa + 1.0 / (__builtin_sqrt(xa * xa + 1.0) + xa));
    } else {
      const double t = xa * xa;
      w = tm_log1p(xa + t / (1.0 + __builtin_sqrt(1.0 + t)));
    }
  }
  return __builtin_copysign(w, x);
}

// fdlibm's acosh (its 64-bit-word form: the branches compare the whole bit pattern): beyond 2^28 log x + ln2;
// above 2 log(2x - 1 / (x + sqrt(x^2 - 1))); above 1 log1p(t + sqrt(2t + t^2)), t = x - 1; 0 at 1; NaN below.
TM_FN double tm_acosh(double x) {
  const double ln2 = 6.93147180559945286227e-01;
  const i64 hx = (i64)tm_d2u(x);
  if (hx > 0x4000000000000000ll) {
    if (hx >= 0x41b0000000000000ll) {
      if (hx >= 0x7ff0000000000000ll) return x + x;
      return tm_log(x) + ln2;
    }
    const double t = x * x;
    return tm_log(2.0 * x - 1.0 / (x + __builtin_sqrt(t - 1.0)));
  }
  if (hx > 0x3ff0000000000000ll) {
    const double t = x - 1.0;
    return tm_log1p(t + __builtin_sqrt(2.0 * t + t * t));
  }
  if (hx == 0x3ff0000000000000ll) return 0.0;
  return (x - x) / (x - x);
}

// fdlibm's erf / erfc: |x| < 0.84375 a rational approximation in x^2; to 1.25 one in |x| - 1 about erf(1) ~ erx;
// beyond, exp(-z^2 - 0.5625) exp((z - x)(z + x) + R / S) / x with z = x with its low word cleared and R / S a
// rational approximation in 1 / x^2 (two of them, split at |x| = 1 / 0.35).  glibc evaluates every polynomial in
// pairs (c_i + s c_{i+1}) combined with powers of s: that order is kept.
TM_FN void tm_erf_tail(double x, bool erfc, double& R, double& S) {
  const double ra0 = -9.86494403484714822705e-03, ra1 = -6.93858572707181764372e-01,
               ra2 = -1.05586262253232909814e+01, ra3 = -6.23753324503260060396e+01,
               ra4 = -1.62396669462573470355e+02, ra5 = -1.84605092906711035994e+02,
               ra6 = -8.12874355063065934246e+01, ra7 = -9.81432934416914548592e+00,
               sa1 = 1.96512716674392571292e+01, sa2 = 1.37657754143519042600e+02, sa3 = 4.34565877475229228821e+02,
               sa4 = 6.45387271733267880336e+02, sa5 = 4.29008140027567833386e+02, sa6 = 1.08635005541779435134e+02,
               sa7 = 6.57024977031928170135e+00, sa8 = -6.04244152148580987438e-02,
               rb0 = -9.86494292470009928597e-03, rb1 = -7.99283237680523006574e-01,
               rb2 = -1.77579549177547519889e+01, rb3 = -1.60636384855821916062e+02,
               rb4 = -6.37566443368389627722e+02, rb5 = -1.02509513161107724954e+03,
               rb6 = -4.83519191608651397019e+02, sb1 = 3.03380607434824582924e+01,
               sb2 = 3.25792512996573918826e+02, sb3 = 1.53672958608443695994e+03, sb4 = 3.19985821950859553908e+03,
               sb5 = 2.55305040643316442583e+03, sb6 = 4.74528541206955367215e+02, sb7 = -2.24409524465858183362e+01;
  const double s = 1.0 / (x * x), s2 = s * s, s4 = s2 * s2, s6 = s4 * s2;
  // (the switch between the two tails: |x| < 1 / 0.35, whose high word is compared against 0x4006DB6E by erf and
  // 0x4006DB6D by erfc)
  const u32 ix = tm_hi32(x) & 0x7fffffffu;
  if (ix < (erfc ? 0x4006DB6Du : 0x4006DB6Eu)) {
    const double s8 = s4 * s4;
    R = (ra0 + s * ra1) + s2 * (ra2 + s * ra3) + s4 * (ra4 + s * ra5) + s6 * (ra6 + s * ra7);
    S = (1.0 + s * sa1) + s2 * (sa2 + s * sa3) + s4 * (sa4 + s * sa5) + s6 * (sa6 + s * sa7) + s8 * sa8;
  } else {
    R = (rb0 + s * rb1) + s2 * (rb2 + s * rb3) + s4 * (rb4 + s * rb5) + s6 * rb6;
    S = (1.0 + s * sb1) + s2 * (sb2 + s * sb3) + s4 * (sb4 + s * sb5) + s6 * (sb6 + s * sb7);
  }
}

TM_FN double tm_erf_small(double z) {                       // (erf x - x) / x for |x| < 0.84375, z = x^2
  const double pp0 = 1.28379167095512558561e-01, pp1 = -3.25042107247001499370e-01,
               pp2 = -2.84817495755985104766e-02, pp3 = -5.77027029648944159157e-03,
               pp4 = -2.37630166566501626084e-05, qq1 = 3.97917223959155352819e-01,
               qq2 = 6.50222499887672944485e-02, qq3 = 5.08130628187576562776e-03,
               qq4 = 1.32494738004321644526e-04, qq5 = -3.96022827877536812320e-06;
  const double z2 = z * z, z4 = z2 * z2;
  const double r = (pp0 + z * pp1) + z2 * (pp2 + z * pp3) + z4 * pp4;
  const double s = (1.0 + z * qq1) + z2 * (qq2 + z * qq3) + z4 * (qq4 + z * qq5);
  return r / s;
}

TM_FN double tm_erf_mid(double s) {                         // erf |x| - erx for 0.84375 <= |x| < 1.25, s = |x| - 1
  const double pa0 = -2.36211856075265944077e-03, pa1 = 4.14856118683748331666e-01,
               pa2 = -3.72207876035701323847e-01, pa3 = 3.18346619901161753674e-01,
               pa4 = -1.10894694282396677476e-01, pa5 = 3.54783043256182359371e-02,
               pa6 = -2.16637559486879084300e-03, qa1 = 1.06420880400844228286e-01,
               qa2 = 5.40397917702171048937e-01, qa3 = 7.18286544141962662868e-02,
               qa4 = 1.26171219808761642112e-01, qa5 = 1.36370839120290507362e-02,
               qa6 = 1.19844998467991074170e-02;
  const double s2 = s * s, s4 = s2 * s2, s6 = s4 * s2;
  const double P = (pa0 + s * pa1) + s2 * (pa2 + s * pa3) + s4 * (pa4 + s * pa5) + s6 * pa6;
  const double Q = (1.0 + s * qa1) + s2 * (qa2 + s * qa3) + s4 * (qa4 + s * qa5) + s6 * qa6;
  return P / Q;
}

TM_FN double tm_erfc_tail(double ax, bool erfc) {          // erfc |x| for 1.25 <= |x| (|x| < 28)
  double R, S;
  tm_erf_tail(ax, erfc, R, S);
  const double z = tm_u2d(tm_d2u(ax) & 0xffffffff00000000ull);
  const double r = tm_exp(-z * z - 0.5625) * tm_exp((z - ax) * (z + ax) + R / S);
  return r / ax;
}

TM_FN double tm_erf(double x) {
  const double erx = 8.45062911510467529297e-01, efx = 1.28379167095512586316e-01;
  const i32 hx = (i32)tm_hi32(x), ix = hx & 0x7fffffff;
  if (ix >= 0x7ff00000) return (double)(1 - (i32)(((u32)hx >> 31) << 1)) + 1.0 / x;
  if (ix < 0x3feb0000) {                                     // |x| < 0.84375
    if (ix < 0x3e300000) {                                   // |x| < 2^-28
      if (ix < 0x00800000) return 0.0625 * (16.0 * x + (16.0 * efx) * x);
      return x + efx * x;
    }
    return x + x * tm_erf_small(x * x);
  }
  if (ix < 0x3ff40000) {                                     // |x| < 1.25
    const double pq = tm_erf_mid(__builtin_fabs(x) - 1.0);
    return hx >= 0 ? erx + pq : -erx - pq;
  }
  if (ix >= 0x40180000) return hx >= 0 ? 1.0 - 1.0e-300 : 1.0e-300 - 1.0;     // |x| >= 6
  const double q = tm_erfc_tail(__builtin_fabs(x), false);
  return hx >= 0 ? 1.0 - q : q - 1.0;
}

TM_FN double tm_erfc(double x) {
  const double erx = 8.45062911510467529297e-01;
  const i32 hx = (i32)tm_hi32(x), ix = hx & 0x7fffffff;
  if (ix >= 0x7ff00000) return (double)(((u32)hx >> 31) << 1) + 1.0 / x;
  if (ix < 0x3feb0000) {                                     // |x| < 0.84375
    if (ix < 0x3c700000) return 1.0 - x;                     // |x| < 2^-56
    const double y = tm_erf_small(x * x);
    if (hx < 0x3fd00000) return 1.0 - (x + x * y);           // x < 1/4
    double r = x * y;
    r += (x - 0.5);
    return 0.5 - r;
  }
  if (ix < 0x3ff40000) {                                     // |x| < 1.25
    const double pq = tm_erf_mid(__builtin_fabs(x) - 1.0);
    if (hx >= 0) return (1.0 - erx) - pq;
    return 1.0 + (erx + pq);
  }
  if (ix < 0x403c0000) {                                     // |x| < 28
    if (hx < 0 && ix >= 0x40180000) return 2.0 - 1.0e-300;   // x <= -6
    const double q = tm_erfc_tail(__builtin_fabs(x), true);
    return hx > 0 ? q : 2.0 - q;
  }
  return hx > 0 ? 1.0e-300 * 1.0e-300 : 2.0 - 1.0e-300;
}

// lax.logistic of float64 as the reference's CPU target computes it (op_table.py:243-247): 1 / (1 + exp(-x)), on
// tm_exp (glibc's exp).
TM_FN double tm_logistic_d(double x) { return 1.0 / (1.0 + tm_exp(-x)); }

// fdlibm's lgamma (double) as glibc 2.35's generic build computes it, on tm_log: the float version's branches with
// the double coefficients and thresholds on the high word, Stirling's series to 2^58.  Bitwise for x > 0 (and the
// tiny and huge negative branches); other negative arguments take glibc's sin(pi x) on its IBM sin / cos and, on
// (-28, -2), its own lgamma_neg (LGPL), neither restated here: there the device's math library is used.
TM_FN double tm_lgamma_pos(double x) {                // x > 0, finite, at least 2^-70
  const double a0 = 7.72156649015328655494e-02, a1 = 3.22467033424113591611e-01, a2 = 6.73523010531292681824e-02,
      a3 = 2.05808084325167332806e-02, a4 = 7.38555086081402883957e-03, a5 = 2.89051383673415629091e-03,
      a6 = 1.19270763183362067845e-03, a7 = 5.10069792153511336608e-04, a8 = 2.20862790713908385557e-04,
      a9 = 1.08011567247583939954e-04, a10 = 2.52144565451257326939e-05, a11 = 4.48640949618915160150e-05;
  const double tc = 1.46163214496836224576e+00, tf = -1.21486290535849611461e-01, tt = -3.63867699703950536541e-18;
  const double t0 = 4.83836122723810047042e-01, t1 = -1.47587722994593911752e-01, t2 = 6.46249402391333854778e-02,
      t3 = -3.27885410759859649565e-02, t4 = 1.79706750811820387126e-02, t5 = -1.03142241298341437450e-02,
      t6 = 6.10053870246291332635e-03, t7 = -3.68452016781138256760e-03, t8 = 2.25964780900612472250e-03,
      t9 = -1.40346469989232843813e-03, t10 = 8.81081882437654011382e-04, t11 = -5.38595305356740546715e-04,
      t12 = 3.15632070903625950361e-04, t13 = -3.12754168375120860518e-04, t14 = 3.35529192635519073543e-04;
  const double u0 = -7.72156649015328655494e-02, u1 = 6.32827064025093366517e-01, u2 = 1.45492250137234768737e+00,
      u3 = 9.77717527963372745603e-01, u4 = 2.28963728064692451092e-01, u5 = 1.33810918536787660377e-02,
      v1 = 2.45597793713041134822e+00, v2 = 2.12848976379893395361e+00, v3 = 7.69285150456672783825e-01,
      v4 = 1.04222645593369134254e-01, v5 = 3.21709242282423911810e-03;
  const double s0 = -7.72156649015328655494e-02, s1 = 2.14982415960608852501e-01, s2 = 3.25778796408930981787e-01,
      s3 = 1.46350472652464452805e-01, s4 = 2.66422703033638609560e-02, s5 = 1.84028451407337715652e-03,
      s6 = 3.19475326584100867617e-05, r1 = 1.39200533467621045958e+00, r2 = 7.21935547567138069525e-01,
      r3 = 1.71933865632803078993e-01, r4 = 1.86459191715652901344e-02, r5 = 7.77942496381893596434e-04,
      r6 = 7.32668430744625636189e-06;
  const double w0 = 4.18938533204672725052e-01, w1 = 8.33333333333329678849e-02, w2 = -2.77777777728775536470e-03,
      w3 = 7.93650558643019558500e-04, w4 = -5.95187557450339963135e-04, w5 = 8.36339918996282139126e-04,
      w6 = -1.63092934096575273989e-03;
  const u32 ix = tm_hi32(x), lx = (u32)tm_d2u(x);
  if (((ix - 0x3ff00000u) | lx) == 0u || ((ix - 0x40000000u) | lx) == 0u) return 0.0;
  if (ix < 0x40000000u) {                             // x < 2
    double r, y;
    int i;
    if (ix <= 0x3fecccccu) {                          // x <= 0.9: lgamma(x + 1) - log x
      r = -tm_log(x);
      if (ix >= 0x3fe76944u) { y = 1.0 - x; i = 0; }
      else if (ix >= 0x3fcda661u) { y = x - (tc - 1.0); i = 1; }
      else { y = x; i = 2; }
    } else {
      r = 0.0;
      if (ix >= 0x3ffbb4c3u) { y = 2.0 - x; i = 0; }
      else if (ix >= 0x3ff3b4c4u) { y = x - tc; i = 1; }
      else { y = x - 1.0; i = 2; }
    }
    if (i == 0) {
      const double z = y * y;
      const double p1 = a0 + z * (a2 + z * (a4 + z * (a6 + z * (a8 + z * a10))));
      const double p2 = z * (a1 + z * (a3 + z * (a5 + z * (a7 + z * (a9 + z * a11)))));
      const double p = y * p1 + p2;
      return r + (p - 0.5 * y);
    }
    if (i == 1) {
      const double z = y * y, w = z * y;
      const double p1 = t0 + w * (t3 + w * (t6 + w * (t9 + w * t12)));
      const double p2 = t1 + w * (t4 + w * (t7 + w * (t10 + w * t13)));
      const double p3 = t2 + w * (t5 + w * (t8 + w * (t11 + w * t14)));
      const double p = z * p1 - (tt - w * (p2 + y * p3));
      return r + (tf + p);
    }
    const double p1 = y * (u0 + y * (u1 + y * (u2 + y * (u3 + y * (u4 + y * u5)))));
    const double p2 = 1.0 + y * (v1 + y * (v2 + y * (v3 + y * (v4 + y * v5))));
    return r + (-0.5 * y + p1 / p2);
  }
  if (ix < 0x40200000u) {                             // 2 <= x < 8
    const int i = (int)x;
    const double y = x - (double)i;
    const double p = y * (s0 + y * (s1 + y * (s2 + y * (s3 + y * (s4 + y * (s5 + y * s6))))));
    const double q = 1.0 + y * (r1 + y * (r2 + y * (r3 + y * (r4 + y * (r5 + y * r6)))));
    double r = 0.5 * y + p / q, z = 1.0;
    if (i >= 7) z *= y + 6.0;
    if (i >= 6) z *= y + 5.0;
    if (i >= 5) z *= y + 4.0;
    if (i >= 4) z *= y + 3.0;
    if (i >= 3) { z *= y + 2.0; r += tm_log(z); }
    return r;
  }
  if (ix < 0x43900000u) {                             // 8 <= x < 2^58
    const double t = tm_log(x), z = 1.0 / x, y = z * z;
    const double w = w0 + z * (w1 + y * (w2 + y * (w3 + y * (w4 + y * (w5 + y * w6)))));
    return (x - 0.5) * (t - 1.0) + w;
  }
  return x * (tm_log(x) - 1.0);
}
TM_FN double tm_lgamma(double x) {
  const u32 hx = tm_hi32(x), ix = hx & 0x7fffffffu, lx = (u32)tm_d2u(x);
  if (ix >= 0x7ff00000u) return x * x;
  if ((ix | lx) == 0u) return 1.0 / __builtin_fabs(x);
  if (ix < 0x3b900000u) return -tm_log(__builtin_fabs(x));    // |x| < 2^-70
  if (!(hx >> 31)) return tm_lgamma_pos(x);
  if (ix >= 0x43300000u) return __builtin_fabs(x) / 0.0;      // x <= -2^52: a negative integer
  return lgamma(x);                                           // the device's math library
}

// float64 erf_inv as the reference CPU target computes it (host.py:106-129): Giles (2010)'s single-precision
// polynomial in double on w = -log((1 - |y|)(1 + |y|)) (separate multiplies and adds, glibc's log and sqrt), then
// Halley steps x -= f / (d (1 + x f / d)) with f = erf x - |y| below |y| = 1/2 and (1 - |y|) - erfc x above (where
// 1 - |y| is exact), d = (2 / sqrt pi) e^(-x^2), at most 8, until a step is within 2.3e-16 x; on the restated
// log, erf, erfc and exp, so every step rounds as the reference's does.
TM_FN double tm_giles_ref(double y) {
  const double a = __builtin_fabs(y);
  double w = -tm_log((1.0 - a) * (1.0 + a)), p;
  if (w < 5.0) {
    w -= 2.5;
    p = 2.81022636e-08;
    p = 3.43273939e-07 + p * w;
    p = -3.5233877e-06 + p * w;
    p = -4.39150654e-06 + p * w;
    p = 0.00021858087 + p * w;
    p = -0.00125372503 + p * w;
    p = -0.00417768164 + p * w;
    p = 0.246640727 + p * w;
    p = 1.50140941 + p * w;
  } else {
    w = __builtin_sqrt(w) - 3.0;
    p = -0.000200214257;
    p = 0.000100950558 + p * w;
    p = 0.00134934322 + p * w;
    p = -0.00367342844 + p * w;
    p = 0.00573950773 + p * w;
    p = -0.0076224613 + p * w;
    p = 0.00943887047 + p * w;
    p = 1.00167406 + p * w;
    p = 2.83297682 + p * w;
  }
  return p * a;
}
TM_FN double tm_erfinv(double y) {
  if (!(y > -1.0 && y < 1.0)) return y == 1.0 ? __builtin_inf() : (y == -1.0 ? -__builtin_inf() : __builtin_nan(""));
  if (y == 0.0) return y;
  const double a = __builtin_fabs(y);
  double x = tm_giles_ref(y);
  for (int i = 0; i < 8; ++i) {
    const double f = a < 0.5 ? tm_erf(x) - a : (1.0 - a) - tm_erfc(x);
    const double d = 1.1283791670955126 * tm_exp(-x * x);
    const double dx = f / (d * (1.0 + x * f / d));
    x -= dx;
    if (__builtin_fabs(dx) <= 2.3e-16 * x) break;
  }
  return __builtin_copysign(x, y);
}

