// tm_device.h -- the CDNA4 device runtime of generated tallymap kernels (gfx950, wave64).
//
// Every generated module is this header + tm_libm.h + the program's own code (backend/codegen.py, kernel.py).  The
// scalar helpers are TM_FN (host + device) so that the same definitions can be compiled for the host and checked
// there; the wave-level pieces (claims, atomics, LDS) are device-only.
//
// Semantics restated from the reference's device prelude (tallymap/backends/kernel/kernel.py:26-188) and its CPU
// target (host.py:43-171), written for AMD hardware:
//   - lax max/min: NaN-propagating, a signed-zero tie gives +0 / -0 (kernel.py:78-83);
//   - lax integer div/rem: x/0 = -1 (unsigned: all ones), INT_MIN/-1 = INT_MIN; x%0 = x, INT_MIN%-1 = 0
//     (kernel.py:95-103);
//   - shifts by >= the width give 0 (logical) or the sign fill (arithmetic) (kernel.py:104-109);
//   - float -> int toward zero, saturating, NaN -> 0 (host.py:133-146; v_cvt_i32_f32 behaves so natively);
//   - threefry2x32, 20 rounds (the function of kernel.py:137-150; Salmon et al. 2011);
//   - float tallies keep subnormals: adds that could meet one go through an IEEE compare-and-swap loop (the
//     guarantee of kernel.py:112-135);
//   - the exact f32 sum: every bin's total is the correctly rounded exact sum of its emits, whatever their order,
//     or NaN when an emit is not finite (the meaning of kernel.py:870-941; the word format here is this runtime's
//     own: words of 32-bit weight, one atomic per emit).
#pragma once

typedef signed char i8;
typedef unsigned char u8;
typedef short i16;
typedef unsigned short u16;
typedef int i32;
typedef unsigned int u32;
typedef long long i64;
typedef unsigned long long u64;
#if defined(__clang__)
typedef u32 tm_u32x4 __attribute__((ext_vector_type(4)));     // a 16-byte unit (one dwordx4 load / store)
typedef u32 tm_u32x2 __attribute__((ext_vector_type(2)));     // an 8-byte unit
#endif

#ifdef __HIPCC_RTC__
#define TM_DEVICE_ONLY 1
#endif
#if defined(__HIP__) || defined(__HIPCC_RTC__)
#define TM_FN __host__ __device__ __forceinline__
#define TM_DFN __device__ __forceinline__
#define TM_DNOINLINE __device__ __noinline__
#else
#define TM_FN static inline
#endif

template <class To, class From> TM_FN To tm_bitcast(From x) { return __builtin_bit_cast(To, x); }
TM_FN float tm_u2f(u32 u) { return __builtin_bit_cast(float, u); }
TM_FN u32 tm_f2u(float f) { return __builtin_bit_cast(u32, f); }
TM_FN double tm_u2d(u64 u) { return __builtin_bit_cast(double, u); }
TM_FN u64 tm_d2u(double d) { return __builtin_bit_cast(u64, d); }

// ------------------------------------------------------------------------- 64-bit shifts by a variable amount
// Built from 32-bit shifts of the two halves, s in [0, 63].  gfx950 returns wrong results from a 64-bit VALU
// shift (v_lshlrev_b64 / v_lshrrev_b64 / v_ashrrev_i64) whose shift-amount VGPR is the last register of an
// 8-register allocation block (v7, v15, ..., v39 in a 40-register kernel): measured on MI355X as corrupted exact
// sums, the register placement being the register allocator's choice.  Every 64-bit shift by a non-constant amount
// in device code goes through these, so that no such instruction is emitted; backend/compile.py rejects a code
// object that still contains one.
TM_FN u64 tm_shl64(u64 x, u32 s) {
  const u32 lo = (u32)x, hi = (u32)(x >> 32);
  const u32 rh = s >= 32u ? lo << (s - 32u) : (s ? (hi << s) | (lo >> (32u - s)) : hi);
  const u32 rl = s >= 32u ? 0u : lo << s;
  return ((u64)rh << 32) | (u64)rl;
}
TM_FN u64 tm_shr64(u64 x, u32 s) {
  const u32 lo = (u32)x, hi = (u32)(x >> 32);
  const u32 rl = s >= 32u ? hi >> (s - 32u) : (s ? (lo >> s) | (hi << (32u - s)) : lo);
  const u32 rh = s >= 32u ? 0u : hi >> s;
  return ((u64)rh << 32) | (u64)rl;
}
TM_FN i64 tm_sar64(i64 x, u32 s) {
  const u32 lo = (u32)(u64)x;
  const i32 hi = (i32)(u32)((u64)x >> 32);
  const u32 rl = s >= 32u ? (u32)(hi >> (s - 32u)) : (s ? (lo >> s) | ((u32)hi << (32u - s)) : lo);
  const u32 rh = (u32)(hi >> (s >= 32u ? 31u : s));
  return (i64)(((u64)rh << 32) | (u64)rl);
}
// u64 -> f32 rounded once, through an exact double (n < 2^53): the direct conversion lowers to a 64-bit shift
TM_FN float tm_u64_f32(u64 n) { return (float)(double)n; }
// u64 / i64 -> f32 for every value, rounded once (to nearest even) from 32-bit halves: the 32 leading significant
// bits with a sticky bit for the bits below them (so the one rounding of the u32 -> f32 conversion is the rounding
// of the whole value), then an exact scaling by a power of two.  The compiler's own expansion normalises the
// operand with a 64-bit shift by its leading-zero count, a variable 64-bit shift (see tm_shl64).
TM_FN float tm_u64f(u64 u) {
  const u32 hi = (u32)(u >> 32), lo = (u32)u;
  if (hi == 0u) return (float)lo;
  const u32 n = (u32)__builtin_clz(hi);
  const u32 m = n ? (hi << n) | (lo >> (32u - n)) : hi;
  const u32 rest = n ? lo << n : lo;
  return __builtin_ldexpf((float)(m | (rest != 0u ? 1u : 0u)), (int)(32u - n));
}
TM_FN float tm_i64f(i64 x) {
  const float f = tm_u64f(x < 0 ? 0ull - (u64)x : (u64)x);
  return x < 0 ? -f : f;
}

// ------------------------------------------------------------------------------------------- lax helpers
// (float32 on gfx950: v_maximum3_f32 / v_minimum3_f32 are exactly these, one instruction for the ~8 of the comparisons)
template <class T> TM_FN T tm_fmax(T a, T b) {
#if defined(__HIP_DEVICE_COMPILE__)
  if constexpr (sizeof(T) == 4) return __builtin_elementwise_maximum(a, b);
#endif
  return (a > b || a != a) ? a : ((b > a || b != b) ? b : (a == (T)0 ? a + b : a));
}
template <class T> TM_FN T tm_fmin(T a, T b) {
#if defined(__HIP_DEVICE_COMPILE__)
  if constexpr (sizeof(T) == 4) return __builtin_elementwise_minimum(a, b);
#endif
  return (a < b || a != a) ? a : ((b < a || b != b) ? b : (a == (T)0 ? -(-a - b) : a));
}
template <class T> TM_FN T tm_imax(T a, T b) { return a > b ? a : b; }
template <class T> TM_FN T tm_imin(T a, T b) { return a < b ? a : b; }
template <class T> TM_FN T tm_fsign(T a) { return a > (T)0 ? (T)1 : (a < (T)0 ? (T)-1 : a); }

TM_FN i32 tm_idiv(i32 a, i32 b) { return b == 0 ? -1 : ((b == -1 && a == (i32)0x80000000u) ? a : a / b); }
TM_FN i32 tm_irem(i32 a, i32 b) { return b == 0 ? a : ((b == -1 && a == (i32)0x80000000u) ? 0 : a % b); }
TM_FN u32 tm_idiv(u32 a, u32 b) { return b == 0u ? 0xffffffffu : a / b; }
TM_FN u32 tm_irem(u32 a, u32 b) { return b == 0u ? a : a % b; }
TM_FN i64 tm_idiv(i64 a, i64 b) {
  return b == 0 ? -1 : ((b == -1 && a == (i64)0x8000000000000000ull) ? a : a / b);
}
TM_FN i64 tm_irem(i64 a, i64 b) {
  return b == 0 ? a : ((b == -1 && a == (i64)0x8000000000000000ull) ? 0 : a % b);
}

template <class T, class U> TM_FN T tm_shl(T a, T b) {
  if ((U)b >= (U)(sizeof(T) * 8)) return (T)0;
  if constexpr (sizeof(T) == 8) return (T)tm_shl64((u64)a, (u32)b);
  else return (T)((U)a << (U)b);
}
template <class T, class U> TM_FN T tm_shrl(T a, T b) {
  if ((U)b >= (U)(sizeof(T) * 8)) return (T)0;
  if constexpr (sizeof(T) == 8) return (T)tm_shr64((u64)a, (u32)b);
  else return (T)((U)a >> (U)b);
}
template <class T, class U> TM_FN T tm_shra(T a, T b) {
  if ((U)b >= (U)(sizeof(T) * 8)) return (T)(a < (T)0 ? (T)-1 : (T)0);
  if constexpr (sizeof(T) == 8) return (T)tm_sar64((i64)a, (u32)b);
  else return (T)(a >> (U)b);
}

// Order keys of floats as signed integers.  tm_tkey: IEEE total order (-NaN < -inf < ... < -0 < +0 < ... < +NaN,
// lax's eq_to / lt_to / le_to): the bits with the magnitude flipped for a negative sign.  tm_skey: lax.sort's order,
// which first makes -0 +0 and every NaN the one +NaN (so NaNs compare equal and sort last).
TM_FN i32 tm_tkey(float x) {
  const u32 b = tm_f2u(x);
  return (i32)(b ^ ((u32)((i32)b >> 31) >> 1));
}
TM_FN i64 tm_tkey(double x) {
  const u64 b = tm_d2u(x);
  return (i64)(b ^ ((u64)((i64)b >> 63) >> 1));
}
TM_FN i32 tm_skey(float x) { return tm_tkey(x != x ? tm_u2f(0x7fc00000u) : (x == 0.0f ? 0.0f : x)); }
TM_FN i64 tm_skey(double x) { return tm_tkey(x != x ? tm_u2d(0x7ff8000000000000ull) : (x == 0.0 ? 0.0 : x)); }

// lax.mulhi: the high half of the double-width product.  64-bit operands from 32-bit partial products (a 128-bit
// type is not relied on in device code); the signed form corrects the unsigned one by the operands' signs.
TM_FN u64 tm_umulhi64(u64 a, u64 b) {
  const u64 al = (u32)a, ah = a >> 32, bl = (u32)b, bh = b >> 32;
  const u64 ll = al * bl, lh = al * bh, hl = ah * bl, hh = ah * bh;
  const u64 mid = (ll >> 32) + (u32)lh + (u32)hl;
  return hh + (lh >> 32) + (hl >> 32) + (mid >> 32);
}
TM_FN i64 tm_smulhi64(i64 a, i64 b) {
  u64 h = tm_umulhi64((u64)a, (u64)b);
  if (a < 0) h -= (u64)b;
  if (b < 0) h -= (u64)a;
  return (i64)h;
}
TM_FN u32 tm_clz32(u32 x) { return x ? (u32)__builtin_clz(x) : 32u; }
TM_FN u64 tm_clz64(u64 x) {
  const u32 hi = (u32)(x >> 32), lo = (u32)x;
  return hi ? (u64)__builtin_clz(hi) : 32ull + tm_clz32(lo);
}

// lax.reduce_precision to E exponent and M mantissa bits, as XLA defines it: round the significand to M bits,
// nearest with ties to even (an add of half an ulp minus one, plus the last kept bit, then truncation: a carry into
// the exponent is the correct rounding); then an exponent above the reduced format's largest becomes +-inf and one
// at or below its smallest normal exponent +-0 (no subnormals); a NaN stays the NaN it was when M > 0.
template <class F, class U, int NE, int NM, int E, int M> TM_FN F tm_reduce_precision(F x) {
  static_assert(E >= 1 && E <= NE && M >= 0 && M <= NM, "reduce_precision: a narrower format only");
  U u = __builtin_bit_cast(U, x);
  const U one = 1;
  if constexpr (M < NM) {
    const U last = one << (NM - M);
    u = (u + ((last >> 1) - one) + ((u & last) >> (NM - M))) & ~(last - one);
  }
  if constexpr (E < NE) {
    const U expo = ((one << NE) - one) << NM, sign = one << (NE + NM);
    const U bias = (one << (NE - 1)) - one, rbias = (one << (E - 1)) - one;
    const U xe = u & expo;
    if (xe > ((bias + rbias) << NM)) u = (u & sign) | expo;
    else if (xe <= ((bias - rbias) << NM)) u = u & sign;
  }
  const F r = __builtin_bit_cast(F, u);
  return (M > 0 && x != x) ? x : r;
}
template <int E, int M> TM_FN float tm_reduce_precisionf(float x) {
  return tm_reduce_precision<float, u32, 8, 23, E, M>(x);
}
template <int E, int M> TM_FN double tm_reduce_precisiond(double x) {
  return tm_reduce_precision<double, u64, 11, 52, E, M>(x);
}

// lax.rem of floats: the exact remainder x - trunc(x / y) y with x's sign (C fmod; the reference's CPU target calls
// glibc's fmodf / fmod, which are exact).  NaN for a NaN operand, an infinite x or a zero y; x itself when |x| < |y|
// (an infinite y included); +-0 when |x| == |y|.  Otherwise |x| = mx 2^ex', |y| = my 2^ey' with integer
// significands, and the remainder is (mx 2^(ex' - ey') mod my) 2^ey': the reduction runs on the significands in
// integer arithmetic (8 bits per step for f32: r < my < 2^24 keeps r << 8 within 32 bits; one bit per step for
// f64, with no variable 64-bit shift), and scaling r (< my, so exact in the format) by 2^ey' rounds nothing.
TM_FN float tm_fmodf(float x, float y) {
  const u32 ux = tm_f2u(x), ax = ux & 0x7fffffffu, ay = tm_f2u(y) & 0x7fffffffu;
  if (ax >= 0x7f800000u || ay > 0x7f800000u || ay == 0u) return __builtin_nanf("");
  if (ax <= ay) return ax == ay ? tm_u2f(ux & 0x80000000u) : x;
  int ex = (int)(ax >> 23), ey = (int)(ay >> 23);
  u32 mx = ax & 0x7fffffu, my = ay & 0x7fffffu;
  if (ex) mx |= 0x800000u; else ex = 1;        // (a subnormal: exponent field 1, no hidden bit)
  if (ey) my |= 0x800000u; else ey = 1;
  u32 r = mx % my;
  for (int d = ex - ey; d > 0;) {
    const int sh = d < 8 ? d : 8;
    r = (r << sh) % my;
    d -= sh;
  }
  if (r == 0u) return tm_u2f(ux & 0x80000000u);
  const float v = __builtin_ldexpf((float)r, ey - 150);
  return (ux >> 31) ? -v : v;
}
TM_FN double tm_fmod(double x, double y) {
  const u64 ux = tm_d2u(x), ax = ux & 0x7fffffffffffffffull, ay = tm_d2u(y) & 0x7fffffffffffffffull;
  if (ax >= 0x7ff0000000000000ull || ay > 0x7ff0000000000000ull || ay == 0ull) return __builtin_nan("");
  if (ax <= ay) return ax == ay ? tm_u2d(ux & 0x8000000000000000ull) : x;
  int ex = (int)(ax >> 52), ey = (int)(ay >> 52);
  u64 mx = ax & 0xfffffffffffffull, my = ay & 0xfffffffffffffull;
  if (ex) mx |= 1ull << 52; else ex = 1;
  if (ey) my |= 1ull << 52; else ey = 1;
  while (!(mx >> 52)) { mx <<= 1; --ex; }     // normalise: both significands in [2^52, 2^53), so ex >= ey
  while (!(my >> 52)) { my <<= 1; --ey; }
  u64 r = mx >= my ? mx - my : mx;
  for (int d = ex - ey; d > 0; --d) {
    r <<= 1;
    if (r >= my) r -= my;
  }
  if (r == 0ull) return tm_u2d(ux & 0x8000000000000000ull);
  const double v = __builtin_ldexp((double)r, ey - 1075);
  return (ux >> 63) ? -v : v;
}

// float -> integer toward zero, saturating, NaN -> 0: what v_cvt_i32 / v_cvt_u32 do, written as the instruction where
// the C conversion would be undefined out of range and the guards around it cost four compares and selects
#if defined(__HIP_DEVICE_COMPILE__)
#define TM_CVT32(name, R, F, ins) \
  TM_FN R name(F x) { \
    R r; \
    asm(ins " %0, %1" : "=v"(r) : "v"(x)); \
    return r; \
  }
TM_CVT32(tm_f2i32, i32, float, "v_cvt_i32_f32")
TM_CVT32(tm_f2u32, u32, float, "v_cvt_u32_f32")
TM_CVT32(tm_d2i32, i32, double, "v_cvt_i32_f64")
TM_CVT32(tm_d2u32, u32, double, "v_cvt_u32_f64")
#else
TM_FN i32 tm_f2i32(float x) {
  return x != x ? 0 : (x <= -2147483648.0f ? (i32)0x80000000u : (x >= 2147483648.0f ? 0x7fffffff : (i32)x));
}
TM_FN u32 tm_f2u32(float x) {
  return x != x ? 0u : (x <= 0.0f ? 0u : (x >= 4294967296.0f ? 0xffffffffu : (u32)x));
}
TM_FN i32 tm_d2i32(double x) {
  return x != x ? 0 : (x <= -2147483648.0 ? (i32)0x80000000u : (x >= 2147483647.0 ? 0x7fffffff : (i32)x));
}
TM_FN u32 tm_d2u32(double x) {
  return x != x ? 0u : (x <= 0.0 ? 0u : (x >= 4294967295.0 ? 0xffffffffu : (u32)x));
}
#endif
TM_FN i64 tm_f2i64(float x) {
  return x != x ? 0 : (x <= -9223372036854775808.0f ? (i64)0x8000000000000000ull
                                                     : (x >= 9223372036854775808.0f ? 0x7fffffffffffffffll : (i64)x));
}
TM_FN i64 tm_d2i64(double x) {
  return x != x ? 0 : (x <= -9223372036854775808.0 ? (i64)0x8000000000000000ull
                                                    : (x >= 9223372036854775808.0 ? 0x7fffffffffffffffll : (i64)x));
}

// x / y in float32 with inv = 1 / y in float64: x * inv is within 2^-52 of the quotient, and a float32 quotient above
// the smallest normal is at least 2^-49 (relative) from the midpoint of two floats -- it would take a dividend of 25
// significant bits to be one -- so rounding the product is the correctly rounded quotient.  A result below that is
// divided.  Infinities, NaN and zeros of either operand pass through the product, or are divided as results of 0.
// Where y is known before the loop (a literal, a value of broadcast operands): three instructions for ~12.
TM_FN float tm_div_by(float x, float y, double inv) {
  float q = (float)((double)x * inv);
  if (__builtin_expect(__builtin_fabsf(q) < 0x1p-126f, 0)) q = x / y;
  return q;
}

// ----------------------------------------------------------------------------------------- threefry2x32
// Threefry-2x32 with 20 rounds, the parameters of Salmon, Moraes, Dror & Shaw (SC'11) that jax.random uses.  The
// key schedule is the three words ks = (k0, k1, k0 ^ k1 ^ 0x1BD11BDA); the counter is whitened with (ks0, ks1);
// then five groups of four mix rounds, the groups alternating between the rotation sets {13, 15, 26, 6} and
// {17, 29, 16, 24}, and after group g (from 0) the words gain (ks[(g + 1) % 3], ks[(g + 2) % 3] + g + 1).  A mix
// round adds the second word into the first and replaces the second by its rotation XOR the new first.  Fully
// unrolled, each round is one v_add_u32, one v_alignbit_b32 (the rotation) and one v_xor_b32 on gfx950.
TM_FN u32 tm_rotl(u32 x, int d) { return (x << d) | (x >> (32 - d)); }

TM_FN void tm_threefry(u32 k0, u32 k1, u32 c0, u32 c1, u32& o0, u32& o1) {
  const u32 ks[3] = {k0, k1, k0 ^ k1 ^ 0x1BD11BDAu};
  constexpr int rot[8] = {13, 15, 26, 6, 17, 29, 16, 24};
  u32 a = c0 + ks[0], b = c1 + ks[1];
#pragma unroll
  for (int g = 0; g < 5; ++g) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      a += b;
      b = tm_rotl(b, rot[4 * (g & 1) + r]) ^ a;
    }
    a += ks[(g + 1) % 3];
    b += ks[(g + 2) % 3] + (u32)(g + 1);
  }
  o0 = a;
  o1 = b;
}

#if defined(__HIP__) || defined(__HIPCC_RTC__)
// ============================================================================================ device only
// lane and wave helpers (wave64)
TM_DFN int tm_lane() { return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); }
TM_DFN u64 tm_ballot(bool p) { return __builtin_amdgcn_ballot_w64(p); }
TM_DFN u32 tm_rank(u64 mask) {     // set bits of mask below this lane
  return __builtin_amdgcn_mbcnt_hi((u32)(mask >> 32), __builtin_amdgcn_mbcnt_lo((u32)mask, 0u));
}
TM_DFN u32 tm_bcast_first(u32 v) { return __builtin_amdgcn_readfirstlane(v); }

// one claim of `n` consecutive items by the first active lane -> the base, broadcast to the wave
TM_DFN u64 tm_claim(u64* ctr, u32 n) {
  u64 base = 0;
  if (tm_lane() == (int)__builtin_ctzll(tm_ballot(true))) base = atomicAdd((unsigned long long*)ctr, (u64)n);
  const u32 lo = tm_bcast_first((u32)base);
  const u32 hi = tm_bcast_first((u32)(base >> 32));
  return ((u64)hi << 32) | lo;
}

// A spawned child's row in the next generation's buffer (reference _tally.py:284-300): the lanes that spawn at this
// point take consecutive tickets with one counter atomic per wave -> the lane's ticket, or -1 (it does not spawn).
TM_DFN i64 tm_qclaim(u64* ctr, bool when) {
  const u64 m = tm_ballot(when);
  if (m == 0ull) return -1;
  const u64 b = tm_claim(ctr, (u32)__builtin_popcountll(m));
  return when ? (i64)(b + tm_rank(m)) : -1;
}

// blocks of range s when n blocks are dealt out to S ranges in turn
TM_FN u64 tm_range(u64 n, u32 s, u32 S) { return n > s ? (n - s + S - 1u) / S : 0ull; }

// A Records output's slot claim (reference _tally.py:141-160): a wave takes raw slots from a private batch of TM_RB
// consecutive slots, refilled with one atomic per TM_RB slots.  The batch state (base, slots left, records appended)
// lives in the wave's LDS words, read by every active lane and written by the first, so lanes that diverged keep one
// view of it.  The lanes that append take the batch's remaining slots in rank order, then a new batch's: only the last
// batch of each wave has unused slots.
// One counter serves ~83M returning atomics/s: at 12M records (47K batches) the claims alone took 0.57 ms of 0.69.  The
// slots are S segments of whole batches (segslots each), a counter (STRIDE u64 apart) per segment; a wave claims from
// its segment and, when that is full, from the next one that is not (the segments together hold every record of the
// capacity and a batch per wave, so one is found as long as the capacity is not passed; *seg_s = S: none was).
// -> the lane's raw slot, or -1 (it does not append, or no slot is left).
#define TM_RB 256u
template <u32 S, u32 STRIDE>
TM_DFN i64 tm_rclaim(u64* ctr, volatile u64* base_s, volatile u32* left_s, volatile u64* cnt_s, volatile u32* seg_s,
                     bool when, u64 segslots) {
  const u64 m = tm_ballot(when);
  if (m == 0ull) return -1;
  const u32 n = (u32)__builtin_popcountll(m), r = tm_rank(m);
  const u32 left = *left_s;
  const u64 base = *base_s, rawcap = segslots * S;
  u64 nb = 0ull;
  u32 seg = *seg_s;
  const bool fresh = n > left;
  if (fresh) {
    nb = rawcap;
    for (u32 t = 0u; t < S && seg < S; ++t) {
      u64* const c = ctr + seg * STRIDE;
      const bool full = t != 0u && __hip_atomic_load(c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= segslots;
      const u64 b = full ? segslots : tm_claim(c, TM_RB);
      if (b < segslots) {
        nb = seg * segslots + b;
        break;
      }
      seg = seg + 1u == S ? 0u : seg + 1u;
    }
    if (S > 1u && nb == rawcap) seg = S;
  }
  const u64 s = r < left ? base + (TM_RB - left) + r : nb + (r - left);
  if (tm_lane() == (int)__builtin_ctzll(tm_ballot(true))) {
    if (fresh) {
      *base_s = nb;
      *left_s = TM_RB - (n - left);
      *seg_s = seg;
    } else {
      *left_s = left - n;
    }
    *cnt_s = *cnt_s + n;
  }
  return (when && s < rawcap) ? (i64)s : -1;
}

// A Records append inside a branch of a divergent if / else: the lanes that append take consecutive raw slots with
// one counter atomic per wave at this point; the wave's record count grows by an LDS atomic of its first lane.
// tm_rclaim's batch passes its state from one append to the next through plain LDS loads and first-lane stores,
// which is sound only where all the wave's lanes run the same code: lanes of one wave in two branches run one
// branch after the other, and the compiler, which reasons per lane (where the branches never meet), may merge the
// branches' identical trailing stores into one store after both, so the second branch would read the state from
// before the first.  An atomic add is unaffected (merged, it still adds each branch's count).
TM_DFN i64 tm_rclaim_direct(u64* ctr, u64* cnt_s, bool when, u64 rawcap) {
  const u64 m = tm_ballot(when);
  if (m == 0ull) return -1;
  const u32 n = (u32)__builtin_popcountll(m);
  const u64 b = tm_claim(ctr, n);
  if (tm_lane() == (int)__builtin_ctzll(tm_ballot(true)))
    __hip_atomic_fetch_add(cnt_s, (u64)n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  const u64 s = b + tm_rank(m);
  return (when && s < rawcap) ? (i64)s : -1;
}

// Float atomic adds that keep subnormals.  The native adds (global_atomic_add_f32 / _f64, ds_add_f32 / _f64) are
// not relied on for denormal operands or results, so an add that could meet one goes through a compare-and-swap
// loop of the IEEE add.  The native add is taken when |v| >= F, F chosen so that ulp(v) >= 2 * (the smallest
// normal) -- f32: 2^-102 (ulp >= 2^-125), f64: 2^-969 (ulp >= 2^-1021).  Then (1) a subnormal bin is below half an
// ulp of v, so IEEE's v + bin is v, as a flushed add gives; (2) with a normal bin b: if |b| <= |v| / 2 the sum is at
// least |v| / 2, normal; otherwise |b| > F / 2, so ulp(b) is at least the smallest normal and v + b is a multiple
// of it -- zero or normal.  NaN and infinities take the native add.  +-0 is skipped: a bin starts at +0 and adding
// +-0 leaves any bin as it is.  The operand is classified by its bits (sign dropped by a left shift).
template <class F, class U, U kSmall> struct TmFloatAdd {
  static TM_DFN U bits(F v) { return __builtin_bit_cast(U, v); }
  static TM_DFN bool zero(F v) { return (bits(v) << 1) == (U)0; }
  static TM_DFN bool small(F v) { return (U)(bits(v) << 1) < (U)(kSmall << 1); }
  // one IEEE add by compare-and-swap, relaxed: the tallies are read after the kernel ends
  template <int Scope> static TM_DFN void cas(F* a, F v) {
    U* const u = (U*)a;
    U seen = __hip_atomic_load(u, __ATOMIC_RELAXED, Scope);
    while (!__hip_atomic_compare_exchange_weak(u, &seen, bits(__builtin_bit_cast(F, seen) + v), __ATOMIC_RELAXED,
                                               __ATOMIC_RELAXED, Scope)) {
    }
  }
};
typedef TmFloatAdd<float, u32, 0x0c800000u> TmAddF32;                 // 2^-102
typedef TmFloatAdd<double, u64, 0x0360000000000000ull> TmAddF64;      // 2^-969
TM_DFN void tm_gadd_f32(float* a, float v) {          // a: global memory
  if (!TmAddF32::small(v)) unsafeAtomicAdd(a, v);
  else if (!TmAddF32::zero(v)) TmAddF32::cas<__HIP_MEMORY_SCOPE_AGENT>(a, v);
}
TM_DFN void tm_ladd_f32(float* a, float v) {          // a: LDS
  if (!TmAddF32::small(v)) atomicAdd(a, v);
  else if (!TmAddF32::zero(v)) TmAddF32::cas<__HIP_MEMORY_SCOPE_WORKGROUP>(a, v);
}
TM_DFN void tm_gadd_f64(double* a, double v) {
  if (!TmAddF64::small(v)) __hip_atomic_fetch_add(a, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else if (!TmAddF64::zero(v)) TmAddF64::cas<__HIP_MEMORY_SCOPE_AGENT>(a, v);
}
TM_DFN void tm_ladd_f64(double* a, double v) {
  if (!TmAddF64::small(v)) atomicAdd(a, v);
  else if (!TmAddF64::zero(v)) TmAddF64::cas<__HIP_MEMORY_SCOPE_WORKGROUP>(a, v);
}
TM_DFN void tm_gadd_i32(i32* a, i32 v) { atomicAdd(a, v); }
TM_DFN void tm_gadd_u64(u64* a, u64 v) { atomicAdd((unsigned long long*)a, (unsigned long long)v); }

#endif  // device only

// ------------------------------------------------------------- the exact f32 sum (words of 32-bit weight)
// A finite f32 v is sign * m * 2^p units of 2^-149 (m < 2^24: the significand with its hidden bit; p = max(biased
// exponent - 1, 0), in [0, 253]).  A bin is TM_XW signed int64 words, word j of weight 2^(32 j) units; its value is
// sum_j w_j 2^(32 j).  An emit adds sign * (m << (p & 31)) -- below 2^55 -- to word p >> 5 (0..7): ONE returning
// 64-bit atomic.  As each add moves a word by less than 2^55, a word leaves the int64 range only after 2^8 adds of
// the largest piece in one direction; the add that wraps it (seen from the old value the atomic returns) left the
// word 2^64 short (or over) = 2^32 units of the next word, so it adds +-2^32 to word j + 1, which may wrap in turn.
// A wrap out of the top word (a running sum beyond 2^(256 + 63) units = 2^170) cannot be kept: the emit reports it
// and the caller flags the bin, so a bin is exact or NaN.  Integer adds commute: the bin's value is the exact sum
// whatever the order of the emits (its words are not canonical; the readout is).  No 64-bit shift by a variable
// amount anywhere: pieces are built from 32-bit halves, the readout shifts by 32 only.
#define TM_XW 9
TM_FN bool tm_wraps(i64 o, i64 q) {             // does o + q leave the int64 range?
  const i64 n = (i64)((u64)o + (u64)q);
  return ((o ^ n) & (q ^ n)) < 0;
}
// add q to word j of the bin at a; `add(a, j, q)` adds and returns the word's old value (the device passes an int64
// atomic, the host checks a plain add) -> true when a carry left the top word
template <class Add> TM_FN bool tm_xadd_with(u64* a, int j, i64 q, Add add) {
  while (tm_wraps(add(a, j, q), q)) {
    if (++j == TM_XW) return true;
    q = q < 0 ? -0x100000000ll : 0x100000000ll;
  }
  return false;
}
// true: flag the bin (a non-finite emit, or a carry lost)
template <class Add> TM_FN bool tm_xemit_with(u64* a, float v, Add add) {
  const u32 b = tm_f2u(v), e = (b >> 23) & 0xffu;
  if (e == 0xffu) return true;
  const u32 m = (b & 0x7fffffu) | (e ? 0x800000u : 0u);
  if (m == 0u) return false;                    // +-0 adds nothing
  const u32 p = e ? e - 1u : 0u, s = p & 31u;
  const i64 piece = (i64)(((u64)(s ? m >> (32u - s) : 0u) << 32) | (u64)(m << s));
  return tm_xadd_with(a, (int)(p >> 5), (b >> 31) ? -piece : piece, add);
}

#if defined(__HIP__) || defined(__HIPCC_RTC__)
struct TmAtomicAdd64 {
  __device__ i64 operator()(u64* a, int j, i64 q) const {
    return (i64)atomicAdd((unsigned long long*)&a[j], (unsigned long long)q);
  }
};
TM_DFN bool tm_xadd(u64* a, int j, i64 q) { return tm_xadd_with(a, j, q, TmAtomicAdd64()); }
TM_DFN bool tm_xemit(u64* a, float v) { return tm_xemit_with(a, v, TmAtomicAdd64()); }
#endif  // device only

// Signed words w_j of weight 2^(32 j) (j < n) -> the same integer as n + 2 digits of 32 bits, two's complement
// (digit n + 1 is the sign fill); true when it is negative.  Low to high: digit j is the low half of (word j's low
// half + the carry in), the carry out the rest plus word j's high half; the carry stays below 2^31 + 2 in
// magnitude, so every step fits an int64.
TM_FN bool tm_canon_digits(const i64* w, int n, u32* d) {
  i64 c = 0;
  for (int j = 0; j < n; ++j) {
    const i64 t = (i64)(u32)(u64)w[j] + c;
    d[j] = (u32)(u64)t;
    c = (t >> 32) + (w[j] >> 32);
  }
  d[n] = (u32)(u64)c;
  d[n + 1] = c < 0 ? 0xffffffffu : 0u;
  return c < 0;
}
TM_FN void tm_negate_digits(u32* d, int n) {    // d <- 0 - d (mod 2^(32 n))
  u32 borrow = 0u;
  for (int j = 0; j < n; ++j) {
    const u32 x = d[j];
    d[j] = 0u - x - borrow;
    borrow = (x | borrow) != 0u ? 1u : 0u;
  }
}
// A magnitude of n little-endian 32-bit digits, times 2^e0, rounded once (nearest, ties to even).  The leading 32
// (f32) or 64 (f64) bits are taken with the OR of every bit below them folded into their last bit: a sticky bit
// below the format's round bit, so the one u32 -> f32 (u64 -> f64) conversion rounds the whole value correctly; the
// power-of-two scaling after it is exact (a result below the smallest normal has at most 23 / 52 significant
// bits and was not rounded).
TM_FN float tm_digits_f32(const u32* d, int n, int e0) {
  int t = n - 1;
  while (t >= 0 && d[t] == 0u) --t;
  if (t < 0) return 0.0f;
  const u32 z = (u32)__builtin_clz(d[t]), n1 = t >= 1 ? d[t - 1] : 0u;
  const u32 lead = z ? (d[t] << z) | (n1 >> (32u - z)) : d[t];
  bool st = (z ? n1 << z : n1) != 0u;
  for (int j = t - 2; j >= 0; --j) st = st || d[j] != 0u;
  return __builtin_ldexpf((float)(lead | (st ? 1u : 0u)), 32 * t - (int)z + e0);
}
TM_FN double tm_digits_f64(const u32* d, int n, int e0) {
  int t = n - 1;
  while (t >= 0 && d[t] == 0u) --t;
  if (t < 0) return 0.0;
  const u32 z = (u32)__builtin_clz(d[t]), n1 = t >= 1 ? d[t - 1] : 0u, n2 = t >= 2 ? d[t - 2] : 0u;
  const u32 hi = z ? (d[t] << z) | (n1 >> (32u - z)) : d[t];
  const u32 lo = z ? (n1 << z) | (n2 >> (32u - z)) : n1;
  bool st = (z ? n2 << z : n2) != 0u;
  for (int j = t - 3; j >= 0; --j) st = st || d[j] != 0u;
  return __builtin_ldexp((double)(((u64)hi << 32) | (u64)(lo | (st ? 1u : 0u))), 32 * (t - 1) - (int)z + e0);
}
// the exact readout: the bin's words rounded once to f32; *bad when the total is beyond f32 (host + device: the host
// build checks it against Python integers)
TM_FN float tm_xread(const u64* a, bool* bad) {
  u32 d[TM_XW + 2];
  const bool neg = tm_canon_digits((const i64*)a, TM_XW, d);
  if (neg) tm_negate_digits(d, TM_XW + 2);
  const float f = tm_digits_f32(d, TM_XW + 2, -149);
  if (!(f <= 3.4028234663852886e38f)) *bad = true;
  return neg ? -f : f;
}

// the same words rounded once to f64 (their range, below 2^320 units of 2^-149, is within f64's)
TM_FN double tm_xread_f64(const u64* a) {
  u32 d[TM_XW + 2];
  const bool neg = tm_canon_digits((const i64*)a, TM_XW, d);
  if (neg) tm_negate_digits(d, TM_XW + 2);
  const double f = tm_digits_f64(d, TM_XW + 2, -149);
  return neg ? -f : f;
}

// --------------------------------------------------------------------- the scaled fixed-point sum (WIDE)
// A bin is an int64 low word (wrapping) and an i32 word counting its signed wraps: an add of q that takes the low
// word out of the int64 range (tm_wraps on the old value the atomic returns) adds sign(q) to the count, so the
// exact total low + count * 2^64 does not depend on the order of the adds.  An emit adds round(v * scale) (nearest,
// ties to even); |v * scale| >= 9.2e18 is not representable: the emit is dropped and flags its bin (reference
// kernel.py:844-869, _api.py:55-84).
// round(v * scale) -> *q; false when not representable
TM_FN bool tm_wvalue(double v, double scale, i64* q) {
  const double x = v * scale;
  if (!(__builtin_fabs(x) < 9.2e18)) return false;
  *q = (i64)__builtin_rint(x);
  return true;
}
// low + count * 2^64 rounded once to double (nearest, ties to even): the int64 conversion alone when nothing wrapped,
// else the digits of the 96-bit total
TM_FN double tm_wide_f64(u64 lo, i32 c) {
  if (c == 0) return (double)(i64)lo;
  const i64 w[3] = {(i64)lo, 0, (i64)c};
  u32 d[5];
  const bool neg = tm_canon_digits(w, 3, d);
  if (neg) tm_negate_digits(d, 5);
  const double m = tm_digits_f64(d, 5, 0);
  return neg ? -m : m;
}
TM_FN u64 tm_d2u64(double x) {
  return x != x ? 0ull : (x <= 0.0 ? 0ull : (x >= 18446744073709551616.0 ? ~0ull : (u64)x));
}

#if defined(__HIP__) || defined(__HIPCC_RTC__)
TM_DFN void tm_wadd(u64* lo, i32* c, i64 q) {
  const i64 o = (i64)atomicAdd((unsigned long long*)lo, (unsigned long long)q);
  if (tm_wraps(o, q)) atomicAdd(c, q < 0 ? -1 : 1);
}
// one emit of v: false when v * scale is not representable (the caller counts it and flags the bin)
TM_DFN bool tm_wemit(u64* lo, i32* c, double v, double scale) {
  i64 q = 0;
  if (!tm_wvalue(v, scale, &q)) return false;
  if (q != 0) tm_wadd(lo, c, q);
  return true;
}
#endif  // device only
