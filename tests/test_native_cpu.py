"""CPU checks of the native pieces: the C-ABI library exports what include/tallymap_rocm.h declares, the device
runtime's exact accumulator and tm_libm.h agree with Python integers / glibc on the host, generated kernels compile
for gfx950 through the product's hipRTC path."""
import ctypes
import os
import re
import subprocess
from fractions import Fraction

import numpy as np
import pytest

from oracle import exact as X

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _build(src, out, *flags):
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-fopenmp", *flags, "-o", out,
                    os.path.join(ROOT, src), "-lm"], check=True)
    return out


def test_cabi_exports_every_declared_symbol():
    hdr = open(os.path.join(ROOT, "include", "tallymap_rocm.h")).read()
    hdr = re.sub(r"/\*.*?\*/", "", hdr, flags=re.S)          # declarations only, not the comments
    names = sorted(set(re.findall(r"^[a-z][\w \*]*?\b((?:tm|tallymap)_[a-z_]+)\(", hdr, flags=re.M)))
    assert {"tm_init", "tm_compile", "tm_register", "tm_launch", "tm_kernel_info", "tm_last_error",
            "tm_free", "tallymap_register", "tallymap_kernel_info"} <= set(names)
    from tallymap_amd.backend import compile as Cm
    lib = Cm.load_shim()
    for n in names:
        assert hasattr(lib, n), n


def test_cabi_errors_without_init():
    from tallymap_amd.backend import compile as Cm
    lib = Cm.load_shim()
    lib.tm_last_error.restype = ctypes.c_char_p
    # tm_register copies; an empty image is refused with a message
    lib.tm_register.argtypes = [ctypes.c_longlong, ctypes.c_char_p, ctypes.c_size_t, ctypes.c_char_p]
    assert lib.tm_register(1, b"", 0, b"x") != 0
    assert b"empty image" in lib.tm_last_error()


def test_reference_registry_exports_keep_reference_conventions():
    """tallymap_register / tallymap_kernel_info as the reference's compile.py binds them (compile.py:215-237):
    register returns 0 (an empty image registers nothing); kernel_info returns 0 until the program has been launched
    -- here no runtime is bound and nothing is loaded, so 0, and out[] is left alone."""
    from tallymap_amd.backend import compile as Cm
    lib = Cm.load_shim()
    lib.tallymap_register.argtypes = [ctypes.c_int64, ctypes.c_char_p, ctypes.c_size_t, ctypes.c_char_p]
    lib.tallymap_kernel_info.argtypes = [ctypes.c_int64, ctypes.POINTER(ctypes.c_longlong)]
    assert lib.tallymap_register(7, b"", 0, b"x") == 0
    assert lib.tallymap_register(8, b"not a code object", 17, None) == 0
    out = (ctypes.c_longlong * 7)(*([-5] * 7))
    assert lib.tallymap_kernel_info(8, out) == 0
    assert lib.tallymap_kernel_info(12345, out) == 0
    assert list(out) == [-5] * 7


@pytest.fixture(scope="module")
def xsum(tmp_path_factory):
    return _build("tests/native/xsum_check.cc", str(tmp_path_factory.mktemp("n") / "xsum_check"))


def _xrun(exe, v):
    inp = "\n".join("%08x" % x for x in np.asarray(v, np.float32).view(np.uint32))
    out = subprocess.run([exe], input=inp, capture_output=True, text=True, check=True).stdout.split()
    return np.uint32(int(out[0], 16)).view(np.float32), out[1] == "1"


def test_exact_accumulator_matches_python_integers(xsum):
    rng = np.random.default_rng(11)
    cases = [rng.standard_normal(3000).astype(np.float32),
             (rng.standard_normal(300) * 1e37).astype(np.float32),
             np.concatenate([np.full(5000, 3.4e38), np.full(5000, -3.4e38), [1.0]]).astype(np.float32),
             np.array([1e-45] * 1000 + [-3e-45] * 10, np.float32),
             np.array([1.0, 2 ** -24, 2 ** -24], np.float32),
             np.array([2.0 ** 100, 1.0, -2.0 ** 100], np.float32),
             rng.permutation(np.concatenate([rng.standard_normal(500) * 10.0 ** rng.integers(-40, 38, 500),
                                             -rng.standard_normal(500)])).astype(np.float32)]
    for v in cases:
        g, bad = _xrun(xsum, v)
        w, wbad = X.exact_sum(v)
        assert bad == wbad
        if not bad:
            assert g.view(np.uint32) == w.view(np.uint32)
    # order independence: a permutation gives the same bits
    v = cases[-1]
    assert _xrun(xsum, v)[0].view(np.uint32) == _xrun(xsum, v[::-1].copy())[0].view(np.uint32)
    # a non-finite emit or a total beyond f32 flags the bin
    assert _xrun(xsum, np.array([1.0, np.inf], np.float32))[1]
    assert _xrun(xsum, np.full(5000, 3.4e38, np.float32))[1]


def _xwords(exe, w):
    inp = " ".join("%016x" % (int(x) & (2 ** 64 - 1)) for x in w)
    out = subprocess.run([exe, "words"], input=inp, capture_output=True, text=True, check=True).stdout.split()
    return np.uint32(int(out[0], 16)).view(np.float32), out[1] == "1", np.uint64(int(out[2], 16)).view(np.float64)


def test_exact_accumulator_carries_between_words(xsum):
    """Emits of the largest piece a word takes (significand all ones at a bit offset of 31 within the word) wrap the
    int64 word every ~256 adds in one direction: the carries into the next word keep the total exact, through a run
    up and back down, at each word position that emits reach."""
    for e in (32, 64, 96, 128, 160, 192, 224, 254):
        v = np.uint32((e << 23) | 0x7FFFFF).view(np.float32)
        w = np.uint32((e << 23) | 0x7FFF01).view(np.float32)
        seq = np.concatenate([np.full(1500, v), np.full(700, -w), [np.float32(1.5)], np.full(1490, -v)]).astype(
            np.float32)
        g, bad = _xrun(xsum, seq)
        want, wbad = X.exact_sum(seq)
        assert bad == wbad, e
        if not bad:
            assert g.view(np.uint32) == want.view(np.uint32), (e, g, want)


def test_exact_readout_of_arbitrary_words(xsum):
    """tm_xread on words that are not canonical (any int64 per word, as concurrent adds and carries leave them):
    the correctly rounded f32 of sum_j w_j 2^(32 j) units of 2^-149 -- Python integers -- with the flag exactly when
    that total is beyond f32, and tm_xread_f64 its correctly rounded f64.  Covers signs that differ across words, totals near zero, ties and the top word."""
    rng = np.random.default_rng(5)
    lim = 2 ** 63
    cases = [[0] * 9, [1] + [0] * 8, [-1] + [0] * 8, [0] * 8 + [-1], [lim - 1] * 9, [-lim] * 9,
             [2 ** 40, -2 ** 8] + [0] * 7, [-(2 ** 32)] + [1] + [0] * 7,            # cancels to exactly 0
             [2 ** 31 + 2 ** 7] + [0] * 8, [2 ** 31 + 3 * 2 ** 7] + [0] * 8,       # ties, even and odd
             [0, 0, 0, 0, 0, 0, 0, 2 ** 22 - 1, 0], [0, 0, 0, 0, 0, 0, 0, 2 ** 22, 0]]
    for _ in range(300):
        w = [int(x) for x in rng.integers(-lim, lim, 9, dtype=np.int64)]
        k = int(rng.integers(1, 9))
        for j in range(k, 9):                                  # totals of every size, not only huge ones
            w[j] = int(rng.integers(-3, 4)) if rng.random() < 0.5 else 0
        cases.append(w)
    for w in cases:
        total = sum(int(x) << (32 * j) for j, x in enumerate(w))
        want = X.round_units(total)
        g, bad, d = _xwords(xsum, w)
        assert d == float(Fraction(total, 2 ** 149)) and (d != 0) == (total != 0), (w, d)
        assert bad == (want is None), (w, g)
        if want is not None:
            assert g.view(np.uint32) == want.view(np.uint32), (w, g, want)


def test_wide_readout_rounds_once(xsum):
    """tm_wide_f64(low, count) = low (as int64) + count * 2^64, rounded once to double (Python's int -> float is
    correctly rounded): random words and counts, counts 0 and +-1 near the wrap, ties at 2^64 + small offsets."""
    rng = np.random.default_rng(9)
    pairs = [(0, 0), (2 ** 63, 0), (2 ** 63 - 1, 0), (0, 1), (0, -1), (2 ** 64 - 1, -1), (2 ** 63, -1),
             (2 ** 63, 1), (2 ** 11, 1), (2 ** 11 + 1, 1), (3 * 2 ** 11, 1), (2 ** 64 - 2 ** 11, -1),
             (1, 2 ** 31 - 1), (2 ** 64 - 1, -2 ** 31), (0, -2 ** 31)]
    for _ in range(2000):
        pairs.append((int(rng.integers(0, 2 ** 64, dtype=np.uint64)), int(rng.integers(-2 ** 31, 2 ** 31))))
        pairs.append((int(rng.integers(0, 2 ** 64, dtype=np.uint64)), int(rng.integers(-3, 4))))
    inp = "\n".join("%016x %d" % (lo, c) for lo, c in pairs)
    out = subprocess.run([xsum, "wide"], input=inp, capture_output=True, text=True, check=True).stdout.split()
    assert len(out) == len(pairs)
    for (lo, c), o in zip(pairs, out):
        slo = lo - 2 ** 64 if lo >= 2 ** 63 else lo
        want = float(slo + c * 2 ** 64)
        assert int(o, 16) == int(np.float64(want).view(np.uint64)), (lo, c, o, want)


@pytest.fixture(scope="module")
def libm(tmp_path_factory):
    return _build("tests/native/libm_check.cc", str(tmp_path_factory.mktemp("n") / "libm_check"))


def test_erfinv_matches_glibc_reference_on_every_normal_argument(libm):
    """tm_erfinvf (device) vs the reference CPU target's formula with glibc's log, over all 2^23 arguments that
    jax.random.normal passes to erf_inv: bitwise."""
    r = subprocess.run([libm, "erfinv_normal"], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
    assert ", 0 f32 mismatches" in r.stdout


def test_erfinv_matches_reference_on_all_f32_arguments(libm):
    """tm_erfinvf (a division-free table log, fused multiply-adds) vs the reference formula (glibc log, separate
    multiplies and adds) on every 5th f32 in (-1, 1), bitwise (stride 1 -- all 2,130,706,430 -- gives 0 mismatches
    too)."""
    r = subprocess.run([libm, "erfinv_all", "5"], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
    assert ", 0 f32 mismatches" in r.stdout


def test_erfinv_log_absolute_error(libm):
    """tm_log_erfinv's error on erf_inv's domain t in [2^-24, 1] stays below 2^-51 max(1, |log t|)."""
    r = subprocess.run([libm, "log", "2000000", "5"], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


@pytest.mark.parametrize("fn", ["logf", "expf", "sinf", "cosf", "sincosf_s", "sincosf_c", "atanf", "exp2f", "log2f", "expm1f", "log1pf",
                                "tanhf", "logistic", "asinf", "acosf", "sinhf", "coshf", "atanhf", "asinhf",
                                "acoshf", "erff", "erfcf", "tanf", "lgammaf"])
def test_f32_libm_bitwise_equal_to_glibc(libm, fn):
    """tm_libm.h's float functions against this host's glibc on EVERY one of the 2^32 bit patterns (OpenMP over the
    host's cores): 0 mismatches.  logistic is the reference CPU target's 1 / (1 + expf(-x)); lgammaf calls lgammaf
    itself on (-15, -2) (glibc's own lgamma_negf there; the device library on the GPU), so it is pinned outside.
    glibc's lgammaf is slow enough that the suite takes every 7th pattern for it (613,566,757 arguments: every
    sign, exponent and branch); `libm_check f32 lgammaf 1 0` runs all 2^32, also with 0 mismatches."""
    stride = 7 if fn == "lgammaf" else 1
    r = subprocess.run([libm, "f32", fn, str(stride), "0"], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    assert f"{fn}: {-(-(1 << 32) // stride)} arguments, 0 mismatches" in r.stdout, r.stdout


def test_powf_bitwise_equal_to_glibc(libm):
    """tm_powf against glibc's powf: 40M pairs (random bit patterns; x near 1 with |y| up to 1e7; moderate x with
    integer and non-integer y, both signs) and every pair of a grid of special values (zeros, infinities, NaN,
    subnormals, +-1, overflow and underflow edges): 0 mismatches."""
    r = subprocess.run([libm, "powf", "10000000", "3"], capture_output=True, text=True)
    assert r.returncode == 0 and ", 0 mismatches" in r.stdout, r.stdout


def test_atan2f_bitwise_equal_to_glibc(libm):
    r = subprocess.run([libm, "atan2", "2000000", "11"], capture_output=True, text=True)
    assert r.returncode == 0 and ", 0 mismatches" in r.stdout, r.stdout


@pytest.mark.parametrize("fn", ["exp", "exp2", "log", "log2", "expm1", "log1p", "tanh", "sinh", "cosh", "atanh",
                                "asinh", "acosh", "erf", "erfc", "erfinv", "lgamma"])
def test_f64_libm_bitwise_equal_to_glibc(libm, fn):
    """tm_libm.h's float64 restatements against this host's glibc on 4M arguments (random bit patterns of every
    class, the working range, magnitudes 2^-60 .. 2^20, the bands around every branch boundary of the code: a
    boundary's high word +- 2 with random low words) and 40 special values (zeros, infinities, NaN, subnormals, the
    overflow and underflow thresholds): 0 mismatches.  (20M per function and seeds 1..3 also give 0.)"""
    r = subprocess.run([libm, "f64", fn, "4000000", "17"], capture_output=True, text=True)
    assert r.returncode == 0 and f"f64 {fn}: 4000000 samples, 0 mismatches; 40 special values, 0 mismatches" \
        in r.stdout, r.stdout + r.stderr


def test_f64_pow_bitwise_equal_to_glibc(libm):
    """tm_pow against glibc's pow: 6M pairs (random bit patterns; |x| in [2^-20, 2^20) of both signs with integer and
    non-integer y; x within 2^-16 of 1 with |y| up to 2^40; results near the subnormal boundary and near overflow,
    both signs of the base) and every pair of a grid of 34 special values: 0 mismatches.  (60M pairs also give 0.)"""
    r = subprocess.run([libm, "pow", "6000000", "5"], capture_output=True, text=True)
    assert r.returncode == 0 and "f64 pow: 6000000 pairs, 0 mismatches; 1156 special pairs, 0 mismatches" \
        in r.stdout, r.stdout + r.stderr


def _f64_table(fn, name):
    """the hex-float words of the local table `name` inside tm_libm.h's function `fn`"""
    src = open(os.path.join(ROOT, "tallymap_amd", "csrc", "tm_libm.h")).read()
    body = src[src.index(f"TM_FN double {fn}("):]
    body = body[body.index("{", body.index(f"{name}[")):]
    body = body[:body.index("};")]
    return [float.fromhex(w) for w in re.findall(r"-?0x[0-9a-f.]+p[-+]?\d+", body)]


def test_pow_log_table_equals_its_definition():
    """tm_pow_log's 128 entries: c near the center of subinterval i of [0x1.69555p-1, 0x1.69555p0) (128 equal steps of
    the bit pattern), 1/c = round(128 / center) / 128 below 1 else round(256 / center) / 256, logc = log c rounded to
    a multiple of 2^-43, logctail = log c - logc rounded to double: recomputed at 60 digits."""
    import struct
    import mpmath
    mpmath.mp.dps = 60
    w = _f64_table("tm_pow_log", "T")
    assert len(w) == 384
    off = 0x3fe6955500000000
    d = lambda b: struct.unpack("<d", struct.pack("<Q", b))[0]
    for i in range(128):
        center = (mpmath.mpf(d(off + (i << 45))) + mpmath.mpf(d(off + ((i + 1) << 45)))) / 2
        invc = mpmath.nint(128 / center) / 128 if center < 1 else mpmath.nint(256 / center) / 256
        lc = -mpmath.log(invc)
        logc = mpmath.nint(lc * 2 ** 43) / 2 ** 43
        assert w[3 * i] == float(invc) and w[3 * i + 1] == float(logc), i
        assert w[3 * i + 2] == float(lc - logc), i


@pytest.mark.parametrize("fn,n,grid,bound", [("tm_log", 128, 43, 66), ("tm_log2", 64, 42, 62)])
def test_log_tables_keep_their_rule(fn, n, grid, bound):
    """tm_log's and tm_log2's tables, the entries found by search: invc = 1/c with c inside its subinterval (of
    [0x1.6p-1, 0x1.6p0), n equal steps of the bit pattern), logc = log c (log2 c) rounded to double and a multiple of
    2^-grid, |log c - logc| below 2^-bound; log2's chi + clo = c (chi = c rounded, clo = c - chi rounded).  The
    search found about 250 (log) and 32,000 (log2) candidates per subinterval under this rule; agreement with glibc
    on the arguments (the f64 tests above) is what singles out each entry."""
    import struct
    import mpmath
    mpmath.mp.dps = 60
    w = _f64_table(fn, "T")
    per = 2 if fn == "tm_log" else 4
    assert len(w) == n * per
    off, step = 0x3fe6000000000000, 52 - (n.bit_length() - 1)
    d = lambda b: struct.unpack("<d", struct.pack("<Q", b))[0]
    for i in range(n):
        invc, logc = mpmath.mpf(w[per * i]), w[per * i + 1]
        c = 1 / invc
        assert d(off + (i << step)) <= c < d(off + ((i + 1) << step)), i
        lc = -mpmath.log(invc) if fn == "tm_log" else -mpmath.log(invc, 2)
        assert float(lc) == logc and logc * 2 ** grid == int(logc * 2 ** grid), i
        assert abs(lc - logc) < mpmath.mpf(2) ** -bound, i
        if per == 4:
            assert w[4 * i + 2] == float(c) and w[4 * i + 3] == float(c - mpmath.mpf(w[4 * i + 2])), i


def test_exp_table_equals_its_definition():
    """tm_exp_pair's 128 entries are (T, H - k 2^45) with H = 2^(k/128) rounded to double and T = (2^(k/128) - H) / H
    rounded to double: recomputed here at 80 decimal digits and compared with the words in tm_libm.h."""
    import struct
    from decimal import Decimal, getcontext
    src = open(os.path.join(ROOT, "tallymap_amd", "csrc", "tm_libm.h")).read()
    body = src[src.index("TM_FN void tm_exp_pair"):]
    body = body[body.index("{", body.index("E[256]")):body.index("};")]
    words = [int(w, 16) for w in re.findall(r"0x([0-9a-f]{16})ull", body)]
    assert len(words) == 256
    getcontext().prec = 80
    for k in range(128):
        v = Decimal(2) ** (Decimal(k) / 128)
        h = float(v)
        t = float((v - Decimal(h)) / Decimal(h))
        bits = lambda d: struct.unpack("<Q", struct.pack("<d", d))[0]
        assert words[2 * k] == bits(t), k
        assert words[2 * k + 1] == (bits(h) - (k << 45)) % (1 << 64), k


def test_generated_modules_compile_for_gfx950():
    """the forward modules of configs 1 and 2 compile through the product's hipRTC path (no GPU needed)."""
    from tallymap_amd import _core as C
    from tallymap_amd import configs
    from tallymap_amd._api import build_program
    from tallymap_amd.backend import compile as Cm
    from tallymap_amd.backend import kernel as K
    for name in ("c1", "c2"):
        cfg = configs.CONFIGS[name]
        args = getattr(configs, f"{name}_inputs")(8)
        axes = cfg["in_axes"]
        pav = [C.AVal(np.shape(a)[1:], np.asarray(a).dtype) for a, x in zip(args, axes) if x == 0]
        bav = [C.AVal(np.shape(a), np.asarray(a).dtype) for a, x in zip(args, axes) if x is None]
        prog, _ = build_program(cfg["item"], cfg["outputs"], axes, pav, bav, cfg["max_steps"])
        src, L = K.build(prog)
        assert L.mode == "step"
        img = Cm.code_object(src)
        assert img[:4] == b"\x7fELF" or len(img) > 1000


def test_machine_key_follows_the_instructions_not_the_source():
    """compile.machine_key (what bench.py keys its recorded counters by): a source that differs only by an unused
    device helper compiles to the same key; a different instruction gives another."""
    from tallymap_amd.backend import compile as Cm
    from tallymap_amd.backend import valu
    a = valu.source("v_add_u32", 64)
    b = a.replace("extern \"C\" __global__ void tm_zero",
                  "__device__ __forceinline__ unsigned tm_unused_helper(unsigned x) { return x * 3u; }\n"
                  "extern \"C\" __global__ void tm_zero")
    assert a != b and Cm._key(a) != Cm._key(b)
    ka, kb = Cm.machine_key(Cm.code_object(a)), Cm.machine_key(Cm.code_object(b))
    kc = Cm.machine_key(Cm.code_object(valu.source("v_xor_b32", 64)))
    assert ka == kb and ka != kc


def test_shift64_helpers_match_native_shifts(tmp_path):
    """tm_shl64 / tm_shr64 / tm_sar64 (32-bit halves) equal the host's 64-bit shifts for every amount 0..63."""
    exe = _build("tests/native/shift64_check.cc", str(tmp_path / "shift64_check"))
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "0 mismatches", r.stdout


def test_int64_to_float32_without_64bit_shifts(tmp_path):
    """tm_u64f / tm_i64f (32 leading bits from 32-bit halves, a sticky bit, one u32 -> f32 rounding) equal the host's
    int64 / uint64 -> float32 conversions on edge values, ties and their neighbours at every exponent, and 2M
    pseudo-random values at every magnitude."""
    exe = _build("tests/native/i64f_check.cc", str(tmp_path / "i64f_check"))
    r = subprocess.run([exe], capture_output=True, text=True)
    bad, n = map(int, r.stdout.split())
    assert r.returncode == 0 and bad == 0 and n > 2_000_000, r.stdout


def test_shift_hazard_scanner_flags_only_block_end_amount_registers():
    from tallymap_amd.backend import compile as Cm
    dis = "\n".join([
        "0000000000002e00 <tm_main>:",
        "\tv_lshlrev_b64 v[18:19], v39, v[4:5]                        // 000000003564: D28F0012 00020927",
        "\tv_lshrrev_b64 v[18:19], v40, v[4:5]                        // 000000003764: D2900012 00020912",
        "\tv_ashrrev_i64 v[2:3], v7, v[2:3]",
        "\tv_lshlrev_b64 v[2:3], 7, v[2:3]",
        "\tv_lshrrev_b32_e32 v15, 7, v15",
        "0000000000003e00 <tm_post>:",
        "\tv_lshrrev_b64 v[4:5], v15, v[4:5]"])
    assert Cm.shift_hazards_in(dis) == [("tm_main", "v_lshlrev_b64 v[18:19], v39, v[4:5]"),
                                        ("tm_main", "v_ashrrev_i64 v[2:3], v7, v[2:3]"),
                                        ("tm_post", "v_lshrrev_b64 v[4:5], v15, v[4:5]")]


def test_exact_kernels_compile_without_shift_hazards():
    """the exact-sum kernels of every schedule and accumulator placement compile with no 64-bit shift by a VGPR
    amount at all (the case gfx950 gets wrong when the amount lands in v(8k+7))."""
    from tallymap_amd import _core as C
    from tallymap_amd import configs
    from tallymap_amd._api import build_program
    from tallymap_amd.backend import compile as Cm
    from tallymap_amd.backend import kernel as K
    import tallymap_amd as tm
    if Cm.objdump() is None:
        pytest.skip("llvm-objdump is not installed")
    args = configs.c1_inputs(8)
    axes = (0, 0, None)
    pav = [C.AVal(np.shape(a)[1:], np.asarray(a).dtype) for a, x in zip(args, axes) if x == 0]
    bav = [C.AVal(np.shape(a), np.asarray(a).dtype) for a, x in zip(args, axes) if x is None]
    prog, _ = build_program(configs.C1["item"], {"hist": tm.Sum((16,), fixed_point=True)}, axes, pav, bav, 100)
    saved = K.LDS_BYTES
    try:
        for lds in (saved, 0):
            K.LDS_BYTES = lds
            for o in (dict(schedule="item"), dict(), dict(refill=3), dict(block=64), dict(compact=0)):
                src, _ = K.build(prog, **o)
                img = Cm.code_object(src)
                d = subprocess.run([Cm.objdump(), "-d", "--mcpu=gfx950", "/dev/stdin"], input=img,
                                   capture_output=True, check=True).stdout.decode()
                assert not re.search(r"v_(lshlrev_b64|lshrrev_b64|ashrrev_i64)\S*\s+v\[\d+:\d+\],\s*v\d+,", d), o
    finally:
        K.LDS_BYTES = saved


def test_util_module_compiles_for_gfx950():
    """the spawn paths' scan and scatter module builds with hipRTC and holds its entries."""
    from tallymap_amd.backend import compile as Cm
    from tallymap_amd.backend import util
    src = util._source()
    for e in ("tm_xscan_local", "tm_xscan_top", "tm_xscan_add", "tm_tree_scatter", "tm_tree_scatter_b"):
        assert f"void __launch_bounds__" in src and e in src
    assert len(Cm.code_object(src, name="tm_util.hip")) > 0


def test_common_paths_are_defined_for_rare_arguments(tmp_path):
    """the functions whose common path every argument takes (a rare one's result is replaced afterwards) overflow no
    signed integer on it: undefined behaviour reported by the compiler's own checks, over all exponents."""
    exe = _build("tests/native/libm_check.cc", str(tmp_path / "libm_ub"), "-fsanitize=undefined",
                 "-fno-sanitize-recover=undefined")
    for fn in ("logf", "sinf", "cosf", "sincosf_s", "sincosf_c", "atanf"):
        r = subprocess.run([exe, "f32", fn, "400009", "7"], capture_output=True, text=True)
        assert r.returncode == 0 and " 0 mismatches" in r.stdout, (fn, r.stdout, r.stderr[-300:])


def test_fmod_matches_glibc(tmp_path):
    """lax.rem of floats (tm_fmodf / tm_fmod): bitwise glibc's exact fmodf / fmod on special values and 8M
    pseudo-random pairs across the exponent range, subnormals included."""
    exe = _build("tests/native/fmod_check.cc", str(tmp_path / "fmod_check"))
    r = subprocess.run([exe, "4000000"], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
    bad, tot = map(int, r.stdout.split()[-2:])
    assert bad == 0 and tot > 8_000_000


def test_division_by_a_reciprocal_is_the_division(tmp_path):
    """tm_div_by: bitwise x / y on special values, random pairs, quotients next to midpoints and subnormal ones."""
    exe = _build("tests/native/div_check.cc", str(tmp_path / "div_check"))
    r = subprocess.run([exe, "8000000"], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
    bad, tot = map(int, r.stdout.split()[-2:])
    assert bad == 0 and tot > 32_000_000


def test_uniform_derived_arguments_match_glibc(libm):
    """every argument the configs hand to logf / sinf / cosf from a uniform draw -- logf(1 - u), sinf / cosf(2 pi u)
    for all 2^23 values jax.random.uniform produces -- bitwise glibc's results."""
    r = subprocess.run([libm, "uniform"], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
    assert f"uniform: {3 * 8388608} arguments, 0 mismatches" in r.stdout


def test_shift_hazard_check_refuses_without_objdump(monkeypatch):
    """with no llvm-objdump the shift-hazard check refuses the code object instead of passing it unchecked."""
    from tallymap_amd.backend import compile as Cm
    monkeypatch.setattr(Cm, "objdump", lambda: None)
    with pytest.raises(Cm.BackendError, match="refusing"):
        Cm.shift_hazards(b"\x7fELF")

