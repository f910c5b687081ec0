"""Float sums privatised in LDS: held in float64 with up to 16 copies of a bin while they fit, in float32 above, at
the numbers of bins where the copies and the format change, against the exact sums."""
import math

import numpy as np
import pytest

import tallymap_amd as tm
from tallymap_amd import numpy as jnp

pytestmark = pytest.mark.gpu


def _run(b, v, S, dtype):
    def item(t, b, v):
        t = t.add("a", b, v if dtype == np.float32 else v.astype(jnp.float64))
        return t.add("n", b, 1.0)
    f = tm.vmap(item, outputs={"a": tm.Sum((S,), dtype=dtype), "n": tm.Sum((S,))}, in_axes=(0, 0))
    r = f(b, v)
    return r.outputs["a"].cpu().numpy(), r.outputs["n"].cpu().numpy(), int(r.stats["dropped_emits"].item())


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("S", [1, 2, 3, 15, 16, 17, 63, 64, 65, 255, 256, 257, 511, 1024, 1025, 4096])
def test_sums_over_bin_counts(S, dtype):
    """one workgroup (256 items) and many (70,001); mixed signs and magnitudes, subnormals, indices out of range."""
    rng = np.random.default_rng(S)
    for n in (256, 70_001):
        b = rng.integers(-1, S + 1, n).astype(np.int32)
        v = (rng.standard_normal(n) * 10.0 ** rng.integers(-3, 4, n)).astype(np.float32)
        v[::7] = np.float32(1.4e-45) * rng.integers(1, 1000, len(v[::7]))
        got, cnt, dropped = _run(b, v, S, dtype)
        ok = (b >= 0) & (b < S)
        assert dropped == 2 * int((~ok).sum())
        assert np.array_equal(cnt, np.bincount(b[ok], minlength=S).astype(np.float32))
        # a bin is at most `parts` workgroup totals, each a sum in float64 (or, past 1,024 bins, in float32: one
        # rounding per add) rounded once to float32 and added in float32: (adds or parts + 1) roundings of at most
        # 2^-24 of the sum of magnitudes each
        eps = 2.0 ** -24 if dtype == np.float32 else 2.0 ** -53
        parts = -(-n // 256)
        for i in range(S):
            x = v[ok & (b == i)].astype(np.float64)
            k = len(x) if dtype == np.float64 or S > 1024 else min(parts, len(x))
            bound = (k + 1) * eps * float(np.abs(x).sum()) + 1e-45
            assert abs(float(got[i]) - math.fsum(x)) <= bound, (S, n, i, got[i], math.fsum(x))


def test_non_finite_values_reach_their_bin_only():
    b = np.arange(32, dtype=np.int32) % 4
    v = np.ones(32, np.float32)
    v[0], v[1], v[2], v[6] = np.nan, np.inf, np.inf, -np.inf
    got, _, _ = _run(b, v, 4, np.float32)
    assert np.isnan(got[0]) and got[1] == np.inf and np.isnan(got[2]) and got[3] == 8.0


@pytest.mark.parametrize("S, n", [(2, 40), (16, 1), (16, 3), (16, 40), (16, 84), (1024, 19)])
def test_sums_of_many_constants(S, n):
    """a counter per constant in LDS: copies of it while the budget lasts, one above, and (1,024 bins of 19 constants)
    no float64 bins beside them.  Multiples of 1/128 below 2^17: every sum is exact in float32."""
    def item(t, b):
        for j in range(n):
            t = t.add("h", (b + 7 * j) % S, np.float32(1.0 + j / 128.0))
        return t
    b = np.random.default_rng(S + n).integers(0, S, 1000).astype(np.int32)
    want = sum(np.bincount((b + 7 * j) % S, minlength=S) * (1.0 + j / 128.0) for j in range(n))
    got = tm.vmap(item, outputs={"h": tm.Sum((S,))}, in_axes=(0,))(b).outputs["h"].cpu().numpy()
    assert np.array_equal(got, want.astype(np.float32))
