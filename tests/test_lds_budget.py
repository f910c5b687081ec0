"""The LDS a workgroup of the item loop takes: the copies of bins and constant counters come out of one budget, and a
program that fits a CU without copies and float64 bins is never refused for them."""
import numpy as np
import pytest

from tallymap_amd import _core as C
from tallymap_amd import numpy as jnp
from tallymap_amd._api import Sum, build_program
from tallymap_amd.backend import compile as Cm
from tallymap_amd.backend import kernel as K


def constants_item(n):
    """n adds of distinct constants, at bins past the value's."""
    def item(t, b):
        for j in range(n):
            t = t.add("h", b + j, np.float32(1.0 + j / 128.0))
        return t
    return item


def _src(item, S):
    return K.build(build_program(item, {"h": Sum((S,))}, (0,), [C.AVal((), C.I32)], [], None)[0])[0]


def _bare(S, n):
    """bytes with one float32 word per bin and one counter of one copy per constant."""
    return S * (4 + 8 * n)


@pytest.mark.parametrize("S", [1, 2, 16, 64])
@pytest.mark.parametrize("n", [1, 3, 40, 84, 90])
def test_copies_share_one_budget(S, n):
    """the copies' words, float64 bins, and the loop's staging of operands."""
    got = K.lds_bytes(_src(constants_item(n), S))
    stage = (K.BLOCK // 64) * K.CHUNK * 4
    assert got <= _bare(S, n) + 4 * S + K.LDS_F64 + stage
    if n == 1 and S <= 64:              # (one constant: as many copies of it as of the sums)
        assert got == 2 * 8 * S * min(16, K.LDS_COPIES // S) + stage


@pytest.mark.parametrize("S, n, copies", [(16, 84, True), (1024, 18, True), (1024, 19, False)])
def test_a_program_near_the_limit_compiles(S, n, copies):
    """(1,024 bins of 19 constants are 159,744 bytes bare: 4,096 more for float64 bins would not fit beside the
    staging)"""
    src = _src(constants_item(n), S)
    assert K.lds_bytes(src) <= K.LDS_MAX
    assert ("double tm_sh0" in src) == copies
    assert Cm.code_object(src, name="tm_lds_budget.hip")
