"""Records outputs at the edges of their raw slots' segments and batches: every record arrives at its canonical slot
whatever the waves' share of them (segments of whole batches with a counter each, one segment for appends in a cond)."""
import numpy as np
import pytest

import tallymap_amd as tm
from tallymap_amd import lax

pytestmark = pytest.mark.gpu


def _item(in_cond):
    def item(t, i, n):
        """n records (item, ordinal)."""
        def append(t, k):
            return t.append("r", dict(i=i, k=k))

        def body(c):
            k, t = c
            t = lax.cond(i % 2 == 0, lambda t: append(t, k), lambda t: append(t, k), t) if in_cond else append(t, k)
            return k + 1, t
        k, t = lax.while_loop(lambda c: c[0] < n, body, (np.int32(0), t))
        return t
    return item


def _check(n_of, N, capacity, in_cond=False, **opts):
    import torch
    i = torch.arange(N, dtype=torch.int32, device="cuda")
    n = torch.as_tensor(n_of(np.arange(N)).astype(np.int32), device="cuda")
    f = tm.vmap(_item(in_cond), outputs={"r": tm.Records({"i": np.int32, "k": np.int32}, capacity=capacity)},
                in_axes=(0, 0), **opts)
    r = f(i, n)
    total = int(n.long().sum())
    assert int(r.stats["appended"]["r"].item()) == total
    assert int(r.stats["records_dropped"]["r"].item()) == max(0, total - capacity)
    gi, gk = r.outputs["r"]["i"], r.outputs["r"]["k"]
    if total > capacity:
        assert bool((gi == -1).all()) and bool((gk == -1).all())
        return
    wi = torch.repeat_interleave(i, n.long())
    off = torch.cumsum(n.long(), 0) - n.long()
    wk = torch.arange(total, device="cuda") - torch.repeat_interleave(off, n.long())
    assert torch.equal(gi[:total], wi) and torch.equal(gk[:total].long(), wk)
    assert not bool(gi[total:].any()) and not bool(gk[total:].any())


@pytest.mark.parametrize("N, per", [(1, 1), (1, 5000), (64, 3), (300, 257), (5000, 20), (70_001, 3)])
def test_capacity_equal_to_the_records(N, per):
    """a capacity of exactly the records, one more, and one fewer (dropped, poisoned)."""
    for d in (0, 1, -1):
        if N * per + d > 0:
            print("case:", N, per, d, flush=True)
            _check(lambda a: np.full(a.shape, per), N, N * per + d)


def test_a_few_waves_hold_all_records():
    """the first items append thousands each, the others nothing: their waves' segments fill up and they go on in the
    others'."""
    for N, heavy, per in ((200_000, 64, 3000), (200_000, 1, 100_000), (3000, 7, 1)):
        print("case:", N, heavy, per, flush=True)
        _check(lambda a: np.where(a < heavy, per, 0), N, heavy * per)
        _check(lambda a: np.where(a < heavy, per, 0), N, heavy * per - 1)


@pytest.mark.parametrize("opts", [dict(), dict(block=64), dict(schedule="item"), dict(post_batch=64)], ids=str)
def test_appends_in_a_cond_and_options(opts):
    for in_cond in (False, True):
        print("case:", opts, in_cond, flush=True)
        _check(lambda a: a % 37, 10_007, int((np.arange(10_007) % 37).sum()), in_cond, **opts)
