"""Every item runs exactly once, whatever the number of items: the claim counters of the item ranges (one chunk per
wave below the resident lanes, ranges of whole chunks above, the last ones short or empty), under both schedules."""
import numpy as np
import pytest

import tallymap_amd as tm
from tallymap_amd import backend as B
from tallymap_amd import lax
from tallymap_amd import numpy as jnp

pytestmark = pytest.mark.gpu


def _item(t, i):
    """i % 5 steps, then one count and the item's number."""
    def body(c):
        return c[0] + 1, c[1] + 3
    k, y = lax.while_loop(lambda c: c[0] < i % 5, body, (np.int32(0), i))
    return t.add("n", i % 8, np.int32(1)), (k, y)


def _check(n, n_active=None, **opts):
    import torch
    f = tm.vmap(_item, outputs={"n": tm.Sum((8,), dtype=np.int32)}, in_axes=0, **opts)
    i = torch.arange(n, dtype=torch.int32, device="cuda")
    r = f(i) if n_active is None else f(i, n_active=n_active)
    k, y = r.per_item
    m = n if n_active is None else n_active
    assert torch.equal(r.outputs["n"].cpu().long(), torch.bincount(i[:m].long() % 8, minlength=8).cpu()), n
    assert torch.equal(k[:m], i[:m] % 5) and torch.equal(y[:m], i[:m] + 3 * (i[:m] % 5)), n
    assert not bool(k[m:].any()) and not bool(y[m:].any())


def _resident(**opts):
    f = tm.vmap(_item, outputs={"n": tm.Sum((8,), dtype=np.int32)}, in_axes=0, **opts)
    prog = f._prepare((np.zeros(4, np.int32),))[0]
    return B.kernel_info(B.compiled(prog, opts))["resident_threads"]


@pytest.mark.parametrize("opts", [dict(), dict(schedule="item"), dict(block=64, blocks_per_cu=1), dict(refill=8),
                                  dict(compact=0)], ids=str)
def test_every_item_runs_once(opts):
    R = _resident(**opts)
    for n in (1, 63, 64, 65, 255, 257, 4095, 4097, R - 1, R, R + 1, R + 64, 2 * R + 4096, 3 * R - 63):
        print("case:", opts, n, flush=True)
        _check(n, **opts)


def test_active_items_only():
    R = _resident()
    for n, m in ((1000, 0), (1000, 1), (R + 5000, R), (R + 5000, R + 1), (2 * R, 7)):
        print("case: n", n, "active", m, flush=True)
        _check(n, n_active=m)
