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


def _doubling(t, x, i):
    """x doubled i % 5 times, then added: the adjoint sweeps back over the steps, from a tape."""
    x = lax.while_loop(lambda c: c[0] < i % 5, lambda c: (c[0] + 1, c[1] * 2.0), (np.int32(0), x))[1]
    return t.add("h", i % 4, x)


@pytest.mark.parametrize("opts", [dict(block=64, blocks_per_cu=1), dict(), dict(refill=8)], ids=str)
def test_a_taped_gradient_runs_every_item_once(opts):
    """the tape programs' ranges deal the chunks out in turn: one chunk per wave, the ranges' first and last ones, and
    the last chunk of the call whole and short."""
    import torch
    f = tm.vmap(_doubling, outputs={"h": tm.Sum((4,))}, in_axes=(0, 0), **opts)
    R = _resident(**opts)
    for n in (1, 65, R, R + 1, R + 64, 2 * R + 4095, 2 * R + 4096, 2 * R + 4097, 3 * R - 63, 5 * R):
        print("case:", opts, n, flush=True)
        i = torch.arange(n, dtype=torch.int32, device="cuda")
        x = 1.0 + (i % 7).float()
        res, g = tm.value_and_grad(f, argnums=0)(x, i)
        want = torch.pow(2.0, (i % 5).float())
        assert torch.equal(g, want), n
        h = torch.zeros(4, dtype=torch.float64, device="cuda").index_add_(0, i.long() % 4, (x * want).double())
        assert torch.allclose(res.outputs["h"].double(), h, rtol=1e-5, atol=0.0), n
