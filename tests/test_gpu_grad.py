"""Reverse mode on the GPU: the replay adjoint kernel against the oracle's forward-mode (dual number) gradients.
Gradients within 1e-4 relative; the per-item cotangents bitwise independent of the replay's
schedule, tape size and checkpoint count (reference tests/reverse.py:216); truncation makes every cotangent NaN (reference _primitive.py:586-594)."""
import numpy as np
import pytest

import tallymap_amd as tm
from tallymap_amd import configs

pytestmark = pytest.mark.gpu
GTOL = 1e-4


def _sync():
    import torch
    torch.cuda.synchronize()


def _np(x):
    return x.cpu().numpy()


def _mapped(cfg, **opts):
    return tm.vmap(cfg["item"], outputs=cfg["outputs"], in_axes=cfg["in_axes"], max_steps=cfg["max_steps"], **opts)


def test_c1_grad_theta(oracle):
    """d(hist.sum())/d theta: one adjoint launch (tm.grad) against the oracle and the closed form hist.sum()/theta."""
    print("case: C1 grad theta N=10000", flush=True)
    xs, keys, theta = configs.c1_inputs()
    g = tm.grad(_mapped(configs.C1), argnums=2)(xs, keys, theta)
    _sync()
    got = float(_np(g))
    want, ntr = oracle.c1_grad(xs, keys, theta, np.ones(16, np.float32))
    assert ntr == 0
    assert abs(got - float(want)) <= GTOL * abs(float(want))
    ref = oracle.c1_fwd(xs, keys, theta)
    closed = ref.tallies64["hist"].sum() / float(theta)
    assert abs(got - closed) <= GTOL * abs(closed)


VARIANTS = [dict(), dict(rev_tape=4), dict(rev_tape=2), dict(rev_tape=1), dict(schedule="item"),
            dict(rev_residual=True), dict(rev_residual=True, rev_tape=4), dict(rev_residual=True, rev_tape=1),
            dict(rev_schedule="step"), dict(rev_schedule="step", rev_tape=4), dict(rev_schedule="step", rev_tape=2),
            dict(rev_schedule="step", rev_refill=1), dict(rev_schedule="step", rev_refill=64),
            dict(rev_schedule="item"), dict(rev_schedule="item", rev_checkpoints=4),
            dict(rev_schedule="item", rev_checkpoints=1), dict(post_batch=64), dict(post_batch=64, rev_residual=True),
            dict(rev_record=False)]


@pytest.mark.parametrize("opts", VARIANTS, ids=["tape", "tape4", "tape2", "tape1", "tape-itemsched", "resid",
                                                "resid-tape4", "resid-tape1", "step", "step-tape4", "step-tape2",
                                                "step-refill1", "step-refill64", "item16", "item4", "item1",
                                                "tape-postbatch", "resid-postbatch", "tape-replayed"])
def test_c1_grad_xs_and_replay_variants(oracle, opts):
    """cotangents of xs (per item, through the loop state: the replay) and of theta with weights ct, against the
    oracle; the replay variants give bitwise the same per-item cotangents and broadcast cotangent (reference
    tests/reverse.py:216): the two-launch tape adjoint (the default; a 4-, 2- or 1-slot tape makes the ~8-step
    items recompute the states past the tape inside the reverse step; the item schedule of the forward template;
    the residual tape forced, alone and with 4- and 1-slot tapes whose later steps replay from the checkpoint),
    the single-kernel step-scheduled replay (an item overflowing a 4- or 2-slot tape takes the checkpointed sweep;
    waves refilled by 1 or 64 free lanes), the one-item-per-lane schedule with C checkpoints (C = 4, 1 force its
    segment re-runs), the tape adjoint with every finished item's POST deferred to a shared pass (post_batch=64;
    state and residual tapes), and the tape adjoint whose count launch runs at pullback time (rev_record=False)
    instead of as vjp's forward."""
    print(f"case: C1 vjp (xs, theta) {opts}", flush=True)
    xs, keys, theta = configs.c1_inputs()
    ct = np.linspace(0.5, 2.0, 16).astype(np.float32)
    res, pull = tm.vjp(_mapped(configs.C1, **opts), xs, keys, theta, argnums=(0, 2))
    gx, gth = pull({"hist": ct})
    _sync()
    want_th, want_x, ntr = oracle.c1_grad(xs, keys, theta, ct, per_item=True)
    gx = _np(gx)
    assert abs(float(_np(gth)) - float(want_th)) <= GTOL * abs(float(want_th))
    err = np.abs(gx - want_x) / np.maximum(np.abs(want_x), 1.0)
    assert err.max() <= GTOL, err.max()
    if opts:
        _, pull0 = tm.vjp(_mapped(configs.C1), xs, keys, theta, argnums=(0, 2))
        gx0, gth0 = pull0({"hist": ct})
        _sync()
        assert np.array_equal(gx.view(np.uint32), _np(gx0).view(np.uint32))
        assert np.float32(_np(gth)).view(np.uint32) == np.float32(_np(gth0)).view(np.uint32)


def test_c1_grad_truncation_is_nan(oracle):
    print("case: C1 grad max_steps=3", flush=True)
    xs, keys, theta = configs.c1_inputs()
    g = tm.grad(_mapped(dict(configs.C1, max_steps=3)), argnums=2)(xs, keys, theta)
    _sync()
    assert np.isnan(float(_np(g)))


def test_c2_grad_drift_is_exactly_zero(oracle):
    """the emitted values are constants: the pathwise gradient w.r.t. drift (and x0) is exactly 0."""
    print("case: C2 grad drift N=65536", flush=True)
    x0, keys, drift = configs.c2_inputs(65_536)
    f = _mapped(configs.C2)
    g = tm.grad(f, argnums=2)(x0, keys, drift)
    _sync()
    want, ntr = oracle.c2_grad(x0, keys, drift, np.ones(128, np.float32), np.ones(2, np.float32))
    assert float(_np(g)) == float(want) == 0.0
    res, pull = tm.vjp(f, x0, keys, drift, argnums=(0, 2))
    gx, gd = pull({"occ": 1.0, "wall": 1.0})
    _sync()
    assert float(_np(gd)) == 0.0 and not np.any(_np(gx))


def test_c2_grad_full_size():
    print("case: C2 grad drift N=4194304", flush=True)
    x0, keys, drift = configs.c2_inputs()
    g = tm.grad(_mapped(configs.C2), argnums=2)(x0, keys, drift)
    _sync()
    assert float(_np(g)) == 0.0


def test_no_stale_runtime_error_after_launches():
    """a forward launch and both adjoint kinds leave no pending runtime error for the framework's next call (the
    launch library clears the errors of its optional symbol lookups)."""
    import torch
    xs, keys, theta = configs.c1_inputs(512)
    f = _mapped(configs.C1)
    f(xs, keys, theta)
    tm.grad(f, argnums=2)(xs, keys, theta)                         # forward-only adjoint
    tm.vjp(f, xs, keys, theta, argnums=(0, 2))[1]({"hist": 1.0})   # checkpointed adjoint
    x = torch.full((8,), 2.0, device="cuda") * 3.0
    torch.cuda.synchronize()
    assert float(x.sum().item()) == 48.0


ROWS = 1024


def _rows(i, k):
    return (i * 7919 + k * 104729) % ROWS


def _table_items():
    from tallymap_amd import lax

    def walk(t, i, x, tab):            # an active carry: the tape adjoint
        def body(c):
            k, s, t_ = c
            s = s * 0.5 + tab[_rows(i, k)] * x
            return k + 1, s, t_.add("h", 0, s)
        return lax.while_loop(lambda c: c[0] < 20, body, (0, np.float32(0.0), t))[2]

    def reads(t, i, x, tab):           # no active carry: the forward-only adjoint
        def body(c):
            k, t_ = c
            return k + 1, t_.add("h", 0, tab[_rows(i, k)] * x)
        return lax.while_loop(lambda c: c[0] < 20, body, (0, t))[1]
    return walk, reads


def _table_grad_want(i, x, geometric):
    """d(sum h)/d tab in float64: each read at step k adds x times its weight, sum_{m >= k} 0.5^(m - k) over the
    20 steps for the walk (the read reaches s_k .. s_19), 1 for the plain reads.  Every term is a dyadic rational
    of at most 21 significant bits, so the float32 gradient (an exact sum rounded once) is this value rounded."""
    w = np.array([sum(0.5 ** (m - k) for m in range(k, 20)) if geometric else 1.0 for k in range(20)])
    g = np.zeros(ROWS)
    for k in range(20):
        np.add.at(g, _rows(i.astype(np.int64), k), x.astype(np.float64) * w[k])
    return g.astype(np.float32)


@pytest.mark.parametrize("kind", ["walk", "reads"])
def test_grad_wrt_a_1024_row_table(kind):
    """the cotangent of a broadcast table read at traced indices is emitted at the row read (one emit per read,
    not a select and an emit per table row): d(sum h)/d tab for a 1024-row table equals the closed form bitwise,
    through the tape adjoint (an active carry) and the forward-only adjoint; n_active=n equals the call over the
    first n items."""
    print(f"case: grad wrt a {ROWS}-row table ({kind}), N=8192", flush=True)
    walk, reads = _table_items()
    item = walk if kind == "walk" else reads
    rng = np.random.default_rng(11)
    n = 8192
    i = rng.integers(0, 1 << 17, n).astype(np.int32)        # (i * 7919 + 19 * 104729 < 2^31: no wrap)
    x = rng.choice(np.array([0.5, 1.0, 2.0, -1.0], np.float32), n)
    tab = rng.standard_normal(ROWS).astype(np.float32)
    f = tm.vmap(item, outputs={"h": tm.Sum((1,))}, in_axes=(0, 0, None))
    g = tm.grad(f, argnums=2)(i, x, tab)
    _sync()
    want = _table_grad_want(i, x, kind == "walk")
    assert np.array_equal(_np(g).view(np.uint32), want.view(np.uint32))
    m = 3000
    ga = tm.grad(f, argnums=2)(i, x, tab, n_active=m)
    gm = tm.grad(f, argnums=2)(i[:m], x[:m], tab)
    _sync()
    assert np.array_equal(_np(ga).view(np.uint32), _np(gm).view(np.uint32))
    assert np.array_equal(_np(ga).view(np.uint32), _table_grad_want(i[:m], x[:m], kind == "walk").view(np.uint32))


def _vg_cases():
    """(config name, inputs, argnums, weights) of the value_and_grad checks: C1 (forward-only adjoint), C3 and C5 (the
    tape adjoint's count launch returns the forward)."""
    n3, n5 = 65_536, 4096
    return [("c1", lambda: configs.c1_inputs(20_000), 2, None),
            ("c3", lambda: configs.c3_inputs(n3), 1, None),
            ("c5", lambda: configs.c5_inputs(n5), 3, {"state": 1.0})]


@pytest.mark.parametrize("mode", ["auto", "reverse"])
@pytest.mark.parametrize("name,inputs,argnums,weights", _vg_cases(), ids=["c1", "c3", "c5"])
def test_value_and_grad_in_fewer_launches(name, inputs, argnums, weights, mode):
    """value_and_grad: the forward's outputs (tallies bitwise where exact, else within the float32 atomic-order
    tolerance; per-item results and truncation flags bitwise) and the gradient equal the separate forward call and
    grad.  By the replay adjoint the gradient is bitwise the same (its broadcast cotangents are exact sums); where
    grad_mode='auto' takes tangent lanes (a few broadcast elements through a swept carry: C3's mu_a, C5's A) the
    gradient contracts tangent tallies that are plain float32 atomic sums, whose last bits change from run to run
    like the forward's tallies, so it agrees within a few ulps."""
    import torch
    print(f"case: value_and_grad {name} grad_mode={mode}", flush=True)
    cfg = configs.SIZED[name](len(inputs()[0])) if name in configs.SIZED else configs.CONFIGS[name]
    f = _mapped(cfg, grad_mode=mode)
    args = inputs()
    res, g = tm.value_and_grad(f, weights=weights, argnums=argnums)(*args)
    ref = f(*args)
    g_ref = tm.grad(f, weights=weights, argnums=argnums)(*args)
    torch.cuda.synchronize()
    if mode == "reverse":
        assert np.array_equal(np.atleast_1d(_np(g)).view(np.uint32), np.atleast_1d(_np(g_ref)).view(np.uint32))
    else:
        assert np.allclose(_np(g), _np(g_ref), rtol=1e-6, atol=0.0), (_np(g), _np(g_ref))
    for k in ref.outputs:
        a, b = _np(res.outputs[k]), _np(ref.outputs[k])
        assert a.shape == b.shape and np.allclose(a, b, rtol=1e-5, atol=1e-6 * float(np.abs(b).max())), k
    ya = [_np(y) for y in (res.per_item if isinstance(res.per_item, (tuple, list)) else [res.per_item])] \
        if res.per_item is not None else []
    yb = [_np(y) for y in (ref.per_item if isinstance(ref.per_item, (tuple, list)) else [ref.per_item])] \
        if ref.per_item is not None else []
    assert len(ya) == len(yb) and all(np.array_equal(x.view(np.uint8), y.view(np.uint8)) for x, y in zip(ya, yb))
    assert np.array_equal(_np(res.truncated), _np(ref.truncated))
    assert int(_np(res.stats["n_truncated"])) == int(_np(ref.stats["n_truncated"]))


def test_accumulator_carry_forward_only_adjoint():
    """an accumulator carry (acc' = acc + theta y_k, started at 2 theta, read by the loop condition, its square
    emitted after the loop) is differentiated by the forward-only adjoint (no tape): d sum acc^2 / d theta =
    sum 2 acc (2 + sum_k y_k), from a float32 emulation of y; and equal to forward mode."""
    from tallymap_amd import lax

    def item(t, x, th):
        def body(c):
            k, y, acc = c
            y = y * 0.5 + x
            return k + 1, y, acc + th * y
        k, y, acc = lax.while_loop(lambda c: (c[0] < 8) & (c[2] < 100.0), body, (0, x, th * 2.0))
        return t.add("h", 0, acc * acc), k
    n = 50_000
    print(f"case: accumulator carry N={n}", flush=True)
    x = np.linspace(0.0, 1.0, n).astype(np.float32)
    th = np.float32(0.5)
    f = tm.vmap(item, outputs={"h": tm.Sum((1,))}, in_axes=(0, None))
    g = float(_np(tm.grad(f, argnums=1)(x, th)))
    y = x.copy()
    S = np.zeros(n, np.float64)
    acc = np.full(n, np.float32(th * np.float32(2.0)))
    for _ in range(8):
        y = (y * np.float32(0.5) + x).astype(np.float32)
        S += y
        acc = (acc + th * y).astype(np.float32)
    want = float(np.sum(2.0 * acc.astype(np.float64) * (2.0 + S)))
    assert abs(g - want) <= 1e-5 * abs(want), (g, want)
    jf = float(_np(tm.jacfwd(f, argnums=1)(x, th)["h"][1]).reshape(-1)[0])
    assert abs(g - jf) <= 1e-5 * abs(want), (g, jf)


@pytest.mark.parametrize("name", ["c3", "c5"])
def test_vjp_forward_records_the_tape(name):
    """vjp's forward call is the tape adjoint's count launch (the pullback is the reverse launch alone): its outputs
    equal the plain forward call's (float32 atomic-order tolerance; per-item results and truncation bitwise), and
    its cotangents are bitwise those of the replayed adjoint (rev_record=False: the plain forward, then the count
    and reverse launches at pullback time) -- for two pullbacks of one vjp with different cotangents (the tape is
    read, not consumed), and with n_active."""
    import torch
    n = 65_536 if name == "c3" else 4096
    print(f"case: vjp records the tape {name} N={n}", flush=True)
    cfg = configs.SIZED[name](n) if name in configs.SIZED else configs.CONFIGS[name]
    args = configs.c3_inputs(n) if name == "c3" else configs.c5_inputs(n)
    argnums = 1 if name == "c3" else (0, 3)
    f, f0 = _mapped(cfg, grad_mode="reverse"), _mapped(cfg, grad_mode="reverse", rev_record=False)
    for n_active in (None, n // 3):
        res, pull = tm.vjp(f, *args, argnums=argnums, n_active=n_active)
        ref = f(*args, n_active=n_active)
        _, pull0 = tm.vjp(f0, *args, argnums=argnums, n_active=n_active)
        torch.cuda.synchronize()
        for k in ref.outputs:
            a, b = _np(res.outputs[k]), _np(ref.outputs[k])
            assert a.shape == b.shape and np.allclose(a, b, rtol=1e-5, atol=1e-6 * float(np.abs(b).max())), k
        assert np.array_equal(_np(res.truncated), _np(ref.truncated))
        if ref.per_item is not None:
            assert np.array_equal(_np(res.per_item).view(np.uint8), _np(ref.per_item).view(np.uint8))
        for scale in (1.0, -0.5):
            ct = {k: (scale * np.linspace(0.5, 2.0, v.numel())).astype(np.float32).reshape(tuple(v.shape))
                  for k, v in ref.outputs.items()}
            got = pull(ct)
            want = pull0(ct)
            torch.cuda.synchronize()
            got, want = (got, want) if isinstance(got, tuple) else ((got,), (want,))
            for x, y in zip(got, want):
                assert np.array_equal(np.atleast_1d(_np(x)).view(np.uint32), np.atleast_1d(_np(y)).view(np.uint32))
            assert any(np.any(_np(x) != 0) for x in got)


def test_grad_through_a_static_loop_before_the_step_loop():
    """y = fori_loop(0, 3, a -> a theta + 0.25, x) in PRE (a static loop: unrolled for reverse mode), then a walk
    whose emits and carry scale with theta: the replay gradient w.r.t. theta, and the xs cotangent dotted with a
    direction, equal forward mode's tangents (the sum of the tangent tally) within 1e-5 -- two independent
    derivations of the same derivative."""
    import torch
    from test_frontend import _static_item

    import tallymap_amd as tm
    from tallymap_amd import random as R
    n = 65_536
    print(f"case: grad through a static loop, N={n}", flush=True)
    xs = np.linspace(0.2, 0.9, n).astype(np.float32)
    keys = R.split(R.PRNGKey(3), n)
    th = np.float32(0.9)
    f = tm.vmap(_static_item(3), outputs={"h": tm.Sum((8,))}, in_axes=(0, 0, None))
    g_th = float(np.asarray(tm.grad(f, argnums=2)(xs, keys, th).cpu()))
    _, tan = tm.jvp(f, (xs, keys, th), (None, None, np.float32(1.0)))
    torch.cuda.synchronize()
    want = float(tan.outputs["h"].cpu().numpy().astype(np.float64).sum())
    assert abs(g_th - want) <= 1e-5 * abs(want), (g_th, want)
    v = np.random.default_rng(1).standard_normal(n).astype(np.float32)
    g_x = tm.grad(f, argnums=0)(xs, keys, th).cpu().numpy().astype(np.float64)
    _, tan_x = tm.jvp(f, (xs, keys, th), (v, None, None))
    torch.cuda.synchronize()
    got, want_x = float(g_x @ v), float(tan_x.outputs["h"].cpu().numpy().astype(np.float64).sum())
    assert abs(got - want_x) <= 1e-5 * abs(want_x) + 1e-6 * float(np.abs(g_x).sum()), (got, want_x)
