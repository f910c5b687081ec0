"""How vjp / grad / value_and_grad differentiate (option grad_mode), decided on the host: by tangent lanes (one jvp
launch with a lane per differentiated broadcast element) or by the replay adjoint.  No GPU: the decision reads the
traced program and its adjoint plan only."""
import numpy as np
import pytest

import tallymap_amd as tm
from tallymap_amd import _api, configs, lax


def _plan(cfg, args, argnums, **opts):
    f = tm.vmap(cfg["item"], outputs=cfg["outputs"], in_axes=cfg["in_axes"], max_steps=cfg["max_steps"],
                **dict(cfg.get("opts", {}), **opts))
    m = f._sized(args, None)
    prog, meta, pi, bc, N, axes = m._prepare(args)
    return _api._tangent_plan(m, prog, args, axes, argnums)


def test_auto_takes_lanes_for_a_swept_carry_and_few_broadcast_elements():
    # C3: mu_a (a scalar) scales the photon weight, a loop carry: one lane
    p = _plan(configs.C3, configs.c3_inputs(64), 1)
    assert p is not None and p[2] == [(0, 0)]
    # C5: A (a scalar) drives the pendulum state: one lane
    p = _plan(configs.c5_config(64), configs.c5_inputs(64), 3)
    assert p is not None and p[2] == [(0, 0)]


def test_auto_keeps_the_replay_adjoint_otherwise():
    # C2: no carry depends on drift -- the forward-only adjoint is one launch already
    assert _plan(configs.C2, configs.c2_inputs(64), 2) is None
    # a per-item argument, alone or beside a broadcast one
    assert _plan(configs.C1, configs.c1_inputs(64), 0) is None
    assert _plan(configs.C1, configs.c1_inputs(64), (0, 2)) is None
    # grad_mode='reverse'
    assert _plan(configs.C3, configs.c3_inputs(64), 1, grad_mode="reverse") is None


def test_auto_lane_budget_and_forced_tangent_mode():
    def item(t, x, th):
        def body(c):
            k, s = c
            return k + 1, s * th[k % th.shape[0]] + x
        k, s = lax.while_loop(lambda c: c[0] < 5, body, (0, x))
        return t.add("h", 0, s)
    x = np.linspace(0, 1, 64).astype(np.float32)
    for P in (8, 9, 20):
        cfg = dict(item=item, outputs={"h": tm.Sum((1,))}, in_axes=(0, None), max_steps=None)
        th = np.full(P, 0.5, np.float32)
        p = _plan(cfg, (x, th), 1)
        assert (p is not None) == (P <= _api.TANGENT_MAX)
        q = _plan(cfg, (x, th), 1, grad_mode="tangent")
        assert q is not None and q[2] == [(0, e) for e in range(P)]
    with pytest.raises(tm.UnsupportedError):
        _plan(cfg, (x, th), (0, 1), grad_mode="tangent")
    with pytest.raises(ValueError):
        _plan(cfg, (x, th), 1, grad_mode="backward")


def test_pytree_broadcast_argument_lanes():
    """a dict argument with two float32 leaves and an int32 one: a lane per float32 element, in leaf order."""
    def item(t, x, p):
        def body(c):
            k, s = c
            return k + 1, s * p["a"] + p["b"][k % 2] * x
        k, s = lax.while_loop(lambda c: c[0] < p["n"], body, (0, x))
        return t.add("h", 0, s)
    x = np.linspace(0, 1, 64).astype(np.float32)
    prm = {"a": np.float32(0.5), "b": np.array([1.0, 2.0], np.float32), "n": np.int32(4)}
    cfg = dict(item=item, outputs={"h": tm.Sum((1,))}, in_axes=(0, None), max_steps=None)
    p = _plan(cfg, (x, prm), 1)
    assert p is not None and len(p[2]) == 3


def test_auto_takes_lanes_for_a_spawning_call():
    """a spawning call w.r.t. a few broadcast elements: lanes (one forward through the generations, children carrying
    their parents' tangents) in place of the tree adjoint; w.r.t. a per-item argument (the roots): the tree adjoint.
    Records outputs always replay, and grad_mode='tangent' refuses them."""
    def particle(t, p, th):
        t = t.add("dep", 0, p["E"] * th[0])
        return t.spawn(dict(E=p["E"] * th[1], g=p["g"] + 1), when=p["g"] < 2)
    roots = dict(E=np.linspace(1.0, 2.0, 64).astype(np.float32), g=np.zeros(64, np.int32))
    th = np.array([0.2, 0.6], np.float32)
    cfg = dict(item=particle, outputs={"dep": tm.Sum((1,))}, in_axes=(0, None), max_steps=None,
               opts=dict(spawn=tm.Queue(1 << 10)))
    p = _plan(cfg, (roots, th), 1)
    assert p is not None and p[2] == [(0, 0), (0, 1)]
    assert _plan(cfg, (roots, th), 0) is None
    assert _plan(cfg, (roots, th), 1, grad_mode="reverse") is None

    def rec(t, x, th):
        return t.append("r", {"v": x * th[0]})
    rcfg = dict(item=rec, outputs={"r": tm.Records({"v": np.float32}, 64)}, in_axes=(0, None), max_steps=None)
    x = np.linspace(0, 1, 64).astype(np.float32)
    assert _plan(rcfg, (x, th), 1) is None
    with pytest.raises(tm.UnsupportedError):
        _plan(rcfg, (x, th), 1, grad_mode="tangent")


def test_vjp_takes_lanes_where_they_cost_less_than_two_launches():
    """vjp needs the outputs before the cotangent: forward and forward-only adjoint are two launches, the lanes one.
    Taken for small float32 sums and few elements, with exact sums as the adjoint's; not where a tangent would leave LDS
    (the disk's maps), goes to a few bins that a wave's lanes would wait for (up-and-out calls) or is a per-item
    result's, not with 'reverse', and grad / value_and_grad (one launch by the adjoint) stay."""
    from tallymap_amd import problems

    def plan(f, args, argnum, pair):
        m = f._sized(args, None)
        prog, _, _, _, _, axes = m._prepare(args)
        return _api._tangent_plan(m, prog, args, axes, argnum, pair=pair)
    rw = problems.PROBLEMS["random_walk"]
    args = rw["inputs"](64)[0]
    p = plan(problems.mapped("random_walk"), args, 2, True)
    assert p is not None and p[2] == [(0, 0), (0, 1), (0, 2)] and p[4] == "exact"
    assert plan(problems.mapped("random_walk"), args, 2, False) is None
    assert plan(problems.mapped("barrier"), problems.PROBLEMS["barrier"]["inputs"](64)[0], 2, True) is None

    # (a fixed-point float32 sum's tangents too are exact to float64; a scaled sum's would be rounded to its scale)
    for dt in (np.float32, np.float64):
        f = tm.vmap(rw["item"], outputs={"hist": tm.Sum((64,), dtype=dt, fixed_point=True)}, in_axes=rw["in_axes"])
        assert (plan(f, args, 2, True) is not None) == (dt == np.float32)
        if dt == np.float32:
            q = _api._jvp_prog(f._prepare(args)[0], (False,), (False, True), 3, "exact")
            assert [(t.dtype, t.exact) for t in q.tallies] == [(dt, True)] + [(np.float64, True)] * 3

    def with_result(t, *a):
        t, k = rw["item"](t, *a)
        return t, (k, a[2][0] * 2.0)
    f = tm.vmap(with_result, outputs=rw["outputs"], in_axes=rw["in_axes"])
    assert plan(f, args, 2, True) is None
    assert plan(problems.mapped("random_walk", grad_mode="reverse"), args, 2, True) is None
    for cfg, inputs, pos in ((configs.c4_config(64), configs.c4_inputs(64), 3), (configs.C1, configs.c1_inputs(64), 0)):
        f = tm.vmap(cfg["item"], outputs=cfg["outputs"], in_axes=cfg["in_axes"], max_steps=cfg["max_steps"])
        assert plan(f, inputs, pos, True) is None
