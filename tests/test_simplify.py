"""Common-subexpression elimination before emission (backend/simplify.py; CPU only)."""
import numpy as np

import tallymap_amd as tm
from tallymap_amd import _core as C
from tallymap_amd import configs, lax
from tallymap_amd import numpy as jnp
from tallymap_amd._api import build_program
from tallymap_amd.backend import kernel as K, reverse as R, simplify as S


def _prims(eqns):
    return [e.prim for e in eqns]


def test_fused_value_and_grad_post_evaluates_once():
    """value_and_grad's fused C4 program runs POST (atan2, sin, two emits) and then POST's VJP, which re-evaluates
    the same primal values on the same loop results: after CSE each is computed once and every emit stays."""
    n = 1024
    cfg = configs.c4_config(n)
    f = tm.vmap(cfg["item"], outputs=cfg["outputs"], in_axes=cfg["in_axes"], max_steps=cfg["max_steps"])
    prog = f._prepare(configs.c4_inputs(n))[0]
    adj = R.adjoint_program(prog, ((), (0,)))
    q = R.forward_only_program(adj, R.plan(adj), keep=True)
    w = K._split(q.jaxpr)
    before = _prims(q.jaxpr.eqns[w + 1:])
    jx = S.cse(q.jaxpr, w)
    after = _prims(jx.eqns[w + 1:])
    assert before.count("atan2") == 2 and after.count("atan2") == 1
    assert after.count("tallymap_emit") == before.count("tallymap_emit") >= 3
    assert len(after) < len(before)
    # every variable an equation reads is defined before it (or is an invar)
    defined = {v.id for v in jx.invars}
    for e in jx.eqns:
        for v in e.invars:
            assert not isinstance(v, C.Var) or v.id in defined
        defined |= {o.id for o in e.outvars}
    for v in jx.outvars:
        assert not isinstance(v, C.Var) or v.id in defined


def test_scopes_and_effects():
    """PRE and POST are separate scopes (a POST value is never renamed to a PRE one, which would keep it live
    through the loop); repeated emits are effects and all stay; duplicates inside the loop body are removed."""
    def item(t, x, key):
        a = jnp.sin(x * 2.0)
        t = t.add("h", 0, a)
        t = t.add("h", 0, a)

        def body(c):
            k, y = c
            return k + 1, y + jnp.cos(y) * jnp.cos(y)
        k, y = lax.while_loop(lambda c: c[0] < 3, body, (0, x))
        b = jnp.sin(x * 2.0)
        return t.add("h", 1, b + y), k
    p = build_program(item, {"h": tm.Sum((2,))}, (0, 0), [C.AVal((), np.float32), C.AVal((2,), np.uint32)], [],
                      None)[0]
    w = K._split(p.jaxpr)
    jx = S.cse(p.jaxpr, w)
    pre, post = _prims(jx.eqns[:w]), _prims(jx.eqns[w + 1:])
    assert pre.count("sin") == 1 and post.count("sin") == 1
    assert pre.count("tallymap_emit") == 2 and post.count("tallymap_emit") == 1
    body = jx.eqns[w].params["body_jaxpr"]
    assert _prims(body.eqns).count("cos") == 1
    assert _prims(p.jaxpr.eqns[w].params["body_jaxpr"].eqns).count("cos") == 2


def test_unchanged_program_is_returned_as_is():
    p = build_program(configs.c1_item, configs.C1["outputs"], (0, 0, None),
                      [C.AVal((), np.float32), C.AVal((2,), np.uint32)], [C.AVal((), np.float32)], 100)[0]
    jx = S.cse(p.jaxpr, K._split(p.jaxpr))
    assert len(jx.eqns) <= len(p.jaxpr.eqns)
    assert S.cse(jx, K._split(jx)) is jx


def _program(item, nb=0):
    return build_program(item, {"h": tm.Sum((4,))}, (0, 0) + (None,) * nb,
                         [C.AVal((), np.float32), C.AVal((2,), np.uint32)], [C.AVal((), np.float32)] * nb, None)[0].jaxpr


def test_sines_and_cosines_of_one_angle_are_paired():
    """one equation per angle and side of the step loop; a lone sine, float64 and other angles stay."""
    def item(t, x, key):
        t = t.add("h", 0, jnp.sin(x) + jnp.cos(x) + jnp.sin(x * 2.0))

        def body(c):
            k, y = c
            return k + 1, y + jnp.cos(y) * jnp.sin(y)
        k, y = lax.while_loop(lambda c: c[0] < 3, body, (0, x))
        return t.add("h", 1, jnp.cos(x * 2.0) + y), k
    jx = _program(item)
    w = K._split(jx)
    out = S.pair_sincos(jx, w)
    w2 = K._split(out)
    assert _prims(out.eqns[:w2]).count("tallymap_sincos") == 1
    assert _prims(out.eqns[:w2]).count("sin") == 1 and "cos" not in _prims(out.eqns[:w2])
    assert _prims(out.eqns[w2 + 1:]).count("cos") == 1 and "tallymap_sincos" not in _prims(out.eqns[w2 + 1:])
    b = _prims(out.eqns[w2].params["body_jaxpr"].eqns)
    assert b.count("tallymap_sincos") == 1 and "sin" not in b and "cos" not in b
    K.build(build_program(item, {"h": tm.Sum((4,))}, (0, 0), [C.AVal((), np.float32), C.AVal((2,), np.uint32)], [],
                          None)[0])
    assert S.pair_sincos(out, w2) is out


def test_draw_clamps_are_dropped_and_other_maxima_stay():
    from tallymap_amd import random
    for lo, hi in ((0.0, 1.0), (-1.0, 1.0), (0.25, 0.25), (-3.0, -2.5)):
        jx = _program(lambda t, x, key: (t.add("h", 0, random.uniform(key, (), np.float32, lo, hi)), x))
        assert "max" in _prims(jx.eqns) and "max" not in _prims(S.drop_draw_clamp(jx).eqns), (lo, hi)
        # the identity itself, in float32, at the ends of the draws and over a sample
        f = np.concatenate([[0.0, 1.0 - 2.0 ** -23], np.random.default_rng(1).integers(0, 2 ** 23, 100_000) * 2.0 ** -23])
        r = f.astype(np.float32) * np.float32(np.float32(hi) - np.float32(lo)) + np.float32(lo)
        assert np.array_equal(np.maximum(np.float32(lo), r).view(np.uint32), r.view(np.uint32))
    for fn in (lambda u, x: jnp.maximum(0.5, u), lambda u, x: jnp.maximum(0.0, x * 2.0 + 0.0),
               lambda u, x: jnp.maximum(-1.0, u * -2.0 - 1.0), lambda u, x: jnp.maximum(np.float32(-0.0), u * 2.0 + 0.0)):
        jx = _program(lambda t, x, key: (t.add("h", 0, fn(random.uniform(key), x)), x))
        assert _prims(S.drop_draw_clamp(jx).eqns).count("max") == 1
