"""What backend/ahead.py takes out of a step: only values that depend on the step through its counters, and every value
the rest of the step reads is one it has."""
import numpy as np
import pytest

from tallymap_amd import _core as C
from tallymap_amd import configs, lax, problems, random
from tallymap_amd import numpy as jnp
from tallymap_amd._api import Sum, build_program
from tallymap_amd.backend import ahead as A
from tallymap_amd.backend import kernel as K


def _prog(item, outputs, axes, args, max_steps=None):
    pav = [C.AVal(np.shape(a)[1:], np.asarray(a).dtype) for a, x in zip(args, axes) if x == 0]
    bav = [C.AVal(np.shape(a), np.asarray(a).dtype) for a, x in zip(args, axes) if x is None]
    return build_program(item, outputs, axes, pav, bav, max_steps)[0]


def _plan(item, outputs, axes, args, max_steps=None):
    prog = _prog(item, outputs, axes, args, max_steps)
    we = prog.jaxpr.eqns[K._split(prog.jaxpr)]
    tallies = {v.id for v in prog.jaxpr.invars[:prog.nT]}
    for e in prog.jaxpr.eqns:           # (a tally stays one through emits)
        if e.prim == "tallymap_emit" and e.invars[0].id in tallies:
            tallies.add(e.outvars[0].id)
    return A.plan(we, lambda v: isinstance(v, C.Var) and v.id in tallies, K.cost), we


def _sound(pl, we):
    """the update side reads only loop operands, its own results and the cut; the ahead side only loop constants,
    counters, carries that never change and its own results; together they hold every equation."""
    bj, nb = we.params["body_jaxpr"], we.params["body_nconsts"]
    have = {v.id for v in bj.invars} | {v.id for v in pl.cut}
    for e in pl.update:
        assert all(v.id in have for v in e.invars if isinstance(v, C.Var)), e
        have |= {o.id for o in e.outvars}
    assert all(v.id in have for v in bj.outvars if isinstance(v, C.Var))
    same = {v.id for v, o in zip(bj.invars[nb:], bj.outvars) if isinstance(o, C.Var) and o.id == v.id}
    have = {v.id for v in bj.invars[:nb]} | same | {bj.invars[nb + j].id for j in pl.counters}
    for e in pl.ahead:
        assert A.pure(e) and A.bounded(e)
        assert all(v.id in have for v in e.invars if isinstance(v, C.Var)), e
        have |= {o.id for o in e.outvars}
    assert {id(e) for e in pl.ahead} | {id(e) for e in pl.update} == {id(e) for e in bj.eqns}


@pytest.mark.parametrize("name, words", [("c1", 1), ("c2", 1), ("c3", 9), ("c4", 2), ("random_walk", 2),
                                         ("transport", 4), ("walk_on_spheres", 6), ("barrier", 1), ("gillespie", 2)])
def test_programs_that_draw(name, words):
    cfg = getattr(configs, name.upper(), None) or problems.PROBLEMS[name]
    args = cfg["inputs"](8)[0] if "inputs" in cfg else getattr(configs, name + "_inputs")(8)
    pl, we = _plan(cfg["item"], cfg["outputs"], cfg["in_axes"], args, cfg.get("max_steps"))
    _sound(pl, we)
    assert sum(max(1, v.aval.size) for v in pl.cut) <= words


@pytest.mark.parametrize("name", ["c5", "ode_ensemble"])
def test_programs_without_draws_have_no_plan(name):
    cfg = getattr(configs, name.upper(), None) or problems.PROBLEMS[name]
    args = cfg["inputs"](8)[0] if "inputs" in cfg else getattr(configs, name + "_inputs")(8)
    assert _plan(cfg["item"], cfg["outputs"], cfg["in_axes"], args, cfg.get("max_steps"))[0] is None


def _walk(draw):
    """a walk whose draw is draw(key, k, x, m) -> (u, the next m)."""
    def item(t, x, key):
        def body(c):
            k, x, m, t = c
            u, m = draw(key, k, x, m)
            return k + 1, x * (0.5 + 0.5 * u), m, t.add("h", (x * 4).astype(jnp.int32), u)
        k, x, m, t = lax.while_loop(lambda c: c[1] > 0.05, body, (np.int32(0), x, np.int32(7), t))
        return t, k
    return _plan(item, {"h": Sum((4,))}, (0, 0), (np.ones(2, np.float32), np.zeros((2, 2), np.uint32)))


def test_what_counts_as_a_counter():
    u = random.uniform
    for gain in (1, -3, 5):             # any literal gain
        pl, we = _walk(lambda key, k, x, m: (u(random.fold_in(key, m)), m + gain))
        _sound(pl, we)
        assert gain in pl.counters.values()
    pl, we = _walk(lambda key, k, x, m: (u(random.fold_in(key, k)) + m.astype(jnp.float32), m))     # never changes
    _sound(pl, we)
    # a gain that is not a literal, or a draw keyed by the state: nothing to compute ahead
    assert _walk(lambda key, k, x, m: (u(random.fold_in(key, m)), m + k))[0] is None
    assert _walk(lambda key, k, x, m: (u(random.fold_in(key, m)), m * 2))[0] is None
    assert _walk(lambda key, k, x, m: (u(random.fold_in(key, (x * 100).astype(jnp.int32))), m + 1))[0] is None


def _walk_args(n):
    return np.linspace(0.2, 1.0, n).astype(np.float32), random.split(random.PRNGKey(3), n)


# Steps with a loop of their own.  Every loop ends for the counters 0 .. 19 that an item reaches; `up`, `shift` and
# `branch` never do (or after 2^32 trips) for 21 and on, `levels` doubles its trips with every step.
def _inner(name, k, u):
    if name == "up":
        return lax.while_loop(lambda c: c[0] != 20 - k, lambda c: (c[0] + 1, c[1] * 0.75 + u), (np.int32(0), u))[1]
    if name == "shift":
        return lax.while_loop(lambda c: c[0] != 0, lambda c: (c[0] >> 1, c[1] * 0.75 + u), (20 - k, u))[1]
    if name == "branch":
        return lax.cond(k % 2 == 0, lambda: _inner("up", k, u), lambda: u)
    if name == "levels":
        return lax.fori_loop(0, (0 * k + 1) << k, lambda i, s: s * 0.75 + u, u)
    assert name == "literal"
    return lax.fori_loop(0, 100, lambda i, s: s * 0.75 + u, u)


def loop_item(name, steps=20):
    """`steps` steps, each with the loop `name` on the counter and a draw."""
    def item(t, x, key):
        def body(c):
            k, x, t = c
            u = random.uniform(random.fold_in(key, k))
            v = _inner(name, k, u)
            return k + 1, x * (0.5 + 0.125 * u) + v, t.add("h", k % 4, np.int32(1))
        k, x, t = lax.while_loop(lambda c: c[0] < steps, body, (np.int32(0), x, t))
        return t, (k, x)
    return item


def condition_item(t, x, key):
    """a loop condition with a loop in it, which ends for the item's own x > 0 alone."""
    def cond(c):
        k, x, t = c
        n = lax.while_loop(lambda c: c[1] < 1.0, lambda c: (c[0] + 1, c[1] * 2.0), (np.int32(0), x))[0]
        return n < 12

    def body(c):
        k, x, t = c
        u = random.uniform(random.fold_in(key, k))
        return k + 1, x * (0.5 + 0.5 * u), t.add("h", k % 4, np.int32(1))
    k, x, t = lax.while_loop(cond, body, (np.int32(0), x, t))
    return t, (k, x)


LOOPS = {"up": 20, "shift": 20, "branch": 20, "levels": 12, "literal": 20}


def _ahead_sides(item):
    """(the plan, the emitted ahead side, the emitted condition) of an item of _walk_args."""
    spec = ({"h": Sum((4,), dtype=np.int32)}, (0, 0), _walk_args(2))
    pl, we = _plan(item, *spec)
    if pl is None:
        return None, None, None
    _sound(pl, we)
    src = K.build(_prog(item, *spec))[0]
    head = src[src.index("u32 tm_h0 = 0u;"):src.index("u32 tm_n0 = (u32)__builtin_amdgcn_ds_bpermute")]
    at = src.index("tm_n0 = (u32)__builtin_amdgcn_ds_bpermute(tm_ba + ")
    return pl, head, src[at:src.index("if (tm_ballot(tm_live && !tm_go_on)", at)]


@pytest.mark.parametrize("name", LOOPS)
def test_loops_without_a_literal_trip_count_stay_in_the_step(name):
    """the draw is computed ahead, a loop on its counter is not: steps past the item's last have no bound on it."""
    pl, head, _ = _ahead_sides(loop_item(name, LOOPS[name]))
    assert pl is not None and "tm_threefry" in head
    inner = [e for e in pl.ahead if e.prim in ("while", "cond")]
    if name == "literal":
        assert len(inner) == 1 and "while (true)" in head
    else:
        assert not inner and "while (true)" not in head and any(e.prim in ("while", "cond") for e in pl.update)


def test_a_condition_with_a_loop_runs_on_live_lanes_alone():
    _, _, cond = _ahead_sides(condition_item)
    assert cond.index("if (tm_live) {") < cond.index("while (true)")
    _, _, cond = _ahead_sides(loop_item("literal"))
    assert "if (tm_live)" not in cond


def test_a_program_that_spreads_has_nothing_sized_by_its_lanes():
    """Records' raw buffers have room for a batch per launched wave: no steps ahead there, and a size taken from a
    spreading program's lanes is refused."""
    import types

    from tallymap_amd import backend as B
    from tallymap_amd._api import Records

    def item(rec):
        def f(t, x, key):
            def body(c):
                k, x, t = c
                u = random.uniform(random.fold_in(key, k))
                t = t.append("r", {"u": u}) if rec else t.add("h", 0, u)
                return k + 1, x * u, t
            return lax.while_loop(lambda c: c[1] > 0.05, body, (np.int32(0), x, t))[2]
        return f
    for rec, out in ((False, {"h": Sum((1,))}), (True, {"r": Records({"u": np.float32}, 64)})):
        src, L = K.build(_prog(item(rec), out, (0, 0), _walk_args(2)))
        assert ("tm_spread" in src) == (L.spread > 0) == (not rec)
        c = types.SimpleNamespace(layout=L, block=256, id=-7 - rec)
        if L.spread:
            with pytest.raises(B.Cm.BackendError, match="spreads"):
                B._lanes(c, 100)
        else:
            B._LANES[c.id] = 1 << 20
            assert B._lanes(c, 257) == 512 and B._lanes(c, 1 << 24) == 1 << 20
