"""The tracer, the tally rules and the cap (CPU only)."""
import numpy as np
import pytest

import tallymap_amd as tm
from tallymap_amd import _core as C
from tallymap_amd import configs, lax, random
from tallymap_amd import numpy as jnp
from tallymap_amd._api import build_program


def _prog(item, outputs, pav, bav, axes, max_steps=None):
    return build_program(item, outputs, axes, [C.AVal(*a) for a in pav], [C.AVal(*a) for a in bav], max_steps)[0]


def test_quickstart_traces_to_one_capped_loop():
    p = _prog(configs.c1_item, configs.C1["outputs"], [((), np.float32), ((2,), np.uint32)], [((), np.float32)],
              (0, 0, None), 100)
    prims = [e.prim for e in p.jaxpr.eqns]
    assert prims.count("while") == 1
    w = p.jaxpr.eqns[prims.index("while")]
    body = [e.prim for e in w.params["body_jaxpr"].eqns]
    assert body.count("threefry2x32") == 2 and "tallymap_emit" in body
    assert p.trunc == 1                                # per-item results: [k, truncated]
    assert [v.aval.dtype for v in p.jaxpr.outvars] == [np.float32, np.int32, np.bool_]


def test_weak_types_follow_jax():
    def item(t, x, key):
        y = x * 3            # f32 * weak int -> f32
        z = (x > 0.5)        # bool
        i = (y * 2).astype(jnp.int32) + 1
        return t.add("h", i, 1.0), i
    p = _prog(item, {"h": tm.Sum((4,))}, [((), np.float32), ((2,), np.uint32)], [], (0, 0))
    assert p.jaxpr.outvars[1].aval.dtype == np.int32
    assert all(e.outvars[0].aval.dtype in (np.float32, np.int32, np.bool_) for e in p.jaxpr.eqns)


def test_python_scalars_take_the_operand_dtype_at_full_precision():
    """a Python float meeting a float64 operand (or a Python int meeting an int64 one) becomes a constant of that
    dtype directly, not through float32 / int32 (JAX's weak typing)."""
    def item(t, x, n):
        t = t.add("f", 0, x * 4e18 + 0.1)
        return t.add("i", 0, n * 4_000_000_000_000_000_000)
    p = _prog(item, {"f": tm.Sum((1,), np.float64), "i": tm.Sum((1,), np.int64)},
              [((), np.float64), ((), np.int64)], [], (0, 0))
    lits = [v.val for e in p.jaxpr.eqns for v in e.invars if isinstance(v, C.Lit) and v.aval.shape == ()]
    assert any(x.dtype == np.float64 and x == 4e18 for x in lits)
    assert any(x.dtype == np.float64 and x == 0.1 for x in lits)
    assert any(x.dtype == np.int64 and x == 4_000_000_000_000_000_000 for x in lits)


def test_tally_read_fork_drop_raise():
    def forked(t, x):
        t1 = t.add("h", 0, x)
        t.add("h", 1, x)
        return t1

    def dropped(t, x):
        t.add("h", 0, x)
        return t

    with pytest.raises(tm.TallyError):
        _prog(forked, {"h": tm.Sum((2,))}, [((), np.float32)], [], (0,))
    with pytest.raises(tm.TallyError):
        _prog(dropped, {"h": tm.Sum((2,))}, [((), np.float32)], [], (0,))


def test_tuple_index_flattening():
    def item(t, i, j):
        return t.add("g", (i, j), 1.0)
    p = _prog(item, {"g": tm.Sum((3, 4))}, [((), np.int32), ((), np.int32)], [], (0, 0))
    prims = [e.prim for e in p.jaxpr.eqns]
    assert "select_n" in prims and "tallymap_emit" in prims


def test_cond_and_fori_trace():
    def item(t, x):
        y = lax.cond(x > 0.5, lambda a: a * 2.0, lambda a: a - 1.0, x)
        s = lax.fori_loop(0, 3, lambda i, a: a + y, 0.0)
        return t.add("h", 0, s)
    p = _prog(item, {"h": tm.Sum((1,))}, [((), np.float32)], [], (0,))
    assert [e.prim for e in p.jaxpr.eqns].count("cond") == 1


def test_uniform_normal_avals():
    def item(t, key):
        u = random.uniform(key, minval=0.2, maxval=0.8)
        n = random.normal(random.fold_in(key, 3))
        return t.add("h", 0, u + n)
    p = _prog(item, {"h": tm.Sum((1,))}, [((2,), np.uint32)], [], (0,))
    prims = [e.prim for e in p.jaxpr.eqns]
    assert prims.count("threefry2x32") == 3 and "erf_inv" in prims


def test_unknown_option_raises():
    with pytest.raises(ValueError):
        tm.vmap(configs.c1_item, outputs=configs.C1["outputs"], bogus=1)


def test_jvp_programs_of_every_config():
    """the forward-mode program of each config (1 and 3 tangent lanes): a tangent tally of the same format per
    float tally, tangent operands after the primal ones, linear tally use, and a gfx950 module that compiles."""
    from tallymap_amd._fwd import jvp_program
    from tallymap_amd.backend import compile as Cm
    from tallymap_amd.backend import kernel as K
    for name in ("c1", "c2", "c3", "c4", "c5"):
        cfg = configs.SIZED[name](8) if name in configs.SIZED else configs.CONFIGS[name]
        args = getattr(configs, f"{name}_inputs")(8)
        axes = cfg["in_axes"]
        pav = [(np.shape(a)[1:], np.asarray(a).dtype) for a, x in zip(args, axes) if x == 0]
        bav = [(np.shape(a), np.asarray(a).dtype) for a, x in zip(args, axes) if x is None]
        p = _prog(cfg["item"], cfg["outputs"], pav, bav, axes, cfg["max_steps"])
        pp = [np.issubdtype(d, np.floating) for _, d in pav]
        pb = [np.issubdtype(d, np.floating) for _, d in bav]
        for lanes in (1, 3):
            q = jvp_program(p, pp, pb, lanes)
            ft = [s for s in p.tallies if s.dtype == np.float32]
            assert [s.name for s in q.tallies[p.nT:]] == [s.name + ("'" if lanes == 1 else f"'{l}")
                                                          for s in ft for l in range(lanes)]
            assert all(t.exact == s.exact and t.shape == s.shape for s in ft for t in q.tallies if
                       t.name.startswith(s.name + "'"))
            assert q.nP == p.nP + sum(pp) * lanes and q.nB == p.nB + sum(pb) * lanes
            assert [v.aval for v in q.jaxpr.invars[:p.nT]] == [v.aval for v in p.jaxpr.invars[:p.nT]]
            if lanes == 1:
                src, L = K.build(q)
                assert L.mode == "step"
                Cm.code_object(src)


def test_jvp_of_a_nested_cond_and_loop():
    """tangents flow through a cond inside the loop body and through a fori_loop carry."""
    from tallymap_amd._fwd import jvp_program

    def item(t, x, a):
        def body(i, c):
            y = lax.cond(c > 0.5, lambda z: z * a, lambda z: z + a, c)
            return y * 0.5
        y = lax.fori_loop(0, 3, body, x)
        return t.add("h", 0, y), y
    p = _prog(item, {"h": tm.Sum((1,))}, [((), np.float32)], [((), np.float32)], (0, None))
    q = jvp_program(p, [False], [True])
    assert q.tangent_ys == [0]
    prims = [e.prim for e in q.jaxpr.eqns]
    assert "while" in prims
    w = next(e for e in q.jaxpr.eqns if e.prim == "while")
    assert len(w.outvars) == len(next(e for e in p.jaxpr.eqns if e.prim == "while").outvars) + 1


def test_records_tracing_and_errors():
    """t.append: hidden field / key tallies of the capacity, a claim per append, the per-item count as a hidden
    per-item result; wrong fields, a float into an integer field and t.add on a Records output raise."""
    from tallymap_amd._tally import FIELD_SEP

    def item(t, x):
        def body(i, t):
            return t.append("r", {"i": i, "v": x * i}, when=x > 0.5)
        return lax.fori_loop(0, 3, body, t), x
    p = _prog(item, {"r": tm.Records({"i": np.int32, "v": np.float32}, capacity=128), "h": tm.Sum((2,))},
              [((), np.float32)], [], (0,))
    names = [s.name for s in p.tallies]
    assert names == ["h", "r" + FIELD_SEP + "i", "r" + FIELD_SEP + "v", "r" + FIELD_SEP + FIELD_SEP + "i", "r" + FIELD_SEP + FIELD_SEP + "k"]
    assert all(s.shape == (128,) for s in p.tallies[1:])
    assert p.records == (("r", 128, (("i", np.dtype(np.int32)), ("v", np.dtype(np.float32)))),)
    assert p.counts == (1,) and p.jaxpr.outvars[p.nT + 1].aval.dtype == np.int32
    w = next(e for e in p.jaxpr.eqns if e.prim == "while")
    assert any(e.prim == "tallymap_claim" for e in w.params["body_jaxpr"].eqns)
    out = {"r": tm.Records({"i": np.int32}, capacity=8)}
    with pytest.raises(TypeError, match="declared fields"):
        _prog(lambda t, x: t.append("r", {"j": 1}), out, [((), np.float32)], [], (0,))
    with pytest.raises(TypeError, match="integer field"):
        _prog(lambda t, x: t.append("r", {"i": x}), out, [((), np.float32)], [], (0,))
    with pytest.raises(KeyError, match="Records output"):
        _prog(lambda t, x: t.add("r", 0, 1), out, [((), np.float32)], [], (0,))
    with pytest.raises(ValueError, match="capacity"):
        tm.Records({"i": np.int32}, capacity=0)
    # without a capacity: the count program (appends only counted, Sums discarded, a count per Records output)
    fc = tm.vmap(item, outputs={"r": tm.Records({"i": np.int32, "v": np.float32}), "h": tm.Sum((2,))}, in_axes=(0,))
    c = fc._prepare((np.ones(4, np.float32),), "count")[0]
    assert c.records == () and len(c.counts) == 1 and [s.kind for s in c.tallies] == ["discard"]
    assert tm.Records(16, {"i": np.int32}) == tm.Records({"i": np.int32}, capacity=16)     # (records.py:461)
    with pytest.raises(TypeError, match="integer"):
        tm.Records({"b": bool}, capacity=4)


def test_spawn_tracing_and_errors():
    """t.spawn: a hidden token tally threaded like an emit, one `tallymap_spawn` per spawn with the child's leaves
    (converted to the mapped inputs' dtypes); the generated kernel stages children per wave, claims their tickets
    per flush and bounds them by the capacity.  Spawn without a Queue, a child of another structure and a float child leaf for an integer input raise
    (reference edge.py:183-188); the jvp program's spawn stores the child's tangents with it; the
    tree adjoint's recording and adjoint programs have the extra columns and operands they need."""
    from tallymap_amd._tally import QKEY
    from tallymap_amd.backend import kernel as K

    def item(t, g, x):
        def body(i, t):
            return t.spawn((g + 1, x * 0.5), when=g < 2)
        return lax.fori_loop(0, 2, body, t.add("h", 0, x))
    f = tm.vmap(item, outputs={"h": tm.Sum((2,))}, spawn=tm.Queue(100))
    g0, xs = np.zeros(10, np.int32), np.ones(10, np.float32)
    p = f._prepare((g0, xs))[0]
    assert p.spawn == 100 and [s.name for s in p.tallies] == ["h", QKEY] and p.tallies[1].kind == "discard"
    w = next(e for e in p.jaxpr.eqns if e.prim == "while")
    sp = [e for e in w.params["body_jaxpr"].eqns if e.prim == "tallymap_spawn"]
    assert len(sp) == 1 and [v.aval.dtype for v in sp[0].invars[2:]] == [np.int32, np.float32]
    src, L = K.build(p)
    # children staged per wave in LDS, one ticket claim per flush, rows past the capacity not stored
    assert "tm_claim(tm_qctr, " in src and "tm_ft < 100ull" in src and "tm_qclaim" not in src.split("tm_main")[1]
    assert len(L.r_q) == 2
    assert "TM_STATS[1] != 0" in src                 # a dropped child poisons the float outputs
    with pytest.raises(ValueError, match="Queue"):
        tm.vmap(lambda t, x: t.spawn(x), outputs={"h": tm.Sum((1,))})._prepare((xs,))
    with pytest.raises(TypeError, match="structure"):
        tm.vmap(lambda t, g, x: t.spawn(x), outputs={"h": tm.Sum((1,))}, spawn=tm.Queue(8))._prepare((g0, xs))
    with pytest.raises(TypeError, match="float spawned child"):
        tm.vmap(lambda t, g, x: t.spawn((x, x)), outputs={"h": tm.Sum((1,))}, spawn=tm.Queue(8))._prepare((g0, xs))
    # Records with spawn: the count pass (no record tallies, a hidden count per Records output) and the fill pass
    # (fields emitted at canonical offsets, an operand per Records output; the Sums discarded; spawn inert)
    fr = tm.vmap(lambda t, x: t.append("r", {"v": x}).spawn(x, when=x > 9.0).add("h", 0, x),
                 outputs={"r": tm.Records({"v": np.float32}, 8), "h": tm.Sum((2,))}, spawn=tm.Queue(8))
    c = fr._prepare((xs,), "record")[0]
    assert c.records == () and len(c.counts) == 1 and [s.name for s in c.tallies] == ["h", QKEY]
    fl = fr._prepare((xs,), "fill")[0]
    assert fl.nP == 2 and fl.spawn is None and [s.kind for s in fl.tallies] == ["discard", "sum", "discard"]
    assert not any(e.prim == "tallymap_spawn" for e in C.walk_eqns(fl.jaxpr))
    # the tree adjoint's programs: the recording forward stores (parent, ordinal) with each child and returns the
    # item's spawn count; the adjoint program takes its first child slot and emits the child's float operands
    r = f._prepare((g0, xs), "record")[0]
    assert r.spawn_mode == "record" and r.qcount == 0 and len(K.build(r)[1].r_q) == 4
    a = f._prepare((g0, xs), "adjoint")[0]
    from tallymap_amd._tally import QF
    assert a.spawn is None and a.nP == 3 and a.p_avals()[2].dtype == np.int32
    assert [s.shape for s in a.tallies if s.name == QF] == [(100,)]
    assert not any(e.prim == "tallymap_spawn" for e in C.walk_eqns(a.jaxpr))
    from tallymap_amd._api import _jvp_prog
    q = _jvp_prog(p, (False, True), (), 2)       # two tangent lanes: the child stores x' of each lane
    w = next(e for e in q.jaxpr.eqns if e.prim == "while")
    sp = [e for e in w.params["body_jaxpr"].eqns if e.prim == "tallymap_spawn"]
    assert q.spawn == 100 and q.nP == 4 and len(sp) == 1 and len(sp[0].invars) == 2 + 4
    with pytest.raises(TypeError, match="Queue"):
        tm.vmap(item, outputs={"h": tm.Sum((2,))}, spawn=100)
    with pytest.raises(ValueError, match="capacity"):
        tm.Queue(0)


def test_tangent_leaves_align_with_primal_leaves():
    """a tangent pytree with None subtrees lines up with the primal's leaves (None per leaf of the subtree)."""
    from tallymap_amd._api import _match_leaves
    prim = dict(a=np.ones(3), b=(np.ones(2), np.ones(4)), c=np.ones(1))
    t = dict(a=None, b=(None, "B1"), c="C")
    assert _match_leaves(prim, t) == [None, None, "B1", "C"]
    assert _match_leaves(prim, None) == [None] * 4


def test_argument_leaves_and_cotangent_structure():
    """reverse mode maps each positional argument to its operand leaves (float32 ones differentiated) and returns
    a cotangent with the argument's structure, None for the other leaves."""
    from tallymap_amd._api import _arg_cotangents, _arg_leaves

    def item(t, p, w):
        return t.add("h", 0, p["x"] * w[0] + p["y"][0])
    p = dict(x=np.ones(8, np.float32), k=np.zeros(8, np.int32), y=np.ones((8, 2), np.float32))
    w = np.ones(3, np.float32)
    f = tm.vmap(item, outputs={"h": tm.Sum((1,))}, in_axes=(0, None))
    prog = f._prepare((p, w))[0]
    spec, wrt = _arg_leaves(prog, (p, w), (0, None), (0, 1))
    assert wrt == ((1, 2), (0,))                  # leaves sorted by key: k (int32), x, y; then w
    g = _arg_cotangents(spec, wrt, ["gx", "gy"], [np.arange(3.0)])
    assert g[0] == {"k": None, "x": "gx", "y": "gy"} and g[1].shape == (3,)


def test_scan_and_switch_trace():
    """lax.scan (unrolled, ys stacked; a long scan without ys as a loop) and lax.switch (a chain of conds, the
    index clamped) trace; a long scan with ys raises."""
    def item(t, x):
        c, ys = lax.scan(lambda c, v: (c + v * x, c * 2.0), 0.0, jnp.stack([x, x + 1.0, x + 2.0]))
        n, _ = lax.scan(lambda c, _: (c + 1, None), 0, length=1000)
        s = lax.switch((x * 3.0).astype(jnp.int32), [lambda v: v, lambda v: v * 2.0, lambda v: v * 3.0], x)
        return t.add("h", 0, c + ys[2] + s), n
    p = _prog(item, {"h": tm.Sum((1,))}, [((), np.float32)], [], (0,))
    prims = [e.prim for e in C.walk_eqns(p.jaxpr)]
    assert prims.count("while") == 1 and prims.count("cond") >= 2
    with pytest.raises(C.TraceError, match="unrolled"):
        _prog(lambda t, x: (t, lax.scan(lambda c, _: (c, c), x, length=1000)[1]), {"h": tm.Sum((1,))},
              [((), np.float32)], [], (0,))


def test_static_loops_are_neither_capped_nor_the_step_loop():
    """A long scan and a static-bound fori_loop are scans in JAX: max_steps does not cap them (no truncation flag,
    no k < max_steps in their cond) and they never become the step loop; a while_loop beside them is both."""
    from tallymap_amd.backend import kernel as K

    def item(t, x):
        c, _ = lax.scan(lambda c, _: (c + x, None), x, length=1000)
        k = lax.fori_loop(0, 300, lambda i, a: a + 1, 0)
        return t.add("h", 0, c), (c, k)
    p = _prog(item, {"h": tm.Sum((1,))}, [((), np.float32)], [], (0,), max_steps=100)
    ws = [e for e in p.jaxpr.eqns if e.prim == "while"]
    assert len(ws) == 2 and all(lax.is_static_loop(e) for e in ws)
    assert all(e.prim != "lt" or all(not (isinstance(v, C.Lit) and v.val == 100) for v in e.invars)
               for w in ws for e in w.params["cond_jaxpr"].eqns)
    tr = p.jaxpr.outvars[len(p.tallies) + p.trunc]
    producer = [e for e in p.jaxpr.eqns if tr in e.outvars][0]
    assert producer.prim == "copy" and isinstance(producer.invars[0], C.Lit) and not producer.invars[0].val
    assert K._split(p.jaxpr) is None                       # (the item schedule: no step loop)

    def item2(t, x):
        c, _ = lax.scan(lambda c, _: (c + x, None), x, length=1000)
        n = lax.while_loop(lambda a: a < c, lambda a: a + 1.0, 0.0)
        return t.add("h", 0, n), n
    p2 = _prog(item2, {"h": tm.Sum((1,))}, [((), np.float32)], [], (0,), max_steps=100)
    w = K._split(p2.jaxpr)
    assert w is not None and not lax.is_static_loop(p2.jaxpr.eqns[w])
    lits = [v.val for e in p2.jaxpr.eqns[w].params["cond_jaxpr"].eqns if e.prim == "lt" for v in e.invars
            if isinstance(v, C.Lit)]
    assert 100 in lits                                     # (the while_loop is capped)

    def item3(t, x):                                       # a traced bound: a while loop, capped
        return t, lax.fori_loop(0, (x * 10.0).astype(jnp.int32), lambda i, a: a + 1, 0)
    p3 = _prog(item3, {"h": tm.Sum((1,))}, [((), np.float32)], [], (0,), max_steps=100)
    assert [lax.is_static_loop(e) for e in p3.jaxpr.eqns if e.prim == "while"] == [False]


def test_scan_of_length_zero_returns_empty_stacked_ys():
    """lax.scan over 0 steps returns the carry unchanged and ys stacked along a leading axis of length 0."""
    got = {}

    def item(t, x):
        c, ys = lax.scan(lambda c, v: (c + v[0], (c * 2.0 + v, (c + v > 0.0).astype(jnp.int32))), x,
                         np.zeros((0, 3), np.float32))
        got["c"], got["ys"] = c, ys
        return t.add("h", 0, c)
    _prog(item, {"h": tm.Sum((1,))}, [((), np.float32)], [], (0,))
    a, b = got["ys"]
    assert np.shape(a) == (0, 3) and np.asarray(a).dtype == np.float32
    assert np.shape(b) == (0, 3) and np.asarray(b).dtype == np.int32
    assert C.is_traced(got["c"])


def test_dynamic_index_traces():
    """x[i] with a traced integer index: one dynamic_index equation after the normalisation and clamp; a float
    index raises."""
    def item(t, x, tab):
        return t.add("h", 0, tab[(x * 10.0).astype(jnp.int32)])
    p = _prog(item, {"h": tm.Sum((1,))}, [((), np.float32)], [((64,), np.float32)], (0, None))
    assert sum(e.prim == "dynamic_index" for e in C.walk_eqns(p.jaxpr)) == 1
    with pytest.raises(C.TraceError, match="integer"):
        _prog(lambda t, x, tab: t.add("h", 0, tab[x]), {"h": tm.Sum((1,))}, [((), np.float32)],
              [((64,), np.float32)], (0, None))


def test_floor_divide_and_remainder_follow_jnp():
    """`//` and `%` trace to JAX's own definitions (jnp.floor_divide / jnp.remainder): signed integers divide with
    lax.div and step down by one where the signs differ and the remainder is nonzero; an integer `%` replaces a zero
    divisor by 1; floats go through rem, the sign correction and round (half away from zero)."""
    def prims(fn, dt):
        p = _prog(lambda t, a, b: (t, fn(a, b)), {}, [((), dt), ((), dt)], [], (0, 0))
        return [e.prim for e in C.walk_eqns(p.jaxpr)], p
    ps, _ = prims(lambda a, b: a // b, np.int32)
    assert ps.count("div") == 1 and ps.count("rem") == 1 and ps.count("sign") == 2 and "select_n" in ps
    ps, _ = prims(lambda a, b: a // b, np.uint32)
    assert ps == ["div"]
    ps, _ = prims(lambda a, b: a % b, np.int32)
    assert ps.count("rem") == 1 and ps.count("select_n") == 2 and "add" in ps
    ps, p = prims(lambda a, b: a // b, np.float32)
    rnd = [e for e in C.walk_eqns(p.jaxpr) if e.prim == "round"]
    assert len(rnd) == 1 and rnd[0].params["rounding_method"] == 0 and ps.count("rem") == 1
    ps, _ = prims(lambda a, b: a % b, np.float32)
    assert ps.count("rem") == 1 and "eq" not in ps           # (no zero-divisor guard for floats)


def test_table_read_cotangents_are_emitted_at_the_row_read():
    """the adjoint programs of an item reading a 1024-row broadcast table at traced indices: the read's cotangent
    leaves by ONE slot-addressed emit where the step's VJP runs (not a select per row and an emit per row at the
    item's end), through the tape adjoint (an active carry) and the forward-only one."""
    from tallymap_amd.backend import reverse as R
    from tallymap_amd.backend import tape as T

    def walk(t, i, x, tab):
        def body(c):
            k, s, t_ = c
            s = s * 0.5 + tab[(i * 7919 + k * 104729) % 1024] * x
            return k + 1, s, t_.add("h", 0, s)
        return lax.while_loop(lambda c: c[0] < 20, body, (0, np.float32(0.0), t))[2]

    def reads(t, i, x, tab):
        def body(c):
            k, t_ = c
            return k + 1, t_.add("h", 0, tab[(i * 7919 + k * 104729) % 1024] * x)
        return lax.while_loop(lambda c: c[0] < 20, body, (0, t))[1]
    pav, bav = [((), np.int32), ((), np.float32)], [((1024,), np.float32)]
    for item, tape in ((walk, True), (reads, False)):
        prog = _prog(item, {"h": tm.Sum((1,))}, pav, bav, (0, 0, None))
        adj = R.adjoint_program(prog, ((), (0,)))
        pl = R.plan(adj)
        assert any(pl.car_act) == tape
        # (the residual tape's reverse program holds the step's VJP twice: from the taped residuals, and from
        # the replayed state in the cold branch of steps past the tape)
        progs = [(T.programs(adj, pl, residual=False).reverse, 1), (T.programs(adj, pl, residual=True).reverse, 2)] \
            if tape else [(R.forward_only_program(adj, pl), 1)]
        for q, n_emit in progs:
            prims = [e.prim for e in C.walk_eqns(q.jaxpr)]
            assert prims.count("tallymap_emit_slot") == n_emit
            assert prims.count("select_n") < 40 and prims.count("tallymap_emit") <= 2


def test_accumulator_carries_need_no_reverse_sweep():
    """a carry whose step is c' = c + d (c read nowhere else in the step, d free of active carries) has the same
    cotangent at every step: the plan marks it an accumulator and the forward-only adjoint handles it (the
    walk-on-spheres estimator's sum); a carry that is also read in the step, scaled, or emitted stays a sweep
    carry (the tape adjoint)."""
    from tallymap_amd.backend import reverse as R

    def item(kind):
        def f(t, x, th):
            def body(c):
                k, y, acc = c
                y = y * 0.5 + x
                d = th * y
                if kind == "acc":
                    acc = acc + d
                elif kind == "read":
                    acc = acc + d * acc
                elif kind == "scaled":
                    acc = acc * 0.9 + d
                return k + 1, y, acc
            k, y, acc = lax.while_loop(lambda c: (c[0] < 8) & (c[2] < 100.0), body, (0, x, th * 2.0))
            return t.add("h", 0, acc * acc), k
        return f

    def emitted(t, x, th):
        def body(c):
            k, acc, t_ = c
            acc = acc + th * x
            return k + 1, acc, t_.add("h", 0, acc)
        return lax.while_loop(lambda c: c[0] < 8, body, (0, np.float32(0.0), t))[2]
    pav, bav = [((), np.float32)], [((), np.float32)]
    for f, want in ((item("acc"), True), (item("read"), False), (item("scaled"), False), (emitted, False)):
        prog = _prog(f, {"h": tm.Sum((1,))}, pav, bav, (0, None))
        pl = R.plan(R.adjoint_program(prog, ((), (0,))))
        assert any(pl.car_act)
        assert (not any(pl.sweep)) == want, f
        if want:
            q = R.forward_only_program(R.adjoint_program(prog, ((), (0,))), pl)
            assert not any(e.prim == "tallymap_tape_put" for e in C.walk_eqns(q.jaxpr))


def _static_item(trips):
    from tallymap_amd import random as R

    def item(t, x, key, th):
        y = lax.fori_loop(0, trips, lambda i, a: a * th + 0.25, x)          # static: PRE work, unrolled for grad

        def body(c):
            k, z, t = c
            u = R.uniform(R.fold_in(key, k))
            t = t.add("h", (u * 8.0).astype(jnp.int32), z * th)
            return k + 1, z * (0.5 + 0.5 * u), t
        k, z, t = lax.while_loop(lambda c: c[1] > 0.05, body, (np.int32(0), y, t))
        return t.add("h", 0, z), k
    return item


def test_static_loop_before_the_step_loop_is_unrolled_for_reverse_mode():
    """grad through a static fori_loop in PRE: the adjoint program has the loop unrolled (3 copies of its body, no
    static while left), the step loop is still the while_loop, and the count and reverse programs build; a lone
    static loop is never taken as the step loop; one of more than 64 trips outside the step loop is refused by
    name."""
    from tallymap_amd import backend as B
    from tallymap_amd.backend import kernel as K
    from tallymap_amd.backend import reverse as Rv
    pav, bav = [((), np.float32), ((2,), np.uint32)], [((), np.float32)]
    p = _prog(_static_item(3), {"h": tm.Sum((8,))}, pav, bav, (0, 0, None))
    assert [lax.is_static_loop(e) for e in p.jaxpr.eqns if e.prim == "while"] == [True, False]
    assert [e.params.get("trips") for e in p.jaxpr.eqns if e.prim == "while"] == [3, None]
    adj, pl = B._adjoint(p, ((0,), (0,)))
    ws = [e for e in adj.prog.jaxpr.eqns if e.prim == "while"]
    assert len(ws) == 1 and not lax.is_static_loop(ws[0])
    sp = Rv.split(adj.prog)
    assert sum(e.prim == "mul" for e in sp.pre.eqns) >= 3
    tp = B._tape_programs(adj, pl, {}, True)
    K.build(tp.count)
    K.build(tp.reverse)

    def lone(t, x, th):
        return t.add("h", 0, lax.fori_loop(0, 5, lambda i, a: a * th, x)), x
    p2 = _prog(lone, {"h": tm.Sum((8,))}, [((), np.float32)], [((), np.float32)], (0, None))
    adj2, pl2 = B._adjoint(p2, ((0,), (0,)))
    assert not any(pl2.sweep) and not any(e.prim == "while" for e in adj2.prog.jaxpr.eqns)

    p3 = _prog(_static_item(100), {"h": tm.Sum((8,))}, pav, bav, (0, 0, None))
    with pytest.raises(Exception, match="static loop of 100 trips"):
        B._adjoint(p3, ((0,), (0,)))


def test_grid_cap_in_the_module():
    """a spawning program's item loop caps its persistent grid at kernel.SPAWN_BLOCKS workgroups per CU (the module's
    tm_grid_cap, read by the launcher); option blocks_per_cu sets the cap of any program; without either the module
    has none (the occupancy sizes the grid)."""
    from tallymap_amd.backend import kernel as K
    from unittest import mock
    from tallymap_amd import backend as B
    seen = []
    orig = K.build

    def fake_build(prog, **kw):
        seen.append(kw.get("grid_cap"))
        return orig(prog, **kw)
    xs = np.ones(10, np.float32)
    g0 = np.zeros(10, np.int32)
    spawn = tm.vmap(lambda t, g, x: t.spawn((g + 1, x), when=g < 1).add("h", 0, x), outputs={"h": tm.Sum((1,))},
                    spawn=tm.Queue(64))
    plain = tm.vmap(lambda t, x: t.add("h", 0, x), outputs={"h": tm.Sum((1,))})
    capped = tm.vmap(lambda t, x: t.add("h", 0, x), outputs={"h": tm.Sum((1,))}, blocks_per_cu=3)
    with mock.patch.object(K, "build", fake_build), mock.patch.object(B, "Cm") as cm:
        cm.code_object.side_effect = RuntimeError("stop")
        for f, args in ((spawn, (g0, xs)), (plain, (xs,)), (capped, (xs,))):
            with pytest.raises(RuntimeError, match="stop"):
                B.compiled(f._prepare(args)[0], f._opts)
    assert seen == [K.SPAWN_BLOCKS, 0, 3]
    assert f"int tm_grid_cap = {K.SPAWN_BLOCKS};" in K.build(spawn._prepare((g0, xs))[0], grid_cap=K.SPAWN_BLOCKS)[0]
    assert "tm_grid_cap" not in K.build(plain._prepare((xs,))[0])[0]


@pytest.mark.parametrize("dt", [np.float32, np.float64], ids=["f32", "f64"])
def test_transcendentals_lower_to_the_glibc_restatements(dt):
    """Every transcendental with a glibc-bitwise restatement in tm_libm.h is emitted as a call to it (the device
    library's own function only for the rest), and every tm_* name the table routes to exists in the header."""
    import os
    import re
    from tallymap_amd.backend import codegen as G
    from tallymap_amd.backend import kernel as K
    unary = ["exp", "exp2", "log", "log1p", "expm1", "log2", "sin", "cos", "tan", "asin", "acos", "atan", "sinh",
             "cosh", "tanh", "asinh", "acosh", "atanh", "cbrt", "erf", "erfc", "lgamma", "logistic", "erf_inv"]
    binary = ["pow", "atan2"]

    def item(t, x):
        vals = [getattr(lax, n)(x[j]) for j, n in enumerate(unary)]
        vals += [getattr(lax, n)(x[len(unary) + j], x[0]) for j, n in enumerate(binary)]
        return t, tuple(vals)
    n = len(unary) + len(binary)
    src, _ = K.build(_prog(item, {}, [((n,), dt)], [], (0,)))
    t = "float" if dt == np.float32 else "double"
    hdr = open(os.path.join(os.path.dirname(G.__file__), "..", "csrc", "tm_libm.h")).read()
    for name in unary + binary:
        fn = G.LIBM[(name, t)]
        assert re.search(r"\b" + re.escape(fn) + r"\(", src), (name, fn)
        if fn.startswith("tm_"):
            assert f"TM_FN {t} {fn}(" in hdr, fn
    glibc_bitwise = {n for n in unary + binary if G.LIBM[(n, t)].startswith("tm_")}
    rest = {"cbrt"} if dt == np.float32 else {"sin", "cos", "tan", "asin", "acos", "atan", "atan2", "cbrt"}
    assert set(unary + binary) - glibc_bitwise == rest


class _Listed:
    """an array whose shape is a list, as some array libraries give it."""
    def __init__(self, a):
        self.a, self.shape, self.dtype = a, list(a.shape), a.dtype


class _Grid(dict):
    """a container of operands with attributes that an array has too."""
    shape, dtype = (4,), np.dtype(np.float32)


def test_a_repeated_call_is_found_by_arrays_alone():
    """a call's program is looked up by its arguments' shapes and types; an argument whose shape cannot be a key, or a
    container that has attributes of these names, is described in full each time."""
    x = np.ones(4, np.float32)
    f = tm.vmap(lambda t, x: t.add("h", 0, x), outputs={"h": tm.Sum((1,))})
    p = f._prepare((x,))[0]
    assert f._prepare((x + 1,))[0] is p and f._prepare((_Listed(x),))[0] is p and f._prepare((_Listed(x),))[4] == 4
    g = tm.vmap(lambda t, x: t.add("h", 0, x["a"]), outputs={"h": tm.Sum((1,))})
    for n in (4, 6, 4):
        got = g._prepare((_Grid(a=np.ones(n, np.float32)),))
        assert got[4] == n and got[2][0].shape == (n,)
    for dt in (np.float32, np.int32):
        assert g._prepare((_Grid(a=np.ones(4, dt)),))[0].p_avals()[0].dtype == dt
