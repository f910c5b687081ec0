"""Common-subexpression elimination over item programs, before they are emitted.

The adjoint programs repeat work by construction: value_and_grad's fused program runs POST and then POST's VJP,
which re-evaluates POST's primal values on the same loop results; a forward-only adjoint's loop body runs the step
and the step's VJP, which recomputes the step's primal values.  Equations of a pure primitive with the same
operands (the same variables, or equal literals), the same parameters and the same result types compute the same
values, so the later one is dropped and its results renamed to the earlier one's.  The device compiler removes
some of these itself, but not where the duplicate sits after a global atomic or a loop whose memory effects it
cannot see through (a libm table load after a store is not provably the same load).

Scopes: every jaxpr (a while's cond and body, a cond's branches) is processed on its own, since the item IR's
sub-jaxprs are closed (their operands are passed in).  The top-level program is cut at its step loop: PRE and POST
are separate scopes, so a POST equation is never renamed to a PRE result, which would keep that value live in a
register through the whole loop.
"""
import numpy as np

from .. import _core as C
from .codegen import EW

# primitives whose results are functions of their operands and parameters alone (no tally, tape, queue or record
# effects, no per-launch state)
PURE = set(EW) | {"integer_pow", "round", "convert_element_type", "bitcast_convert_type", "select_n", "copy",
                  "stop_gradient", "tallymap_ct_read", "threefry2x32", "slice", "dynamic_index", "squeeze",
                  "reshape", "broadcast_in_dim", "concatenate"}


def _pkey(x):
    """a hashable key of a parameter value (None: not keyable, the equation is left alone)."""
    if isinstance(x, (bool, int, float, str, type(None), np.dtype)):
        return (type(x).__name__, x)
    if isinstance(x, np.generic):
        return ("np", x.dtype.str, x.tobytes())
    if isinstance(x, np.ndarray):
        return ("arr", x.dtype.str, x.shape, x.tobytes())
    if isinstance(x, (tuple, list)):
        ks = tuple(_pkey(y) for y in x)
        return None if any(k is None for k in ks) else ("seq", ks)
    if isinstance(x, type) and issubclass(x, np.generic):
        return ("npt", np.dtype(x).str)
    return None


def _vkey(v):
    if isinstance(v, C.Lit):
        a = np.asarray(v.val)
        return ("lit", v.aval.dtype.str if hasattr(v.aval.dtype, "str") else str(v.aval.dtype), a.shape,
                a.tobytes(), bool(getattr(v.aval, "weak", False)))
    return ("var", v.id)


def _akey(a):
    return (tuple(a.shape), str(a.dtype))


def cse(jx, cut=None):
    """-> jx with repeated pure equations removed (the same Jaxpr object when nothing changes).  cut: the index of
    an equation (the step loop) that separates two scopes; the equation itself is kept and processed."""
    sub = {}
    eqns = []
    seen = {}
    changed = False

    def r(v):
        return sub.get(v.id, v) if isinstance(v, C.Var) else v

    for i, e in enumerate(jx.eqns):
        if i == cut:
            seen = {}
        ins = [r(v) for v in e.invars]
        params = e.params
        if C.subjaxprs(e):
            new = {}
            for k, p in e.params.items():
                if isinstance(p, C.Jaxpr):
                    p2 = cse(p)
                elif isinstance(p, (list, tuple)) and any(isinstance(x, C.Jaxpr) for x in p):
                    xs = [cse(x) if isinstance(x, C.Jaxpr) else x for x in p]
                    p2 = p if all(a is b for a, b in zip(xs, p)) else type(p)(xs)
                else:
                    p2 = p
                new[k] = p2
            if any(new[k] is not p for k, p in e.params.items()):
                params = new
        if e.prim in PURE and params is e.params:
            pk = tuple(sorted((k, _pkey(p)) for k, p in params.items()))
            if all(k[1] is not None for k in pk):
                key = (e.prim, tuple(_vkey(v) for v in ins), pk, tuple(_akey(o.aval) for o in e.outvars))
                prev = seen.get(key)
                if prev is not None:
                    for o, p in zip(e.outvars, prev):
                        sub[o.id] = p
                    changed = True
                    continue
                seen[key] = e.outvars
        if i == cut:
            seen = {}
        if params is not e.params or any(a is not b for a, b in zip(ins, e.invars)):
            e = C.Eqn(e.prim, ins, e.outvars, params)
            changed = True
        eqns.append(e)
    if not changed:
        return jx
    return C.Jaxpr(jx.invars, [r(v) for v in jx.outvars], eqns)


def _map_subs(e, f):
    """e with f applied to each of its sub-programs (the same equation when nothing changes)."""
    new = {}
    for k, p in e.params.items():
        if isinstance(p, C.Jaxpr):
            new[k] = f(p)
        elif isinstance(p, (list, tuple)) and any(isinstance(x, C.Jaxpr) for x in p):
            xs = [f(x) if isinstance(x, C.Jaxpr) else x for x in p]
            new[k] = p if all(a is b for a, b in zip(xs, p)) else type(p)(xs)
        else:
            new[k] = p
    if all(new[k] is p for k, p in e.params.items()):
        return e
    return C.Eqn(e.prim, e.invars, e.outvars, new)


def pair_sincos(jx, cut=None):
    """sin x and cos x of one float32 x in a jaxpr (on one side of `cut`) -> one tallymap_sincos equation (two results):
    the reduction and the polynomials of the two calls are the same values, which the device compiler does not share
    (they sit in two divergent branches).  Programs that draw a direction, and the derivatives of either function,
    hold such pairs."""
    eqns = [_map_subs(e, pair_sincos) for e in jx.eqns]
    first = {}                      # x -> index of the first of the pair
    drop = set()
    for i, e in enumerate(eqns):
        if i == cut:
            first = {}
        if e.prim not in ("sin", "cos") or e.outvars[0].aval.dtype != C.F32 or not isinstance(e.invars[0], C.Var):
            continue
        k = e.invars[0].id
        j = first.setdefault(k, i)
        if j == i or eqns[j].prim not in ("sin", "cos") or eqns[j].prim == e.prim:
            continue
        a, b = (eqns[j], e) if eqns[j].prim == "sin" else (e, eqns[j])
        eqns[j] = C.Eqn("tallymap_sincos", [e.invars[0]], [a.outvars[0], b.outvars[0]], {})
        drop.add(i)
    if not drop and all(a is b for a, b in zip(eqns, jx.eqns)):
        return jx
    return C.Jaxpr(jx.invars, jx.outvars, [e for i, e in enumerate(eqns) if i not in drop])


def drop_draw_clamp(jx):
    """max(lo, f * span + lo) -> f * span + lo, where f = (bits >> 9 | 1.0f's bits) as a float - 1 and span >= 0
    (jax.random.uniform's clamp): f is in [0, 1), so f * span + lo >= lo in float32 too (rounding is monotonic), never
    -0 for lo = 0, and the max is its operand."""
    eqns = [_map_subs(e, drop_draw_clamp) for e in jx.eqns]
    by = {o.id: e for e in eqns for o in e.outvars}

    def lit(v):
        return float(np.asarray(v.val).reshape(-1)[0]) if isinstance(v, C.Lit) and np.asarray(v.val).size == 1 else None

    def of(v, prim):
        e = by.get(v.id) if isinstance(v, C.Var) else None
        return e if e is not None and e.prim == prim else None

    def pick(e, f):
        """the (literal, other operand) of a binary equation with f(other) true, else (None, None)."""
        for a, b in (e.invars, e.invars[::-1]):
            if lit(a) is not None and isinstance(b, C.Var) and f(b):
                return lit(a), b
        return None, None

    def unit(v):
        """v = bitcast(shift_right_logical(bits, 9) | 0x3F800000) - 1"""
        e = of(v, "sub")
        e = of(e.invars[0], "bitcast_convert_type") if e is not None and lit(e.invars[1]) == 1.0 else None
        e = of(e.invars[0], "or") if e is not None and e.outvars[0].aval.dtype == C.F32 else None
        if e is None:
            return False
        c, x = pick(e, lambda b: of(b, "shift_right_logical") is not None)
        return c == 0x3F800000 and lit(of(x, "shift_right_logical").invars[1]) == 9.0

    def clamped(e):
        """the operand that max equation e returns, or None."""
        if e.prim != "max" or e.outvars[0].aval.dtype != C.F32 or e.outvars[0].aval.shape != ():
            return None
        lo, s = pick(e, lambda b: of(b, "add") is not None)
        if lo is None or not np.isfinite(lo) or (lo == 0.0 and np.signbit(lo)):
            return None
        lo2, m = pick(of(s, "add"), lambda b: of(b, "mul") is not None)
        if lo2 != lo or np.signbit(lo2) != np.signbit(lo):
            return None
        span, _ = pick(of(m, "mul"), unit)
        return s if span is not None and 0.0 <= span < np.inf else None

    sub, out = {}, []
    for e in eqns:
        if any(isinstance(v, C.Var) and v.id in sub for v in e.invars):
            e = C.Eqn(e.prim, [sub.get(v.id, v) if isinstance(v, C.Var) else v for v in e.invars], e.outvars, e.params)
        s = clamped(e)
        if s is not None:
            sub[e.outvars[0].id] = s
            continue
        out.append(e)
    if not sub and all(a is b for a, b in zip(eqns, jx.eqns)):
        return jx
    return C.Jaxpr(jx.invars, [sub.get(v.id, v) if isinstance(v, C.Var) else v for v in jx.outvars], out)
