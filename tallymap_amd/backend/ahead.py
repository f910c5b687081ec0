"""Which part of a loop step can be computed ahead of its turn.

A step of most random programs is a hash of the item's key and the step index, a few transcendentals of the draws,
and a short update of the item's state by them.  Everything up to the update depends on the step only through its
counters (carries that gain a constant per step): the value for step k + g is known at step k.  When fewer items
than lanes are left -- a small call, or the tail of a large one -- the kernel gives each item a power of two of
lanes: lane g of the group computes the values of step k + g, then the group runs that many updates, each reading
its values from the lane that computed them (kernel.py's tail loop).  A step then takes the latency of its update
and a share of the rest, where it took the whole chain.

`plan` splits the step's equations:
  inv     from loop constants alone: emitted on both sides (the compiler takes them out of the loops)
  ahead   from counters and loop constants by pure primitives, and by loops whose trip count is a literal: the ahead
          side also runs for steps past the item's last, and a loop that ends for every counter the item reaches need
          not end for those
  cheap   the ahead equations of a couple of instructions whose operands the update has anyway (a counter's own
          increment): recomputed there
  update  the rest
and lists the values that pass from ahead to update (`cut`)."""
import dataclasses

import numpy as np

from .. import _core as C
from . import simplify

MIN_COST = 64              # instructions (kernel.cost) the ahead part has to save per step: about one hash
MAX_WORDS = 16             # 32-bit words that pass per step (a register and a cross-lane read each)
PURE = simplify.PURE | {"tallymap_item_index", "tallymap_sincos"}


@dataclasses.dataclass
class Plan:
    ahead: list            # equations of the ahead side (inv included), in order
    update: list           # equations of the update side (inv and cheap included), in order
    cut: list              # variables passed from ahead to update
    counters: dict         # carry index -> its gain per step


def pure(e):
    """whether e computes values alone (no tally, tape, queue or record effect)."""
    if e.prim in ("while", "cond"):
        return all(pure(x) for j in C.subjaxprs(e) for x in j.eqns)
    return e.prim in PURE or (not C.subjaxprs(e) and not e.prim.startswith("tallymap_"))


def bounded(e):
    """whether e ends whatever its operands: every loop in it has a literal trip count."""
    if e.prim == "while" and not e.params.get("static", False):
        return False
    return all(bounded(x) for j in C.subjaxprs(e) for x in j.eqns)


def _counters(bj, nb):
    """{carry index: gain} of the scalar 32-bit integer carries that gain a literal per step."""
    by = {o.id: e for e in bj.eqns for o in e.outvars}
    out = {}
    for j, (v, o) in enumerate(zip(bj.invars[nb:], bj.outvars)):
        e = by.get(o.id) if isinstance(o, C.Var) else None
        if e is None or e.prim != "add" or e.outvars[0].aval.shape != () or e.outvars[0].aval.dtype not in (C.I32, C.U32):
            continue
        a, b = e.invars
        if isinstance(a, C.Lit):
            a, b = b, a
        if isinstance(a, C.Var) and a.id == v.id and isinstance(b, C.Lit):
            out[j] = int(np.asarray(b.val).reshape(-1)[0])
    return out


def plan(we, is_tally, cost):
    """the Plan of loop equation `we`, or None where computing ahead would not pay.  is_tally(v): whether an operand
    of the loop is a tally; cost: kernel.cost."""
    bj, nb = we.params["body_jaxpr"], we.params["body_nconsts"]
    nc = we.params["cond_nconsts"]
    ops = we.invars[nc:]
    counters = _counters(bj, nb)
    kind = {}              # variable -> inv | counter | ahead | cheap | update
    for j, v in enumerate(bj.invars):
        c = j - nb
        if is_tally(ops[j]):
            kind[v.id] = "update"
        elif c < 0 or (isinstance(bj.outvars[c], C.Var) and bj.outvars[c].id == v.id):
            kind[v.id] = "inv"
        else:
            kind[v.id] = "counter" if c in counters else "update"
    ahead, update = [], []
    for e in bj.eqns:
        ks = {kind[v.id] for v in e.invars if isinstance(v, C.Var)}
        if "update" in ks or not pure(e) or not bounded(e):
            k = "update"
        elif ks <= {"inv"}:
            k = "inv"
        elif ks <= {"inv", "counter", "cheap"} and cost([e]) <= 2 and not C.subjaxprs(e):
            k = "cheap"
        else:
            k = "ahead"
        for o in e.outvars:
            kind[o.id] = k
        if k != "update":
            ahead.append((k, e))
        if k != "ahead":
            update.append((k, e))
    used = {v.id for k, e in update if k == "update" for v in e.invars if isinstance(v, C.Var)}
    used |= {v.id for v in bj.outvars if isinstance(v, C.Var)}
    cut = [o for k, e in ahead if k == "ahead" for o in e.outvars if o.id in used]
    words = sum(max(1, v.aval.size) * (2 if v.aval.dtype.itemsize == 8 else 1) for v in cut)
    # (the ahead equations some cut value needs; the compiler drops the others)
    need, saved = {v.id for v in cut}, []
    for k, e in reversed(ahead):
        if any(o.id in need for o in e.outvars):
            need |= {v.id for v in e.invars if isinstance(v, C.Var)}
            if k == "ahead":
                saved.append(e)
    if not cut or words > MAX_WORDS or cost(saved) < MIN_COST:
        return None
    return Plan([e for _, e in ahead], [e for _, e in update], cut, counters)
