"""The user contract: Sum, Result, STATS, ItemProgram and vmap (reference tallymap/_api.py).

`vmap(item, outputs={name: Sum(shape)}, in_axes=..., max_steps=...)` returns `mapped(*args)`.  A call traces the
item once per argument signature into an ItemProgram (invars [tallies] + [per-item operands] + [broadcast
operands]; outvars [tallies] + [per-item results] (+ [truncated])), checks that the tallies are used linearly,
and launches the HIP kernel backend (tallymap_amd.backend).  Its meaning is the reference's: jax.vmap(item) over
the items followed by a sum of their tallies, with the resource-limit poison of _api.py:898-958 (any truncated
item makes every float tally NaN; integer tallies are left alone).
"""
import collections
import dataclasses
import hashlib

import numpy as np

from . import _core as C
from . import lax as L
from ._tally import Tally
from ._tree import flatten, unflatten

STATS = ("spawned", "children_dropped", "children_truncated", "fixed_point_overflow", "dropped_emits")
ST = {n: i for i, n in enumerate(STATS)}
MAX_ITEMS = 2 ** 31 - 1
SUM_DTYPES = (C.F32, C.F64, C.I32, C.U32, C.I64, C.U64)
PROG_CACHE = 64
OPTS = ("schedule", "block", "cuda_math", "min_blocks_per_sm", "rev_checkpoints", "refill", "compact", "rev_schedule",
        "rev_tape", "rev_refill", "rev_residual", "rev_record", "post_batch", "lds_tables", "grad_mode",
        "blocks_per_cu")


class UnsupportedError(NotImplementedError):
    """the backend cannot run this program (it never falls back: reference _api.py:198-200)."""


class TallyError(TypeError):
    """a tally used non-linearly: read, forked or dropped (reference _rewrite.py:31)."""


@dataclasses.dataclass(frozen=True)
class Sum:
    """a commutative (sum) output of `shape` and `dtype` (reference _api.py:55-84); dtype float32, float64, int32,
    uint32, int64 or uint64.

    fixed_point=True with float32 is the EXACT sum: each bin the correctly rounded f32 of the exact sum of every
    finite value emitted into it (`scale` unused); a non-finite emit or a total beyond float32 makes the bin NaN,
    counted in stats['fixed_point_overflow'].
    fixed_point=True with another dtype accumulates round(v * scale) (nearest, ties to even) in an int64 low word
    with a signed carry word, so a bin's total is exact past 2^63 / scale and bitwise independent of the order of
    the emits; the output is that total / scale in `dtype`.  An emit with |v * scale| >= 9.2e18 is dropped, counted
    in 'fixed_point_overflow', and makes its bin NaN (a float output); a total that does not fit `dtype` is counted
    there too (a float output is NaN, an integer one saturates)."""
    shape: object
    dtype: object = np.float32
    fixed_point: bool = False
    scale: float = 2.0 ** 32


class Records:
    """A Records output (reference _api.py:101-140): each item appends records with
    ``t = t.append(name, {field: value, ...}, when=...)``.

        Records({"sensor": np.int32, "t": np.float32}, capacity=1 << 20)   (or Records(capacity, fields))

    Result.outputs[name] is {field: array[capacity]}: the concatenation over items, in item order, of each item's
    records in the order it appended them (record k of item i at slot offset[i] + k, offset the exclusive prefix
    sum of the per-item counts); slots past the last record are zero.  Result.stats['appended'][name] is the number
    of records (exact also beyond the capacity) and stats['records_dropped'][name] the number that did not fit.  A
    call in which any Records output receives more than its capacity (or any item is truncated) makes every float
    output of the call NaN (records and sums) and every integer record field -1.  Without a capacity, each call
    first runs a count pass and sizes the output to the next power of two at or above its record count (reference
    _api.py:838-852).  Fields are scalars of float32, float64, int32, uint32, int64 or
    uint64; float fields carry tangents (jvp, jacfwd).  One pass: each append claims a raw slot with one atomic and
    the same launch moves the records to the canonical slots (reference _records.py)."""

    def __init__(self, fields, capacity=None):
        if isinstance(fields, (int, np.integer)) and isinstance(capacity, dict):
            fields, capacity = capacity, fields
        if not isinstance(fields, dict) or not fields:
            raise TypeError("tallymap: Records(fields, capacity): fields is a non-empty {name: dtype} dict")
        fl = {str(k): np.dtype(v) for k, v in fields.items()}
        for k, dt in fl.items():
            if dt == np.bool_:
                raise TypeError(f"tallymap: Records field {k!r} of dtype bool: use an integer dtype (0 / 1)")
        if capacity is not None:
            capacity = int(capacity)
            if not 0 < capacity <= MAX_ITEMS:
                raise ValueError(f"tallymap: Records capacity must be in [1, 2^31 - 1], got {capacity}")
        self.fields = fl
        self.capacity = capacity

    def __eq__(self, o):
        return isinstance(o, Records) and o.fields == self.fields and o.capacity == self.capacity

    def __hash__(self):
        return hash((tuple(self.fields.items()), self.capacity))

    def __repr__(self):
        return f"Records({ {k: v.name for k, v in self.fields.items()} }, capacity={self.capacity})"


@dataclasses.dataclass(frozen=True)
class Queue:
    """The spawn queue of `capacity` pending children (reference _api.py:88-96): with vmap(..., spawn=Queue(Q)) an
    item may call t = t.spawn(child, when=...), a new item with the per-item inputs `child` (the structure of the
    mapped arguments) that runs the same function on the same broadcast arguments; its per-item result is
    discarded.  This backend runs the children generation by generation: every launch's children wait in a buffer
    of Q slots and become the next launch's items.  A child beyond Q in one generation is dropped and counted in
    stats['children_dropped'], and the call's float outputs are NaN (never a silently truncated shower; integer
    outputs cannot be NaN and are left as they are).  stats['spawned'] counts the children that ran and
    stats['children_truncated'] those that hit max_steps (which poisons like a truncated item)."""
    capacity: int

    def __post_init__(self):
        if not 0 < int(self.capacity) <= MAX_ITEMS:
            raise ValueError(f"tallymap: Queue capacity must be in [1, 2^31 - 1], got {self.capacity}")


class Result(collections.namedtuple("Result", "outputs per_item truncated stats")):
    """outputs: {name: summed output}; per_item: per-item results (None if the item returns only its tally);
    truncated: bool[N]; stats: {name: int32 scalar} (reference _api.py:180-189)."""


@dataclasses.dataclass(frozen=True)
class TSpec:
    name: str
    shape: tuple
    dtype: np.dtype
    exact: bool = False
    kind: str = "sum"          # 'sum' | 'discard' (a derived program's tally that is not output)
    fixed: bool = False        # the scaled fixed-point sum (Sum(fixed_point=True) of a dtype other than float32)
    scale: float = 0.0

    @property
    def S(self):
        return int(np.prod(self.shape, dtype=np.int64))


@dataclasses.dataclass(eq=False)
class ItemProgram:
    """jaxpr invars: [tallies] + [per-item operands] + [broadcast operands]; outvars: [tallies (same slots)] +
    [per-item results]; trunc: index of the truncation flag among the per-item results (None: no cap)."""
    jaxpr: C.Jaxpr
    tallies: tuple
    nP: int
    nB: int
    trunc: object = None
    tag: str = "primal"
    where: str = ""
    records: tuple = ()        # ((name, capacity, ((field, dtype), ...)), ...): the Records outputs
    counts: tuple = ()         # per Records output: the index among the per-item results of its per-item count
    spawn: int = None          # the spawn Queue's capacity (None: the item cannot spawn)
    spawn_mode: str = None     # the tree adjoint's programs: 'record' (children also store parent and ordinal) or
                               # 'adjoint' (spawns emit into the child-slot tally; per-item operand `off` last)
    qcount: int = None         # 'record': the index among the per-item results of the item's spawn count

    @property
    def nT(self):
        return len(self.tallies)

    def y_avals(self):
        return [v.aval for v in self.jaxpr.outvars[self.nT:]]

    def p_avals(self):
        a = self.__dict__.get("_pav")
        if a is None:
            a = self.__dict__["_pav"] = [v.aval for v in self.jaxpr.invars[self.nT:self.nT + self.nP]]
        return a

    def b_avals(self):
        a = self.__dict__.get("_bav")
        if a is None:
            a = self.__dict__["_bav"] = [v.aval for v in self.jaxpr.invars[self.nT + self.nP:]]
        return a

    @property
    def out_tallies(self):
        return [k for k, s in enumerate(self.tallies) if s.kind == "sum"]

    def digest(self):
        d = self.__dict__.get("_digest")
        if d is None:
            d = self.__dict__["_digest"] = digest(self.jaxpr, self.tallies, (self.nP, self.nB, self.trunc, self.tag,
                                                                            repr(self.records), self.counts,
                                                                            self.spawn, self.spawn_mode, self.qcount))
        return d


# ----------------------------------------------------------------------------------------- tally checks
TALLY_OPS = ("tallymap_emit", "tallymap_claim", "tallymap_put", "tallymap_spawn",     # operand 0: the tally threaded
             "tallymap_tape_put")


def check_tallies(jx, nT, where=""):
    """every tally value is used exactly once, only to thread it: by an emit (its operand 0), as a while / cond
    carry, or as a program output (reference _rewrite.py:41-56).  Raises TallyError."""
    pos = _flow(jx, {v.id for v in jx.invars[:nT]}, where)
    if pos != set(range(nT)):
        raise TallyError(f"tallymap: the item function {where} must return its tally (the last t = t.add(...))")


def _flow(jx, tin, where, allow_drop=False):
    """validate the tally use of jx, whose invars with ids in `tin` are tallies -> the indices of jx.outvars that
    are tallies."""
    tv, used = set(tin), set()

    def consume(v):
        if v.id in used:
            raise TallyError(f"tallymap: a tally is used twice (forked) in the item function {where}")
        used.add(v.id)
    for e in jx.eqns:
        for j, v in enumerate(e.invars):
            if isinstance(v, C.Var) and v.id in tv:
                if not ((e.prim in TALLY_OPS and j == 0)
                        or e.prim in ("while", "cond", "copy")):
                    raise TallyError(f"tallymap: a tally is read by `{e.prim}` in the item function {where}: "
                                     "tallies are write-only (t = t.add(...)), used linearly")
        if e.prim in TALLY_OPS:
            consume(e.invars[0])
            tv.add(e.outvars[0].id)
        elif e.prim == "copy":
            if isinstance(e.invars[0], C.Var) and e.invars[0].id in tv:
                consume(e.invars[0])
                tv.add(e.outvars[0].id)
        elif e.prim == "while":
            nc, nb = e.params["cond_nconsts"], e.params["body_nconsts"]
            if any(isinstance(v, C.Var) and v.id in tv for v in e.invars[:nc + nb]):
                raise TallyError(f"tallymap: a loop closes over a tally in {where}: thread it as a carry")
            init = e.invars[nc + nb:]
            flags = [isinstance(v, C.Var) and v.id in tv for v in init]
            for v, f in zip(init, flags):
                if f:
                    consume(v)
            bj, cj = e.params["body_jaxpr"], e.params["cond_jaxpr"]
            got = _flow(bj, {v.id for v, f in zip(bj.invars[nb:], flags) if f}, where)
            if got != {k for k, f in enumerate(flags) if f}:
                raise TallyError(f"tallymap: a loop body does not return its tally carries in place in {where}")
            _flow(cj, {v.id for v, f in zip(cj.invars[nc:], flags) if f}, where, allow_drop=True)
            for o, f in zip(e.outvars, flags):
                if f:
                    tv.add(o.id)
        elif e.prim == "cond":
            nco = e.params["nconsts"]
            if any(isinstance(v, C.Var) and v.id in tv for v in e.invars[1:1 + nco]):
                raise TallyError(f"tallymap: a cond branch closes over a tally in {where}: pass it as an operand")
            ops = e.invars[1 + nco:]
            flags = [isinstance(v, C.Var) and v.id in tv for v in ops]
            for v, f in zip(ops, flags):
                if f:
                    consume(v)
            outs = None
            for br in e.params["branches"]:
                got = _flow(br, {v.id for v, f in zip(br.invars[nco:], flags) if f}, where)
                if outs is not None and got != outs:
                    raise TallyError(f"tallymap: the branches of a cond return tallies in different slots in {where}")
                outs = got
            if len(outs) != sum(flags):
                raise TallyError(f"tallymap: a cond branch drops or duplicates a tally in {where}")
            for k in outs:
                tv.add(e.outvars[k].id)
    for o in jx.outvars:
        if isinstance(o, C.Var) and o.id in tv:
            consume(o)
    if not allow_drop and tv - used:
        raise TallyError(f"tallymap: a tally update is dropped in the item function {where}: return the last "
                         "tally (t = t.add(...) returns a NEW tally)")
    return {i for i, o in enumerate(jx.outvars) if isinstance(o, C.Var) and o.id in tv}


# -------------------------------------------------------------------------------------------- digests
def _pval(v):
    if isinstance(v, C.Jaxpr):
        return ("J", _jx_key(v))
    if isinstance(v, (tuple, list)):
        return tuple(_pval(x) for x in v)
    if isinstance(v, np.dtype):
        return v.name
    return repr(v)


def _jx_key(jx):
    names = {}

    def nm(v):
        if isinstance(v, C.Lit):
            return ("L", v.aval.dtype.name, v.aval.shape, v.val.tobytes())
        return names.setdefault(v.id, ("V", len(names), v.aval.dtype.name, v.aval.shape))
    key = [tuple(nm(v) for v in jx.invars)]
    for e in jx.eqns:
        key.append((e.prim, tuple(nm(v) for v in e.invars), tuple(nm(v) for v in e.outvars),
                    tuple(sorted((k, _pval(x)) for k, x in e.params.items()))))
    key.append(tuple(nm(v) for v in jx.outvars))
    return tuple(key)


def digest(jx, tallies=(), extra=()):
    """structural sha256 of a program (reference _jaxpr.py:301-309): variable names are canonical, literals by
    their bytes."""
    h = hashlib.sha256(repr((_jx_key(jx), tuple((s.name, s.shape, s.dtype.name, s.exact, s.kind, s.fixed,
                                                   s.scale) for s in tallies), extra)).encode())
    return h.hexdigest()


# ---------------------------------------------------------------------------------------------- vmap
_PROGS = collections.OrderedDict()


_NPDT = {}


def _np_dtype(x):
    dt = getattr(x, "dtype", None)
    if dt is None:
        return np.asarray(x).dtype
    hit = _NPDT.get(dt)
    if hit is None:
        name = str(dt)
        hit = np.dtype(name.replace("torch.", "").replace("bool", "bool_")) if name.startswith("torch.") \
            else np.dtype(dt)
        _NPDT[dt] = hit
    return hit


def _shape(x):
    sh = getattr(x, "shape", None)
    if sh is None:
        return np.shape(x)
    return sh if type(sh) is tuple else tuple(int(s) for s in sh)


def item_name(fn):
    code = getattr(fn, "__code__", None)
    q = getattr(fn, "__qualname__", repr(fn))
    return f"{q} ({code.co_filename}:{code.co_firstlineno})" if code else q


def build_program(fn, outs_spec, axes, pav, bav, max_steps, ptree=None, btree=None, spawn=None, ctree=None,
                  spawn_mode=None):
    """trace `fn(tally, *args)` into an ItemProgram.  pav / bav: per-item / broadcast operand avals (leaves);
    spawn: the Queue capacity (ctree: the structure a spawned child must have); spawn_mode: None, or a derived
    program: 'record' (the recording forward of a spawning item: children store parent and ordinal; Records appends
    are only counted), 'adjoint' (spawns and Records appends emit their float values at canonical slots, the
    offsets being per-item operands) or 'fill' (Records with spawn: every field emitted at its canonical slot, the
    Sums discarded, spawns inert)."""
    from ._tally import KI, KK, QF, QKEY, RADJ, FIELD_SEP, rkey
    tspecs = []
    recs = []
    # how appends run: one pass (claimed raw slots), only counted, or emitted at canonical offsets (operands)
    rmode = ({None: None, "record": "count" if spawn is not None else None, "adjoint": "adjoint", "fill": "fill",
              "count": "count"}[spawn_mode])
    for n in sorted(outs_spec):
        s = outs_spec[n]
        if FIELD_SEP in n:
            raise ValueError(f"tallymap: output name {n!r} contains a reserved character")
        if isinstance(s, Records):
            fields = tuple(s.fields.items())
            for f, dt in fields:
                if dt not in SUM_DTYPES:
                    raise UnsupportedError(f"tallymap: Records field {n}.{f} of dtype {dt}: supported are "
                                           f"{', '.join(d.name for d in SUM_DTYPES)}")
                if rmode == "adjoint":                 # (the adjoint program: float fields at canonical slots)
                    if dt == C.F64:
                        raise UnsupportedError(f"tallymap: reverse mode through the float64 Records field {n}.{f}")
                    if dt == C.F32:
                        tspecs.append(TSpec(rkey(n, f), (s.capacity,), dt))
                    continue
                if rmode != "count":
                    tspecs.append(TSpec(rkey(n, f), (s.capacity,), dt))
            if rmode is None:
                tspecs.append(TSpec(rkey(n, KI), (s.capacity,), C.I32))
                tspecs.append(TSpec(rkey(n, KK), (s.capacity,), C.I32))
            recs.append((n, s.capacity, fields))
            continue
        shape = (s.shape,) if isinstance(s.shape, int) else tuple(s.shape)
        dt = np.dtype(s.dtype)
        if dt not in SUM_DTYPES:
            raise UnsupportedError(f"tallymap: Sum output {n!r} of dtype {dt}: supported are "
                                   f"{', '.join(d.name for d in SUM_DTYPES)}")
        exact = bool(s.fixed_point) and dt == C.F32
        fixed = bool(s.fixed_point) and not exact
        scale = float(s.scale) if fixed else 0.0
        if fixed and not (np.isfinite(scale) and scale > 0.0):
            raise ValueError(f"tallymap: Sum output {n!r}: scale must be finite and positive, got {s.scale!r}")
        if int(np.prod(shape, dtype=np.int64)) > MAX_ITEMS:
            raise ValueError(f"tallymap: output {n!r} has more than 2^31 - 1 cells")
        tspecs.append(TSpec(n, shape, dt, exact, fixed=fixed, scale=scale,
                            kind="discard" if spawn_mode in ("fill", "count") else "sum"))
    if spawn is not None:
        tspecs.append(TSpec(QKEY, (1,), C.I32, kind="discard"))    # the spawn token (orders t.spawn like an emit)
        nf = sum(a.size for a in pav if a.dtype in (C.F32, C.F64))
        if spawn_mode == "adjoint" and nf:
            if int(spawn) * nf > MAX_ITEMS:
                raise UnsupportedError("tallymap: reverse mode through spawn needs Queue capacity x the float "
                                       "elements of a child below 2^31")
            tspecs.append(TSpec(QF, (int(spawn) * nf,), C.F32))     # the child slots of the tree adjoint
    names = [s.name for s in tspecs]
    where = item_name(fn)
    tav = [C.AVal((s.S,), s.dtype) for s in tspecs]
    shapes = {s.name: s.shape for s in tspecs}
    meta = {}
    b = C.Builder()
    C._STACK.append(b)
    capctx = L._CapCtx(b, max_steps) if max_steps is not None else None
    if capctx is not None:
        L._CAP.append(capctx)
    try:
        tin = [C.Tracer(b.new_invar(a)) for a in tav]
        pin = [C.Tracer(b.new_invar(a)) for a in pav]
        off = C.Tracer(b.new_invar(C.AVal((), C.I32))) if spawn_mode == "adjoint" and spawn is not None else None
        # (the Records adjoint program: each item's canonical offset per Records output, one operand each)
        roff = [C.Tracer(b.new_invar(C.AVal((), C.I32))) for _ in recs] if rmode in ("adjoint", "fill") else []
        bin_ = [C.Tracer(b.new_invar(a)) for a in bav]
        rec0 = {}
        if roff:
            rec0 = {r: (0, o) for (r, _, _), o in zip(recs, roff)}
        elif recs:
            cid = C.bind("tallymap_item_index", [], [C.AVal((), C.I32)])[0]
            rec0 = {r: (0, cid) for r, _, _ in recs}
        if spawn_mode == "record" and spawn is not None:
            rec0[QKEY] = (0, C.bind("tallymap_item_index", [], [C.AVal((), C.I32)])[0])
        elif spawn_mode == "adjoint" and spawn is not None:
            rec0[QKEY] = (0, off)
        rinfo = tuple(recs) + (((QKEY, ctree, tuple(pav), spawn_mode),) if spawn is not None else ())
        rinfo += ((RADJ, rmode, None),) if rmode is not None and recs else ()
        t = Tally({n: x for n, x in zip(names, tin)}, shapes, rec0, rinfo or None)
        m = unflatten(ptree, pin) if ptree is not None else pin
        bb = unflatten(btree, bin_) if btree is not None else bin_
        mi, bi = iter(m), iter(bb)
        uargs = [next(mi) if x == 0 else next(bi) for x in axes]
        r = fn(t, *uargs)
        if isinstance(r, Tally):
            t2, y = r, None
        elif isinstance(r, tuple) and len(r) == 2 and isinstance(r[0], Tally):
            t2, y = r
        else:
            raise TypeError("tallymap: the item function must return its Tally or (Tally, per_item_result)")
        yl, meta["ytree"] = flatten(y)
        outs = []
        for n in names:
            outs.append(b.local(t2._vals[n].var))
        for v in yl:
            if not C.is_traced(v):
                v = C.Tracer(C.bind("copy", [C.literal(v)], [C.literal(v).aval.strong()])[0].var)
            outs.append(b.local(v.var))
        counts = []
        for r, _, _ in (recs if not roff else ()):      # the per-item record counts (hidden per-item results)
            k = t2._r[r][0]
            if not C.is_traced(k):
                k = C.Tracer(C.bind("copy", [C.Lit(int(k), C.AVal((), C.I32))], [C.AVal((), C.I32)])[0].var)
            elif k.dtype != C.I32:
                k = C.convert(k, C.I32)
            counts.append(len(outs) - len(names))
            outs.append(b.local(k.var))
        qcount = None
        if spawn_mode == "record":        # the item's spawn count (hidden per-item result: its children)
            k = t2._r[QKEY][0]
            if not C.is_traced(k):
                k = C.Tracer(C.bind("copy", [C.Lit(int(k), C.AVal((), C.I32))], [C.AVal((), C.I32)])[0].var)
            elif k.dtype != C.I32:
                k = C.convert(k, C.I32)
            qcount = len(outs) - len(names)
            outs.append(b.local(k.var))
        trunc = None
        if capctx is not None:
            tr = capctx.trunc
            if tr is None:
                tr = C.Tracer(C.bind("copy", [C.Lit(False, C.AVal((), C.BOOL))], [C.AVal((), C.BOOL)])[0].var)
            outs.append(b.local(tr.var))
            trunc = len(outs) - len(names) - 1
    finally:
        C._STACK.pop()
        if capctx is not None:
            L._CAP.pop()
    jx = C.Jaxpr(b.invars, outs, b.eqns)
    if b.captured:
        raise C.TraceError("tallymap: the item function closes over a traced value of another call")
    check_tallies(jx, len(tspecs), where)
    prog = ItemProgram(jx, tuple(tspecs), len(pav) + (off is not None) + len(roff), len(bav), trunc,
                       "primal" if spawn_mode is None else f"spawn_{spawn_mode}", where,
                       tuple(recs) if rmode is None else (), tuple(counts),
                       int(spawn) if spawn is not None and spawn_mode not in ("adjoint", "fill") else None,
                       spawn_mode, qcount)
    return prog, meta


def _records_spawn(prepare, opts, names, args):
    """Records outputs of a spawning call (reference _api.py:817-890), in two passes.  The recording forward runs
    the tree (the Sums, the stats, each item's record counts, every generation in canonical order); record k of
    node m sits at offset[m] + k, the nodes numbered roots first, then generation by generation (a parent's
    children consecutive, by ordinal: the reference's _tree_order), offset the exclusive prefix sum of the nodes'
    counts.  The fill pass runs the known generations again with every append EMITTED at its slot into zeroed
    tallies of the capacity (0 + v = v).  A Records output past its capacity, a dropped child or a truncated item
    or child makes every float output NaN and every integer record field -1."""
    import torch

    from . import backend as B
    prog, meta, pi, bc, N, _ = prepare(args, "record")
    fprog = prepare(args, "fill")[0]
    o = B.run(prog, pi, bc, N, opts)
    res_out = _sum_outputs(prog, o, names)
    stats = {n: o.stats[ST[n]] for n in ("fixed_point_overflow", "dropped_emits")}
    stats.update((n, o.stats[ST[n]]) for n in ("spawned", "children_dropped", "children_truncated"))
    ys, trunc = _split_ys(prog, list(o.ys))
    trunc, stats["n_truncated"] = _truncation(trunc, o, N)
    recs = list(prepare(args)[0].records)      # (name, capacity, fields) of each Records output
    bad, over, offs = _tree_records(o, recs, prog, stats)
    rt = {}
    if offs is not None:
        gens = [(list(ops) + [offs[j][g] for j in range(len(recs))], n)
                for g, (ops, _, n) in enumerate(o.generations)]
        fo = B.run_generations(fprog, gens, bc, opts)
        rt = {fprog.tallies[k].name: t for k, t in zip(fprog.out_tallies, fo.tallies)}
    _tree_records_out(res_out, rt, recs, bad, over, [""])
    return Result(res_out, unflatten(meta["ytree"], ys), trunc, stats)


def _tree_records(o, recs, prog, stats):
    """the Records bookkeeping of a spawning call from its recording forward `o`: each output's exact count
    (stats appended / records_dropped / records_mismatch), whether any output is past its capacity (`over`) or the
    call is poisoned (`bad`: that, a dropped child, a truncated item or child), and per output and generation the
    nodes' canonical offsets (None when the tree is incomplete or an output overflowed)."""
    import torch

    from . import backend as B
    allc = [torch.cat([gc[j] for gc in o.gen_counts]) for j in range(len(recs))]
    scans = [B.util.exclusive_scan(c) for c in allc]
    appended = [x[-1] + c[-1] if len(c) else torch.zeros((), dtype=torch.int64, device="cuda")
                for x, c in zip(scans, allc)]
    over = any(bool((a > cap).item()) for a, (_, cap, _) in zip(appended, recs))
    bad = over or bool((o.stats[ST["children_dropped"]] != 0).item()) or (
        prog.trunc is not None and bool(((o.stats[ST["children_truncated"]] != 0)
                                         | (stats["n_truncated"] != 0)).item()))
    stats["appended"], stats["records_dropped"], stats["records_mismatch"] = {}, {}, {}
    for (r, cap, _), a in zip(recs, appended):
        stats["appended"][r], stats["records_dropped"][r] = a, (a - cap).clamp(min=0)
        stats["records_mismatch"][r] = 0
    if o.generations is None or over:
        return bad, over, None
    sizes = [n for _, _, n in o.generations]
    return bad, over, [x.clamp(max=cap).to(torch.int32).split(sizes) for x, (_, cap, _) in zip(scans, recs)]


def _tree_records_out(res_out, rt, recs, bad, over, sfx):
    """res_out[r] = {field: the fill tally rkey(r, field) + suffix}, for each suffix in sfx ('' the primal, "'" or
    "'l" a tangent lane: float fields only), zeros where the fill did not run; poisoned when `bad` (floats NaN,
    integers -1); an output past its capacity poisons every float Sum too."""
    import torch

    from . import backend as B
    from ._tally import rkey
    outs = [res_out] if len(sfx) == 1 and sfx[0] == "" else res_out
    for d, x in zip(outs, sfx):
        for r, cap, fields in recs:
            d[r] = {}
            for f, dt in fields:
                if x and dt not in (C.F32, C.F64):
                    continue
                t = rt.get(rkey(r, f) + x)
                if t is None:
                    t = torch.zeros((cap,), dtype=B.torch_dtype(dt), device="cuda")
                if bad:
                    t = t.fill_(float("nan")) if dt in (C.F32, C.F64) else t.fill_(-1)
                d[r][f] = t
        if over:                               # (a Records output past its capacity poisons every float Sum too)
            for n in list(d):
                v = d[n]
                if not isinstance(v, dict) and v.dtype in (torch.float32, torch.float64):
                    v.fill_(float("nan"))


def _result(prog, meta, o, names, N):
    """the Result of a forward launch's Outputs."""
    res_out = _sum_outputs(prog, o, names)
    stats = {n: o.stats[ST[n]] for n in ("fixed_point_overflow", "dropped_emits")}
    if prog.spawn is not None:
        stats.update((n, o.stats[ST[n]]) for n in ("spawned", "children_dropped", "children_truncated"))
    ys, trunc = _split_ys(prog, list(o.ys))
    trunc, stats["n_truncated"] = _truncation(trunc, o, N)
    _record_outputs(prog, o, res_out, stats)
    return Result(res_out, unflatten(meta["ytree"], ys), trunc, stats)


def _split_ys(prog, ys):
    """the backend's per-item results -> (the item's own results, the truncation flag or None): the hidden
    per-item record counts are removed."""
    hidden = set(prog.counts) | ({prog.trunc} if prog.trunc is not None else set())
    hidden |= {prog.qcount} if getattr(prog, "qcount", None) is not None else set()
    own = [y for j, y in enumerate(ys) if j not in hidden]
    return own, (ys[prog.trunc] if prog.trunc is not None else None)


def _sum_outputs(prog, o, names):
    """{name: the summed output} of the user's outputs among a launch's tallies (in prog.out_tallies order)."""
    tn = [s.name for s in prog.tallies]
    at = {slot: i for i, slot in enumerate(prog.out_tallies)}
    return {n: o.tallies[at[tn.index(n)]].reshape(prog.tallies[tn.index(n)].shape) for n in names if n in tn}


def _truncation(trunc, o, N):
    """Result.truncated and stats['n_truncated']: without max_steps no item is truncated (bool[N] zeros, an int32
    zero), as in the reference (_api.py:689-693)."""
    if trunc is not None:
        return trunc, o.n_truncated
    import torch
    z = torch.zeros(((N + 3) // 4,), dtype=torch.int32, device="cuda").view(torch.bool)[:N]     # (a word per store)
    # (without a cap the launch counts no truncated children either: its zero, of a buffer of 20 bytes and not of z,
    # which a kept count would keep)
    return z, o.stats[ST["children_truncated"]]


def _record_outputs(prog, o, res_out, stats):
    """Records outputs ({field: canonical array}) and their stats from a launch's Outputs."""
    if not prog.records:
        return
    stats["appended"], stats["records_dropped"], stats["records_mismatch"] = {}, {}, {}
    for j, (r, cap, fields) in enumerate(prog.records):
        res_out[r] = {f: o.records[r][f] for f, _ in fields}
        n = o.rcount[j]
        stats["appended"][r] = n
        stats["records_dropped"][r] = (n - cap).clamp(min=0)
        stats["records_mismatch"][r] = 0          # (one pass: no replay whose counts could disagree)


def vmap(fn=None, *, outputs, in_axes=0, max_steps=None, spawn=None, backend="auto", **opts):
    """Map `fn(tally, *args) -> tally | (tally, y)` over the leading axis of the mapped args (reference
    _api.py:428-700).

    outputs:   {name: Sum(shape, dtype=float32, fixed_point=False)}
    in_axes:   0 (mapped) or None (broadcast) per positional argument
    max_steps: cap on every top-level while loop; an item that hits it is flagged in Result.truncated and makes
               every float tally of the call NaN
    spawn:     tallymap_amd.Queue(capacity) to allow t.spawn(child) (forward calls; run generation by generation)
    The returned function also takes n_active=n: only items i < n run (a fixed capacity N with a varying active
    count, reference _api.py:469-472); the others emit nothing, are never truncated and get zero per-item results.
    backend:   'auto' / 'hip' (the HIP kernel backend; it never falls back)
    opts:      schedule 'step' (default: a lane refills at loop-step granularity) | 'item'; block (threads per
               block, default 256); refill (idle lanes a wave waits for before it claims, default 1); compact
               (iterations between the tail-phase repacks of a workgroup's live items, default 16; 0: off);
               post_batch (the deferred item end: a lane whose item ended waits this many times the ski-rental
               break-even for the wave's other ending lanes, default 2.0; 0: off); rev_schedule (reverse mode:
               'tape', the default, a count launch that tapes the step states in HBM and a reverse launch over
               the tape, both step-refilled; 'step', one step-refilled replay kernel over a tape; 'item', one item
               per lane with in-lane checkpoints); rev_tape (states a lane's tape holds, default sized to a 16 GiB
               tape budget, at least 16 per item; an item longer than the tape re-runs its steps past the tape
               from a checkpoint, (K - cap)^2 / 2 extra steps in its lane; a tape larger than the device's free
               memory is refused); rev_residual (the tape adjoint's tape: None, the
               default, tapes what the step's VJP reads when that is no wider than the step's state, True / False
               force the residual / state tape); rev_record (vjp's forward call is the tape adjoint's count launch,
               default True; False: the plain forward, and the whole adjoint at pullback time); rev_refill (free
               lanes a wave waits for before the step-scheduled replay hands it items, default 32; 64 suits items
               of equal length); rev_checkpoints (the 'item' schedule's C states per checkpoint buffer); lds_tables
               (bytes of broadcast tables of at most 16 KiB each -- a reverse launch's cotangent tally, a lookup
               table -- copied into LDS at each workgroup's start and read there; default 0: none); grad_mode
               (how vjp, grad and value_and_grad differentiate w.r.t. broadcast arguments: 'auto', the default,
               runs one forward launch with a tangent lane per differentiated element when every differentiated
               argument is broadcast, they hold at most 8 float32 elements and a loop carry needs the reverse
               sweep (or, with exact sums, in a vjp of 2^19 items or more where that launch costs less than the
               forward and the adjoint), else the replay adjoint; 'reverse' always the replay adjoint; 'tangent' lanes whenever the
               arguments are broadcast); blocks_per_cu (at most this many workgroups per CU in the item loop's
               persistent grid; default: the occupancy, and 2 for a spawning call, whose shower ran 13 % faster
               at 2 than at 8); min_blocks_per_sm (workgroups per CU the compiler must leave registers for:
               the launch bounds' minimum); cuda_math is accepted for drop-in compatibility and has no meaning on
               ROCm.
    """
    if fn is None:
        return lambda f: vmap(f, outputs=outputs, in_axes=in_axes, max_steps=max_steps, spawn=spawn, backend=backend,
                              **opts)
    if spawn is not None and not isinstance(spawn, Queue):
        raise TypeError("tallymap: spawn must be tallymap_amd.Queue(capacity)")
    bad = sorted(set(opts) - set(OPTS))
    if bad:
        raise ValueError(f"tallymap: unknown option(s) {bad}; options are " + ", ".join(OPTS))
    if opts.get("schedule", "step") not in ("item", "step"):
        raise ValueError(f"tallymap: schedule must be 'item' or 'step', got {opts['schedule']!r}")
    if backend not in ("auto", "hip", "rocm"):
        raise ValueError(f"tallymap: unknown backend {backend!r}; this package is the ROCm (HIP) kernel backend")
    outs_spec = {k: (v if isinstance(v, (Sum, Records)) else Sum(v)) for k, v in outputs.items()}
    names = sorted(outs_spec)

    spec_key = tuple(sorted((n, repr(v)) for n, v in outs_spec.items()))     # (the program cache key's outputs)

    calls = {}          # (program kind, per argument: shape, dtype) -> prepare's answer for calls with array arguments

    def prepare(args, spawn_mode=None):
        """(program, meta, per-item operands, broadcast operands, N, axes) of a call."""
        # a repeated call with arrays alone (no pytrees, no Python scalars) differs from an earlier one in its data
        # only: shapes and types decide the program
        key = [spawn_mode]
        for a in args:
            sh, dt = getattr(a, "shape", None), getattr(a, "dtype", None)
            # (a shape of another type may not be hashable; a container of leaves may have fields of these names)
            if not isinstance(sh, tuple) or dt is None or isinstance(a, (tuple, list, dict)):
                key = None
                break
            key.append(sh)
            key.append(dt)
        if key is not None:
            key = tuple(key)
            hit = calls.get(key)
            if hit is not None:
                prog, meta, mapped_at, bcast_at, N, axes = hit
                return prog, meta, [args[i] for i in mapped_at], [args[i] for i in bcast_at], N, axes
        prog, meta, pi, bc, N, axes = prepare_call(args, spawn_mode)
        if key is not None:
            if len(calls) >= PROG_CACHE:
                calls.clear()
            calls[key] = (prog, meta, [i for i, x in enumerate(axes) if x == 0],
                          [i for i, x in enumerate(axes) if x is None], N, axes)
        return prog, meta, pi, bc, N, axes

    def prepare_call(args, spawn_mode):
        axes = in_axes if isinstance(in_axes, (tuple, list)) else (in_axes,) * len(args)
        if len(axes) != len(args) or any(a not in (0, None) for a in axes):
            raise ValueError("tallymap: in_axes must be 0/None or a tuple of 0/None per positional argument")
        margs = tuple(a for a, x in zip(args, axes) if x == 0)
        bargs = tuple(a for a, x in zip(args, axes) if x is None)
        pi, ptree = flatten(margs)
        bc, btree = flatten(bargs)
        if not pi:
            raise ValueError("tallymap: at least one argument must be mapped (in_axes=0)")
        Ns = {_shape(x)[0] if len(_shape(x)) else -1 for x in pi}
        if len(Ns) != 1 or -1 in Ns:
            raise ValueError(f"tallymap: mapped arguments must share one leading axis length, got {sorted(Ns)}")
        N = Ns.pop()
        if N > MAX_ITEMS:
            raise ValueError(f"tallymap: N={N} items exceeds 2^31-1; split the call")
        pav = [C.AVal(_shape(x)[1:], _np_dtype(x)) for x in pi]
        bav = [C.AVal(_shape(x), _np_dtype(x)) for x in bc]
        key = (tuple(pav), tuple(bav), tuple(axes), repr(ptree), repr(btree), max_steps, spec_key, spawn, spawn_mode)
        hit = _PROGS.get((id(fn), key))
        if hit is not None and hit[0] is fn:
            _PROGS.move_to_end((id(fn), key))
            prog, meta = hit[1], hit[2]
        else:
            ctree = flatten(margs[0] if len(margs) == 1 else margs)[1] if spawn is not None else None
            prog, meta = build_program(fn, outs_spec, axes, pav, bav, max_steps, ptree, btree,
                                       spawn.capacity if spawn is not None else None, ctree, spawn_mode)
            _PROGS[(id(fn), key)] = (fn, prog, meta)
            while len(_PROGS) > PROG_CACHE:
                _PROGS.popitem(last=False)
        return prog, meta, pi, bc, N, axes

    def mapped(*args, n_active=None):
        from . import backend as B
        prog, meta, pi, bc, N, _ = prepare(args)
        if prog.records and prog.spawn is not None:
            if n_active is not None:
                raise ValueError("tallymap: n_active with spawn is not supported")
            return _records_spawn(prepare, opts, names, args)
        o = B.run(prog, pi, bc, N, opts, n_active=None if n_active is None else int(n_active))
        return _result(prog, meta, o, names, N)

    # Records outputs without a capacity: each call runs a count pass first and then the call sized by it
    dyn = [n for n in names if isinstance(outs_spec[n], Records) and outs_spec[n].capacity is None]
    sized_cache = {}

    def sized(args, n_active=None):
        """the mapped function with every Records capacity fixed for this call's arguments (itself when all are
        given): the capacity-less ones sized by a count pass to the next power of two >= their record count (over
        the first n_active items when given, as the call itself runs)."""
        if not dyn:
            return mapped
        if spawn is not None:
            raise ValueError("tallymap: Records outputs of a spawning call need a capacity")
        from . import backend as B
        prog, _, pi, bc, N, _ = prepare(args, "count")
        o = B.run(prog, pi, bc, N, opts, n_active=n_active)
        rnames = [n for n in names if isinstance(outs_spec[n], Records)]
        caps = {}
        for j, r in enumerate(rnames):
            if r in dyn:
                tot = int(o.ys[prog.counts[j]].long().sum().item())
                c = 1 << max(0, (tot - 1).bit_length())
                if c > MAX_ITEMS:
                    raise ValueError(f"tallymap: Records output {r!r} has no capacity and its call appended {tot} "
                                     "records: more than the largest capacity (2^30 as a power of two): split the call")
                caps[r] = c
        key = tuple(sorted(caps.items()))
        f = sized_cache.get(key)
        if f is None:
            spec = {n: (Records(outs_spec[n].fields, caps[n]) if n in caps else outs_spec[n]) for n in names}
            f = sized_cache[key] = vmap(fn, outputs=spec, in_axes=in_axes, max_steps=max_steps, spawn=spawn,
                                        backend=backend, **opts)
        return f

    def entry(*args, n_active=None):
        return (sized(args, n_active) if dyn else mapped)(*args, n_active=n_active)

    for g in (mapped, entry):
        g.__wrapped__ = fn
        g._prepare = prepare
        g._opts = opts
        g._names = names
        g._sized = sized if dyn else (lambda args, n_active=None: mapped)
    return entry


# ----------------------------------------------------------------------------------------- reverse mode
def _arg_leaves(prog, args, axes, argnums):
    """the operand leaves of the positional arguments in argnums -> ({pos: (in_axis, operand indices of its leaves,
    treedef, leaf shapes)}, wrt = (float32 per-item operand indices, float32 broadcast operand indices))."""
    pav, bav = prog.p_avals(), prog.b_avals()
    spec, wp, wb = {}, [], []
    p = b = 0
    for pos, x in enumerate(axes):
        leaves, td = flatten(args[pos])
        base = p if x == 0 else b
        idx = list(range(base, base + len(leaves)))
        if pos in argnums:
            spec[pos] = (x, idx, td, [_shape(v) for v in leaves])
            for i in idx:
                if (pav if x == 0 else bav)[i].dtype == C.F32:
                    (wp if x == 0 else wb).append(i)
        if x == 0:
            p += len(leaves)
        else:
            b += len(leaves)
    return spec, (tuple(wp), tuple(wb))


def _arg_cotangents(spec, wrt, g_pi, g_bc):
    """the cotangents of the arguments in spec, each with its argument's structure (None for a leaf that is not
    float32), in positional order; one argument alone is returned bare."""
    gp, gb = dict(zip(wrt[0], g_pi)), dict(zip(wrt[1], g_bc))
    out = []
    for pos in sorted(spec):
        x, idx, td, shapes = spec[pos]
        src = gp if x == 0 else gb
        leaves = [src.get(i) if x == 0 else (src[i].reshape(sh) if i in src else None) for i, sh in zip(idx, shapes)]
        out.append(unflatten(td, leaves) if td is not None else leaves[0])
    return tuple(out) if len(out) != 1 else out[0]


def _argnums(argnums, nargs):
    if argnums is None:
        return tuple(range(nargs))
    return (argnums,) if isinstance(argnums, int) else tuple(argnums)


def vjp(mapped, *args, argnums=None, n_active=None):
    """(Result, pullback): the forward call, and pullback(ct_outputs, ct_per_item=None) -> the cotangents of the
    positional arguments in `argnums` (float32 ones; broadcast arguments' cotangents are exact float32 sums).
    ct_outputs: {name: array or scalar (broadcast to the output)}.  The pullback launches the replay adjoint: the
    reference's jax.vjp through tallymap_call (_primitive.py:565-667, _reverse.py:1079-1180).  n_active=n runs the
    forward and the adjoint over the first n items only (the others' cotangents are zero), as the reference's
    n_active composes with jax.vjp (_api.py:469-472).
    Where the adjoint is the tape schedule's (a loop carry needs the reverse sweep), the forward call IS the
    adjoint's count launch: it writes the step states' tape beside the forward's outputs, and the pullback is the
    reverse launch alone (the tape stays allocated while the pullback lives; the option rev_record=False runs the
    plain forward and the whole adjoint at pullback time instead).
    Where the gradient runs as tangent lanes (option grad_mode; by default a few broadcast elements through a loop
    carry, or, in large calls, where one launch of them costs less than the forward and the adjoint), the forward call
    is the jvp launch with one lane per differentiated element and the pullback is a contraction of its tangent
    outputs with the cotangents, on the device, with no launch of its own (through a loop carry, plain float32 tallies'
    tangents accumulate in float64 atomics: reproducible to float64 reassociation; grad_mode='reverse' gives the replay
    adjoint's exact, bitwise reproducible broadcast cotangents.  Where the lanes replace a forward-only adjoint, their
    sums are exact and as reproducible as its)."""
    m = mapped._sized(args, n_active)
    prog, meta, pi, bc, N, axes = m._prepare(args)
    tg = _tangent_plan(m, prog, args, axes, argnums,
                       pair=(N if n_active is None else int(n_active)) >= LANES_PAIR_ITEMS)
    if tg is not None:
        return _tangent_vjp(m, args, tg, n_active)
    if prog.spawn is None and not prog.records:
        from . import backend as B
        spec, wrt = _arg_leaves(prog, args, axes, _argnums(argnums, len(args)))
        got = B.record(prog, wrt, pi, bc, N, m._opts, n_active=n_active)
        if got is not None:
            taped, fo = got

            def pullback(ct_outputs=None, ct_per_item=None):
                cys = {}
                if ct_per_item is not None:
                    for j, x in enumerate(flatten(ct_per_item)[0]):
                        if x is not None:
                            cys[j] = x
                g_pi, g_bc, _ = B.run_vjp(prog, wrt, pi, bc, N, _tally_cts(prog, ct_outputs), cys, m._opts,
                                          n_active=n_active, taped=taped)
                return _arg_cotangents(spec, wrt, g_pi, g_bc)
            return _result(prog, meta, fo, m._names, N), pullback
    res = mapped(*args, n_active=n_active)
    return res, _pullback(mapped, args, argnums, n_active)


def _pullback(mapped, args, argnums, n_active=None, prep=None):
    from . import backend as B
    if prep is not None:                   # (the caller's mapped._sized(...) and its _prepare(args))
        mapped, (prog, meta, pi, bc, N, axes) = prep
    else:
        mapped = mapped._sized(args, n_active)
        prog, meta, pi, bc, N, axes = mapped._prepare(args)
    if prog.spawn is not None:
        if n_active is not None:
            raise ValueError("tallymap: n_active with spawn is not supported")
        return _tree_pullback(mapped, args, argnums)
    an = _argnums(argnums, len(args))
    vprog, extra, bad = prog, [], False
    if prog.records:
        # reverse mode through Records (the reference's fill twin, _api.py:856-870): the forward gives each item's
        # record count, hence its canonical offset per output; the adjoint program emits every float field at its
        # record's slot, so the records' cotangents reach the appended values
        import torch
        vprog = mapped._prepare(args, "adjoint")[0]
        o = B.run(prog, pi, bc, N, mapped._opts, n_active=n_active)
        for j, (r, cap, _) in enumerate(prog.records):
            extra.append(B.util.exclusive_scan(o.ys[prog.counts[j]]).clamp(max=cap).to(torch.int32))
            bad = bad or bool((o.rcount[j] > cap).item())     # (an output past its capacity: NaN, as the forward)
    spec, wrt = _arg_leaves(vprog, args, axes, an)

    def pullback(ct_outputs=None, ct_per_item=None):
        cts = _tally_cts(vprog, ct_outputs)
        cys = {}
        if ct_per_item is not None:
            yl, _ = flatten(ct_per_item)
            for j, x in enumerate(yl):
                if x is not None:
                    cys[j] = x
        g_pi, g_bc, ntr = B.run_vjp(vprog, wrt, list(pi) + extra, bc, N, cts, cys, mapped._opts, n_active=n_active)
        if bad:
            g_pi = [x.float().fill_(float("nan")) for x in g_pi]
            g_bc = [x.float().fill_(float("nan")) for x in g_bc]
        return _arg_cotangents(spec, wrt, g_pi, g_bc)
    return pullback


def _tally_cts(prog, ct_outputs):
    """{tally slot: cotangent} of prog from {output name: cotangent} (a Records field: {name: {field: ...}})."""
    from ._tally import FIELD_SEP
    cts = {}
    for k, s in enumerate(prog.tallies):
        if not ct_outputs:
            break
        if s.name in ct_outputs:
            cts[k] = ct_outputs[s.name]
        elif FIELD_SEP in s.name:
            r, f = s.name.split(FIELD_SEP, 1)
            if isinstance(ct_outputs.get(r), dict) and f in ct_outputs[r]:
                cts[k] = ct_outputs[r][f]
    return cts


def _tree_pullback(mapped, args, argnums):
    """reverse mode through spawn: the tree adjoint (reference _reverse_spawn.py).  The recording forward runs the
    generations with each child's parent and ordinal and keeps them in canonical order (item i's children at
    off[i] + ordinal).  The adjoint program is the item with every spawn an EMIT of the child's float operands into
    a child-slot tally at (off + ordinal) x floats + element, so the cotangent of a child's initial state reaches
    its parent as the cotangent of that emitted value, at the spawn step, inside the ordinary replay adjoint.  One
    adjoint launch per generation, deepest first: generation g's child-slot cotangents are generation g + 1's
    per-item operand cotangents; broadcast cotangents are summed over the generations, the roots' per-item operand
    cotangents are the per-item arguments'.  A dropped child (incomplete tree) makes every cotangent NaN."""
    import torch

    from . import backend as B
    from ._tally import QF
    rprog, meta, pi, bc, N, axes = mapped._prepare(args, "record")
    aprog = mapped._prepare(args, "adjoint")[0]
    an = _argnums(argnums, len(args))
    spec, want = _arg_leaves(rprog, args, axes, an)
    pav = rprog.p_avals()
    fpi = tuple(j for j, a in enumerate(pav) if a.dtype in (C.F32, C.F64))
    if any(pav[j].dtype == C.F64 for j in fpi):
        raise UnsupportedError("tallymap: reverse mode through spawn with float64 per-item operands")
    wrt = (fpi, want[1])        # (every float per-item operand: the children's cotangents flow through them)
    o = B.run(rprog, pi, bc, N, mapped._opts)
    gens = o.generations
    Q = int(rprog.spawn)
    # Records outputs of the call: their appends emit at the canonical node order's offsets (per generation)
    recs = list(mapped._prepare(args)[0].records)
    roffs, over = [[] for _ in (gens or ())], False
    if recs and gens is not None:
        sizes = [n for _, _, n in gens]
        for j, (_, cap, _) in enumerate(recs):
            c = torch.cat([gc[j] for gc in o.gen_counts])
            x = B.util.exclusive_scan(c)
            over = over or (len(c) > 0 and bool((x[-1] + c[-1] > cap).item()))
            for g, xg in enumerate(x.clamp(max=cap).to(torch.int32).split(sizes)):
                roffs[g].append(xg)
    nf = sum(max(1, pav[j].size) for j in fpi)
    an_slots = {s.name: k for k, s in enumerate(aprog.tallies)}
    qf = an_slots.get(QF)

    def pullback(ct_outputs=None, ct_per_item=None):
        from ._tally import FIELD_SEP
        cts = {an_slots[n]: v for n, v in (ct_outputs or {}).items() if n in an_slots}
        for n, k in an_slots.items():             # a Records field: ct_outputs[name][field]
            if FIELD_SEP in n and not n.startswith(FIELD_SEP):
                r, f = n.split(FIELD_SEP, 1)
                if isinstance((ct_outputs or {}).get(r), dict) and f in ct_outputs[r]:
                    cts[k] = ct_outputs[r][f]
        cys = {}
        if ct_per_item is not None:
            yl, _ = flatten(ct_per_item)
            cys = {j: x for j, x in enumerate(yl) if x is not None}
        nan = gens is None or over
        z = torch.zeros((N,), dtype=torch.int32, device="cuda")
        runs = gens if gens is not None else [(list(pi), z, N)]
        ct_next, g_bc, g_root = None, None, None
        for g in reversed(range(len(runs))):
            ops, off, n = runs[g]
            ct = dict(cts)
            if qf is not None:
                ct[qf] = ct_next if ct_next is not None else 0.0
            ro = roffs[g] if gens is not None else [z] * len(recs)
            gp, gb, _ = B.run_vjp(aprog, wrt, list(ops) + [off] + ro, bc, n, ct, cys if g == 0 else {},
                                  mapped._opts)
            g_bc = gb if g_bc is None else [a + b for a, b in zip(g_bc, gb)]
            if g == 0:
                g_root = gp
            elif nf:
                flat = torch.cat([x.reshape(n, -1).float() for x in gp], 1).reshape(-1)
                ct_next = torch.zeros((Q * nf,), dtype=torch.float32, device="cuda")
                ct_next[:n * nf] = flat
        if nan:
            g_root = [torch.full_like(x, float("nan")) for x in g_root]
            g_bc = [torch.full_like(x, float("nan")) for x in g_bc]
        gr = dict(zip(fpi, g_root))
        return _arg_cotangents(spec, want, [gr[i] for i in want[0]], g_bc)
    return pullback


def grad(mapped, weights=None, argnums=None):
    """the gradient of sum_name <weights[name], outputs[name]> (weights: a scalar or an array per output; default
    1 for every float output, i.e. the gradient of the sum of all float tallies) w.r.t. the arguments in
    argnums.  ONE launch of the replay adjoint, no forward launch (as jax.grad of a tallymap call under jit).  The
    returned function takes n_active=n as the mapped call does."""
    def g(*args, n_active=None):
        w = weights if weights is not None else {n: 1.0 for n in mapped._names}
        m = mapped._sized(args, n_active)
        prep = m._prepare(args)
        tg = _tangent_plan(m, prep[0], args, prep[5], argnums)
        if tg is not None:
            return _tangent_vjp(m, args, tg, n_active)[1](w)
        return _pullback(mapped, args, argnums, n_active, prep=(m, prep))(w)
    return g


def value_and_grad(mapped, weights=None, argnums=None):
    """(Result, gradient) of the mapped call: the forward's outputs and the gradient grad(mapped, weights, argnums)
    gives, from the adjoint's launches alone where the adjoint replays the whole forward anyway (jax.value_and_grad
    of a tallymap call).  The forward-only adjoint (no loop carry needs a reverse sweep) returns both from ONE
    launch; the tape adjoint's count launch returns the forward's outputs beside the tape, so the pair takes two
    launches instead of a forward launch and two adjoint ones.  Records outputs, spawn and the checkpointed replay
    schedules run the forward and the adjoint separately.  The returned function takes n_active=n as the call does."""
    def g(*args, n_active=None):
        w = weights if weights is not None else {n: 1.0 for n in mapped._names}
        m = mapped._sized(args, n_active)
        prog, meta, pi, bc, N, axes = m._prepare(args)
        tg = _tangent_plan(m, prog, args, axes, argnums)
        if tg is not None:
            res, pull = _tangent_vjp(m, args, tg, n_active)
            return res, pull(w)
        if prog.records or prog.spawn is not None or m._opts.get("rev_schedule", "tape") != "tape":
            return m(*args, n_active=n_active), _pullback(m, args, argnums, n_active)(w)
        from . import backend as B
        spec, wrt = _arg_leaves(prog, args, axes, _argnums(argnums, len(args)))
        g_pi, g_bc, _, fo = B.run_vjp(prog, wrt, pi, bc, N, _tally_cts(prog, w), {}, m._opts, n_active=n_active,
                                      forward=True)
        return _result(prog, meta, fo, m._names, N), _arg_cotangents(spec, wrt, g_pi, g_bc)
    return g


# ------------------------------------------------------------------------------- gradients by tangent lanes
TANGENT_MAX = 8                # broadcast float32 elements up to which grad_mode='auto' differentiates by lanes
_UNITS = {}                    # (shape, dtype, element) -> the unit tangent on the device
_TPLAN = collections.OrderedDict()   # (program, argnums, axes, mode, argument trees) -> _tangent_plan's answer


def _tangent_plan(m, prog, args, axes, argnums, pair=False):
    """how the gradient w.r.t. argnums is computed (option grad_mode): None for the replay adjoint (reverse mode),
    else (spec, wrt, lanes, bav, wide) with lanes = [(broadcast operand, flat element)], one forward-mode tangent lane
    per float32 element of the broadcast arguments (bav: the program's broadcast operand avals; wide: jvp_program's).

    The gradient of a tally's <ct, T> w.r.t. a broadcast parameter theta of P elements is sum_k ct[k] dT[k]/dtheta:
    P directional derivatives, which one forward launch computes as P tangent lanes beside the primal (jvp), for
    any cotangent given afterwards.  The replay adjoint instead runs the count launch (the forward, taping the loop
    states) and the reverse launch (each step's VJP, newest first).  'auto' (the default) takes the lanes where
    they are cheaper: every differentiated argument is broadcast, P <= TANGENT_MAX, and a loop carry needs the
    reverse sweep (the tape adjoint; a forward-only adjoint is one launch already) or the call spawns (the tree
    adjoint is a recording forward, a canonical ordering and a count and a reverse launch per generation; the lanes
    are one forward through the generations, the children carrying their parents' tangents).  pair: the caller needs
    the forward's outputs before the cotangent (vjp), so a forward-only adjoint is a second launch after the
    forward's; the lanes are taken where one launch of them costs less (_lanes_beat_pair), with exact sums as the
    adjoint's, so that a gradient is reproducible at every size.  'reverse' always
    replays; 'tangent' takes the lanes whenever the arguments allow (any P, 16 lanes per launch).  Per-item
    arguments and Records outputs always replay."""
    mode = m._opts.get("grad_mode") or "auto"
    if mode not in ("auto", "reverse", "tangent"):
        raise ValueError(f"tallymap: grad_mode must be 'auto', 'reverse' or 'tangent', got {mode!r}")
    if mode == "reverse":
        return None
    an = _argnums(argnums, len(args))
    key = (prog.digest(), an, tuple(axes), mode, pair, tuple(repr(flatten(args[a])[1]) for a in an))
    hit = _TPLAN.get(key, _TPLAN)
    if hit is not _TPLAN:
        return hit
    plan = _TPLAN[key] = _tangent_plan_of(prog, args, axes, an, mode, pair)
    while len(_TPLAN) > PROG_CACHE:
        _TPLAN.popitem(last=False)
    return plan


LANES_PAIR = 0.85              # vjp takes lanes for a forward-only adjoint when a lane step costs at most this share of a
                               # forward step and an adjoint step together (kernel.cost, an exact emit at 30): the
                               # random walk problem's three lanes are 0.80 of them, and its loss gradient at 4,194,304
                               # items took 1,179 us by the two launches against 919 by one; the quickstart's lane is
                               # 0.58 (661 against 400), walk on spheres' five 0.55 (at 1,048,576: 514 against 358) ...
LANES_PAIR_BINS = 16           # ... and every tangent is emitted into at least this many bins: the lanes of a wave that
                               # add to one exact bin take turns (up-and-out calls, eight lanes onto one and eight bins,
                               # at 1,048,576: 3,903 by the two launches against 4,465) ...
LANES_PAIR_ITEMS = 1 << 19     # ... in calls of at least this many items: the contraction with the cotangent is ~60 us of
                               # small device operations against a launch that grows with the items' steps, which are
                               # not known (at 524,288 items: the walk of ~130 steps 4,234 us by two launches against
                               # 2,301, walk on spheres 391 against 262, random walk 320 against 286, but the quickstart
                               # of ~8 steps 130 against 181; at 1,048,576 that is 228 against 188)


def _lanes_beat_pair(prog, wrt, nlanes):
    """whether one launch of the program with its tangent lanes costs less than the forward launch and the forward-only
    adjoint's: by the static cost of a step of each (kernel.cost), and only where every tangent is an exact sum in LDS
    (the adjoint's sums are exact) and none is a per-item result's."""
    from . import backend as B
    from .backend import kernel as K
    from .backend import reverse as R
    from .backend import simplify
    if K._split(prog.jaxpr) is None:
        return False
    q = _jvp_prog(prog, (False,) * prog.nP, tuple(i in wrt[1] for i in range(prog.nB)), nlanes, "exact")
    if q.tangent_ys:           # (their tangents are N x lanes values that the adjoint does not store)
        return False
    L = K.build(q)[1]
    for k in L.emitted:
        t = q.tallies[k]       # (an exact sum rounded to float32 per bin would lose what bins of opposite signs cancel)
        if k >= prog.nT and not (t.exact and t.dtype == C.F64 and k in L.priv and t.S >= LANES_PAIR_BINS):
            return False
    adj, pl = B._adjoint(prog, wrt)

    def step(p):
        """(cost of a step, its emits)"""
        at = K._split(p.jaxpr)
        if at is None:
            return None
        eqns = simplify.cse(p.jaxpr.eqns[at].params["body_jaxpr"]).eqns
        return K.cost(eqns), sum(e.prim == "tallymap_emit" for e in C.walk_eqns(C.Jaxpr([], [], eqns)))
    costs = [step(p) for p in (q, prog, R.forward_only_program(adj, pl))]
    if None in costs:
        return False
    (lane, ne), (fwd, n0), (back, _) = costs
    return lane + 24 * (ne - n0) <= LANES_PAIR * (fwd + back)


def _tangent_plan_of(prog, args, axes, an, mode, pair):
    why = None
    if prog.records:
        why = "Records outputs are differentiated by the replay adjoint"
    spec, wrt = _arg_leaves(prog, args, axes, an)
    if why is None and any(axes[a] == 0 for a in an):
        why = "a per-item argument is differentiated by the replay adjoint"
    bav = prog.b_avals()
    lanes = [(i, e) for i in wrt[1] for e in range(max(1, bav[i].size))]
    if mode == "tangent":
        if why is not None:
            raise UnsupportedError(f"tallymap: grad_mode='tangent': {why}")
        return (spec, wrt, lanes, bav, True) if lanes else None
    if why is not None or not lanes or len(lanes) > TANGENT_MAX:
        return None
    from . import backend as B
    if prog.spawn is not None or B.needs_sweep(prog, wrt):
        return spec, wrt, lanes, bav, True
    return (spec, wrt, lanes, bav, "exact") if pair and _lanes_beat_pair(prog, wrt, len(lanes)) else None


def _unit(shape, dt, e):
    """the unit tangent of one element (flat index e) of a broadcast operand, kept on the device."""
    import torch

    from . import backend as B
    key = (tuple(shape), np.dtype(dt).str, e)
    t = _UNITS.get(key)
    if t is None:
        t = torch.zeros(int(np.prod(shape, dtype=np.int64)), dtype=B.torch_dtype(np.dtype(dt)), device="cuda")
        t[e] = 1
        t = _UNITS[key] = t.reshape(tuple(shape))
    return t


def _ct_f64(c, shape):
    """a cotangent (scalar, numpy array or tensor, broadcast to `shape`) as a float64 device tensor."""
    import torch
    if not isinstance(c, torch.Tensor):
        c = torch.from_numpy(np.ascontiguousarray(np.asarray(c, np.float64)))
    return torch.broadcast_to(c.to(device="cuda", dtype=torch.float64), tuple(shape))


def _tangent_vjp(m, args, plan, n_active):
    """(Result, pullback) of the gradient by tangent lanes (_tangent_plan): ONE launch of the jvp program with a
    unit tangent per differentiated element (16 per launch), then pullback(ct_outputs, ct_per_item) contracts:
    g[p] = sum over the float outputs of <ct, dT/dtheta_p> + sum over the float per-item results of
    <ct_y, dy/dtheta_p>, in float64 on the device, rounded to float32.  A plain float32 Sum's tangent tally
    accumulates in float64 here (an atomic sum whose reassociation from run to run stays ~1e-16 relative, against
    float32's ~n ulp over n emits into a bin: 1e-4 at millions of emits); an exact or fixed-point Sum's tangent is
    exact.  The replay adjoint sums the items' float32 contributions to a broadcast cotangent exactly; the two
    differ in the rounding of the items' float32 derivatives only.  A truncated item, or in a spawning call a
    dropped or truncated child, makes every cotangent NaN, as the replay and tree adjoints do."""
    import torch
    spec, wrt, lanes, bav, wide = plan
    primal, t_tal, t_ys = None, [], []
    for s in range(0, len(lanes), MAX_LANES):
        chunk = lanes[s:s + MAX_LANES]
        tans = [None] * len(args)
        for pos in spec:
            x, idx, td, shapes = spec[pos]
            if x == 0:
                continue
            per = []
            for i, e in chunk:
                leaves = [_unit(sh, bav[k].dtype, e) if k == i else None for k, sh in zip(idx, shapes)]
                per.append(unflatten(td, leaves) if td is not None else leaves[0])
            tans[pos] = per
        pr, tt, ty, _ = _run_tangents(m, args, tans, len(chunk), n_active, wide=wide)
        primal = pr if primal is None else primal
        t_tal += tt
        t_ys += ty
    ntr = primal.stats["n_truncated"]
    for k in ("children_dropped", "children_truncated"):     # (a spawning call: an incomplete or truncated tree)
        if k in primal.stats:
            ntr = ntr + primal.stats[k]

    def pullback(ct_outputs=None, ct_per_item=None):
        P = len(lanes)
        acc = torch.zeros((P,), dtype=torch.float64, device="cuda")
        for name, c in (ct_outputs or {}).items():
            ts = [t_tal[l].get(name) for l in range(P)]
            if ts[0] is None or isinstance(ts[0], dict):
                continue
            J = torch.stack(ts, 0).double()
            if not isinstance(c, torch.Tensor) and np.ndim(c) == 0:     # (a scalar: no copy to the device)
                acc += J.reshape(P, -1).sum(1) * float(c)
            else:
                acc += (J * _ct_f64(c, J.shape[1:])).reshape(P, -1).sum(1)
        if ct_per_item is not None:
            tys = [flatten(t_ys[l])[0] for l in range(P)]
            for j, c in enumerate(flatten(ct_per_item)[0]):
                if c is None or j >= len(tys[0]) or tys[0][j] is None:
                    continue
                J = torch.stack([tys[l][j] for l in range(P)], 0).double()
                acc += (J * _ct_f64(c, J.shape[1:])).reshape(P, -1).sum(1)
        g = torch.where(ntr != 0, torch.full_like(acc, float("nan")), acc).float()
        g_bc, k = [], 0
        for i in wrt[1]:
            sz = max(1, bav[i].size)
            g_bc.append(g[k:k + sz].reshape(tuple(bav[i].shape)))
            k += sz
        return _arg_cotangents(spec, wrt, [], g_bc)
    return primal, pullback


# ----------------------------------------------------------------------------------------- forward mode
MAX_LANES = 16                 # tangent directions per jacfwd kernel (reference: dual lanes <= 16 per kernel)
_JVP = collections.OrderedDict()


def _jvp_prog(prog, pp, pb, lanes, wide=False):
    from ._fwd import jvp_program
    key = (prog.digest(), pp, pb, lanes, wide)
    q = _JVP.get(key)
    if q is None:
        q = _JVP[key] = jvp_program(prog, pp, pb, lanes, wide)
        while len(_JVP) > PROG_CACHE:
            _JVP.popitem(last=False)
    return q


def _match_leaves(prim, tan):
    """the leaves of the tangent pytree `tan` aligned with the leaves of `prim` (a None subtree of tan stands for
    zeros: one None per leaf of prim's subtree)."""
    if tan is None:
        return [None] * len(flatten(prim)[0])
    if isinstance(prim, dict):
        return [v for k in sorted(prim) for v in _match_leaves(prim[k], tan.get(k))]
    if isinstance(prim, (list, tuple)):
        return [v for p, t in zip(prim, tan) for v in _match_leaves(p, t)]
    return [tan]


def _run_tangents(mapped, args, tans, lanes, n_active=None, wide=False):
    """one launch of the jvp program with `lanes` directions.  tans[pos]: None or a list of `lanes` tangent arrays
    for positional argument pos (its shape) -> (primal Result, per lane {name: tangent tally}, per lane [tangents
    of the float per-item results (None for the others)]).  wide: plain float32 tallies' tangents in float64 (True) or
    exact, rounded to float64 ('exact')."""
    from . import backend as B
    mapped = mapped._sized(args, n_active)
    prog, meta, pi, bc, N, axes = mapped._prepare(args)
    recs = list(prog.records)
    rs = bool(recs) and prog.spawn is not None
    if n_active is not None and prog.spawn is not None:
        raise ValueError("tallymap: n_active with spawn is not supported")
    if rs:      # Records of a spawning call: the recording forward's jvp, then the fill program's over the tree
        prog = mapped._prepare(args, "record")[0]
    pt, bt, pp, pb = [], [], [], []
    for pos, x in enumerate(axes):
        leaves, _ = flatten(args[pos])
        tl = tans[pos]
        for j, leaf in enumerate(leaves):
            dt = _np_dtype(leaf)
            isf = np.issubdtype(dt, np.floating)
            # (a spawning program carries a tangent of every float per-item operand: its children's tangents)
            on = isf and (tl is not None or (x == 0 and prog.spawn is not None))
            (pp if x == 0 else pb).append(on)
            if on and tl is None:
                import torch
                z = torch.zeros(_shape(leaf), dtype=B.torch_dtype(dt), device="cuda")
                pt += [z] * lanes
            elif on:
                for t in tl:
                    tv = _match_leaves(args[pos], t)[j]
                    if tv is None:                 # (a None subtree of the tangent: zero)
                        import torch
                        tv = torch.zeros(_shape(leaf), dtype=B.torch_dtype(dt), device="cuda")
                    (pt if x == 0 else bt).append(tv)
    q = _jvp_prog(prog, tuple(pp), tuple(pb), lanes, wide)
    o = B.run(q, list(pi) + pt, list(bc) + bt, N, mapped._opts, n_active=n_active)
    names = mapped._names
    nT = prog.nT
    res_out = _sum_outputs(prog, o, names)
    ny = len(prog.y_avals())
    ys, trunc = _split_ys(prog, list(o.ys[:ny]))
    stats = {n: o.stats[ST[n]] for n in ("fixed_point_overflow", "dropped_emits")}
    if prog.spawn is not None:
        stats.update((n, o.stats[ST[n]]) for n in ("spawned", "children_dropped", "children_truncated"))
    trunc, stats["n_truncated"] = _truncation(trunc, o, N)
    t_tal = [dict() for _ in range(lanes)]
    if rs:
        bad, over, offs = _tree_records(o, recs, prog, stats)
        rt = {}
        if offs is not None:
            fprog = mapped._prepare(args, "fill")[0]
            qf = _jvp_prog(fprog, tuple(pp) + (False,) * len(recs), tuple(pb), lanes)
            gens = [(list(ops[:prog.nP]) + [offs[j][g] for j in range(len(recs))] + list(ops[prog.nP:]), n)
                    for g, (ops, _, n) in enumerate(o.generations)]
            fo = B.run_generations(qf, gens, list(bc) + bt, mapped._opts)
            rt = {qf.tallies[k].name: t for k, t in zip(qf.out_tallies, fo.tallies)}
        _tree_records_out(res_out, rt, recs, bad, over, [""])
    else:
        _record_outputs(prog, o, res_out, stats)
    primal = Result(res_out, unflatten(meta["ytree"], ys), trunc, stats)
    at = {slot: i for i, slot in enumerate(q.out_tallies)}     # (the launch returns the "sum" tallies only)
    k = nT
    for slot in q.tangent_tallies:
        for l in range(lanes):
            if prog.tallies[slot].kind == "sum" and prog.tallies[slot].name in names:
                t_tal[l][prog.tallies[slot].name] = o.tallies[at[k]].reshape(prog.tallies[slot].shape)
            k += 1
    for r, cap, fields in (prog.records if not rs else ()):     # tangents of the float record fields (canonical)
        for l in range(lanes):
            t_tal[l][r] = {f: o.records[r][f + ("'" if lanes == 1 else f"'{l}")] for f, dt in fields
                           if dt in (C.F32, C.F64)}
    if rs:
        _tree_records_out(t_tal, rt, recs, bad, over, ["'"] if lanes == 1 else [f"'{l}" for l in range(lanes)])
    t_ys = [[None] * ny for _ in range(lanes)]
    m = ny
    for j in q.tangent_ys:
        for l in range(lanes):
            t_ys[l][j] = o.ys[m]
            m += 1
    return primal, t_tal, [unflatten(meta["ytree"], _split_ys(prog, t)[0]) for t in t_ys], meta


def jvp(mapped, primals, tangents, n_active=None):
    """(Result, tangent Result): the forward-mode derivative of the mapped call along `tangents` (jax.jvp of a
    tallymap call, reference _api.py:305-345, _primitive.py:419-436).  primals: the positional arguments;
    tangents: one per argument, None (not perturbed) or an array (pytree) of the argument's shape; only float
    leaves are perturbed.  The tangent Result holds the tangent of every float output and of every float per-item
    result (None for the others); ONE launch of the fused jvp kernel (primal and tangents in one pass).
    n_active=n runs the first n items only, as the mapped call does."""
    primals, tangents = tuple(primals), tuple(tangents)
    if len(tangents) != len(primals):
        raise ValueError("tallymap: jvp needs one tangent (or None) per primal argument")
    primal, t_tal, t_ys, _ = _run_tangents(mapped, primals, [None if t is None else [t] for t in tangents], 1,
                                           n_active)
    return primal, Result(t_tal[0], t_ys[0], None, None)


def _host_meta(x):
    """(shape, numpy dtype) of an argument, a numpy array or a (device) torch tensor alike, without a copy."""
    if type(x).__module__.startswith("torch"):
        return tuple(x.shape), np.dtype(str(x.dtype).replace("torch.", ""))
    x = np.asarray(x)
    return x.shape, x.dtype


def jacfwd(mapped, argnums=0, with_primal=False):
    """the forward-mode Jacobian of every float output w.r.t. the BROADCAST float arguments in argnums (jax.jacfwd
    of a tallymap call): -> f(*args) -> {name: {argnum: array of shape output.shape + arg.shape}}.  The unit
    tangents of the argument's elements run as dual lanes, up to 16 per fused kernel.  with_primal: f returns
    (jacobian, the call's Result) -- the primal the first launch computes beside its lanes (what jax.jacfwd of a
    loss of the outputs evaluates the loss's derivative at)."""
    an = (argnums,) if isinstance(argnums, int) else tuple(argnums)

    def jac(*args, n_active=None):
        m = mapped._sized(args, n_active)
        prog, meta, pi, bc, N, axes = m._prepare(args)
        dirs = []
        for a in an:
            if axes[a] == 0:
                raise UnsupportedError("tallymap: jacfwd is supported w.r.t. broadcast (in_axes=None) arguments; "
                                       "use jvp for a per-item argument")
            shp, dt = _host_meta(args[a])
            if not np.issubdtype(dt, np.floating):
                raise TypeError(f"tallymap: jacfwd w.r.t. argument {a} of dtype {dt}")
            size = int(np.prod(shp, dtype=np.int64))
            for i in range(size):
                e = np.zeros(size, dt)
                e[i] = 1
                dirs.append((a, e.reshape(shp)))
        cols = {n: [] for n in m._names}
        primal = None
        for s in range(0, len(dirs), MAX_LANES):
            chunk = dirs[s:s + MAX_LANES]
            tans = [None] * len(args)
            for a in an:
                shp, dt = _host_meta(args[a])
                lanes = [d if aa == a else np.zeros(shp, dt) for aa, d in chunk]
                tans[a] = lanes
            pr, t_tal, _, _ = _run_tangents(m, args, tans, len(chunk), n_active)
            primal = pr if primal is None else primal
            for l in range(len(chunk)):
                for n in m._names:
                    if n in t_tal[l]:
                        cols[n].append(t_tal[l][n])
        out = {}
        import torch
        for n, cs in cols.items():
            if not cs:
                continue
            full = torch.stack(cs, dim=-1)
            per, k = {}, 0
            for a in an:
                shp, _ = _host_meta(args[a])
                sz = int(np.prod(shp, dtype=np.int64))
                per[a] = full[..., k:k + sz].reshape(tuple(full.shape[:-1]) + tuple(shp))
                k += sz
            out[n] = per
        return (out, primal) if with_primal else out
    return jac
