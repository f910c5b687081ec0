"""The HIP kernel backend: run(prog, per-item operands, broadcast operands) on the current device and stream.

The plugin point of the reference is `KB.run(p, pi, bc, target, ...)` (reference backends/kernel/__init__.py:135-185),
called by `_primitive._run1` for the kernel platforms; this is its ROCm counterpart.  Operands are torch tensors on
the GPU (numpy arrays are copied there); results are allocated with torch and filled by the kernels, which
tm_launch queues on torch's current stream.  Device memory and streams come from torch; everything else is
this package's code.  There is no CPU path: without a GPU or without libtallymap_rocm.so it raises.
"""
import collections
import dataclasses
import threading

import numpy as np

from . import compile as Cm
from . import kernel as K
from . import util as U

_KERNELS = collections.OrderedDict()
_LOCK = threading.Lock()
KERNEL_CACHE = 256


@dataclasses.dataclass
class Compiled:
    id: int
    layout: object
    block: int
    src: str
    tag: str


@dataclasses.dataclass
class Outputs:
    tallies: list          # in prog.out_tallies order
    stats: object          # int32[5]
    ys: list               # per-item results (the truncation flag last when the program has a cap)
    n_truncated: object    # int32 scalar (None: no cap)
    records: dict = None   # Records name -> {field (or field' tangent): canonical array}
    rcount: list = None    # per Records output: records appended (int64 scalar tensor)


_TDT = {}
_GPU = []                   # [True] once a GPU was seen (the check runs until then)


def torch_dtype(dt):
    t = _TDT.get(dt)
    if t is None:
        import torch
        t = {"float32": torch.float32, "float64": torch.float64, "int32": torch.int32, "uint32": torch.uint32,
             "int64": torch.int64, "uint64": torch.uint64, "bool": torch.bool,
             "uint8": torch.uint8}[np.dtype(dt).name]
        _TDT[dt] = t
    return t


def device_tensor(x, dtype):
    """x as a contiguous tensor of `dtype` on the current GPU (a numpy array or scalar is copied there)."""
    import torch
    td = torch_dtype(dtype)
    if not _GPU:
        if not torch.cuda.is_available():
            raise Cm.BackendError("tallymap_amd: no GPU is visible (torch.cuda.is_available() is False); the HIP "
                                  "backend has no CPU fallback")
        _GPU.append(True)
    if isinstance(x, torch.Tensor):
        if x.is_cuda and x.dtype == td and x.is_contiguous():
            return x
        if x.device.type != "cuda":
            x = x.to("cuda")
        if x.dtype != td:
            raise TypeError(f"tallymap_amd: operand dtype {x.dtype} != traced {td}")
        return x.contiguous()
    a = np.array(x, dtype=dtype, order="C")          # (keeps a 0-d scalar 0-d)
    return torch.from_numpy(a).to("cuda")


def raw_stream():
    """torch's current stream on the current device, as a hipStream_t."""
    import torch
    return torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice())


def compiled(prog, opts, adjoint=None):
    """the registered kernel of prog under opts (in-memory LRU, then the disk cache, then hipRTC)."""
    block = int(opts.get("block", K.BLOCK))
    schedule = opts.get("schedule", "step")
    refill = int(opts.get("refill", 1))
    compact = int(opts.get("compact", K.COMPACT))
    mb = int(opts.get("min_blocks_per_sm", 0) or 0)
    pb = float(opts.get("post_batch", K.POST_BATCH))
    lt = int(opts.get("lds_tables", K.LDS_TABLES))
    cap = opts.get("blocks_per_cu")
    cap = int(cap) if cap else (K.SPAWN_BLOCKS if getattr(prog, "spawn", None) is not None else 0)
    key = (prog.digest(), block, schedule, refill, compact, mb, pb, lt, cap)
    with _LOCK:
        hit = _KERNELS.get(key)
        if hit is not None:
            _KERNELS.move_to_end(key)
            return hit
    src, L = K.build(prog, block=block, schedule=schedule, refill=refill, compact=compact, min_blocks=mb,
                     post_batch=pb, lds_tables=lt, grid_cap=cap)
    img = Cm.code_object(src, name=f"tm_{prog.tag}.hip")
    kid = int(Cm._key(src)[:15], 16)
    Cm.check(Cm.lib().tm_register(kid, img, len(img), f"{prog.tag} {prog.where}".encode()))
    c = Compiled(kid, L, block, src, prog.tag)
    with _LOCK:
        _KERNELS[key] = c
        while len(_KERNELS) > KERNEL_CACHE:
            _KERNELS.popitem(last=False)
    return c


def launch(c, ins, N, stream=None, tape=None):
    """allocate c's results and queue its kernels -> the result tensors (in layout order).  tape: the tape
    adjoint's item-major tape buffer (a program with a tape result uses it instead of allocating)."""
    outs = _alloc(c, N, tape)
    _queue(c, ins, outs, N, c.layout.n_zero, c.layout.flags, stream)
    return outs


_SPECS = {}                 # (kernel id, N) -> the result tensors' (shape, torch dtype), None for the tape


def _alloc(c, N, tape=None):
    """c's result tensors for a launch over N items (uninitialised: tm_zero clears what must start at zero)."""
    import torch
    specs = _SPECS.get((c.id, N))
    if specs is None:
        specs = _alloc_specs(c, N)
        if len(_SPECS) > 4096:
            _SPECS.clear()
        _SPECS[(c.id, N)] = specs
    outs = []
    for sp in specs:
        if sp is None:
            if tape is None:
                raise ValueError("tallymap_amd: a tape program launched without its tape buffer")
            outs.append(tape)
        else:
            outs.append(torch.empty(sp[0], dtype=sp[1], device="cuda"))
    return outs


def _alloc_specs(c, N):
    L = c.layout
    outs = []
    for shape, dt, per_item in L.res:
        if per_item == ("itape",):
            outs.append(None)
            continue
        if per_item == "tape":          # (rev_schedule='step') per launched lane: the persistent grid at this N
            sh = (_lanes(c, N),) + tuple(shape)
        elif isinstance(per_item, tuple) and per_item[0] == "rraw":
            # a Records raw buffer: the capacity and room for a partly used batch per launched wave
            S = per_item[1]
            sh = (S * K.raw_segment_slots(int(shape[0]), _lanes(c, N) // 64, S) if N > 0 else int(shape[0]),)
            if sh[0] > 2 ** 31 - 1:
                raise ValueError(f"tallymap_amd: a Records capacity of {shape[0]} leaves no room for the launch's "
                                 "batch slack below 2^31 slots")
        else:
            sh = ((N,) + tuple(shape)) if per_item else tuple(shape)
        outs.append((sh, torch_dtype(dt)))
    return outs


def _queue(c, ins, outs, N, n_zero, flags, stream=None, n_main=None):
    """queue c's kernels over N items on `stream` (default: torch's current one): tm_zero when n_zero, tm_main
    when N > 0 (over the first n_main items when given: n_active), tm_post when flags & 2, then the auxiliary
    passes of the layout (over all N)."""
    import ctypes

    import torch
    L = c.layout
    bufs = [t.data_ptr() for t in ins] + [t.data_ptr() for t in outs]
    arr = (ctypes.c_void_p * len(bufs))(*bufs)
    s = stream if stream is not None else raw_stream()
    Cm.check(Cm.lib().tm_launch(c.id, ctypes.c_void_p(s), arr, len(bufs), n_zero, flags,
                                N if n_main is None else n_main, c.block))
    if n_main == 0:
        N = 0          # (tm_main did not run: no item has a record, so the passes see no items)
    for name, kind, block, cap in (getattr(L, "aux", None) or []):
        if N == 0 and kind != "cap":         # (no item ran: only the canonical outputs are written, as zeros)
            continue
        grid = {"items": -(-int(N) // 1024), "one": 1, "cap": min(-(-int(cap) // 256), 4096)}[kind]
        Cm.check(Cm.lib().tm_launch_aux(c.id, name.encode(), ctypes.c_void_p(s), arr, len(bufs), N, grid, block))


def launch_noalloc(c, ins, N, stream=None):
    """c over N items through tm_launch_noalloc: the outputs are allocated here (torch), the scratch buffers of the
    layout (exact / fixed-point words, ctl) live in the library's per-device array -> the result tensors in layout
    order, with None at the scratch slots.  A program with Records or spawn (their passes and generations run
    through tm_launch_aux and the host) is refused."""
    import ctypes

    import torch
    L = c.layout
    if getattr(L, "aux", None) or getattr(L, "r_q", None) or not L.n_claim:
        raise ValueError("tallymap_amd: launch_noalloc runs plain forward programs (no Records, no spawn)")
    scr = set(L.scratch)
    outs, slots, nbytes = [], [], []
    for j, (shape, dt, per_item) in enumerate(L.res):
        r = L.n_in + j
        sh = ((N,) + tuple(shape)) if per_item else tuple(shape)
        if r in scr:
            outs.append(None)
            slots.append(r)
            nbytes.append(int(np.prod(sh, dtype=np.int64)) * np.dtype(dt).itemsize)
        else:
            outs.append(torch.empty(sh, dtype=torch_dtype(dt), device="cuda"))
    bufs = [t.data_ptr() for t in ins] + [0 if t is None else t.data_ptr() for t in outs]
    arr = (ctypes.c_void_p * len(bufs))(*bufs)
    sl = (ctypes.c_int * max(1, len(slots)))(*slots)
    nb = (ctypes.c_longlong * max(1, len(nbytes)))(*nbytes)
    s = stream if stream is not None else raw_stream()
    Cm.check(Cm.lib().tm_launch_noalloc(c.id, ctypes.c_void_p(s), arr, len(bufs), sl, nb, len(slots), L.n_zero,
                                        L.flags, N, c.block))
    return outs


def run(prog, pi, bc, N, opts, n_active=None):
    """the kernel backend's run(): outputs of prog over N items (only the first n_active of them run when given:
    the others emit nothing, count as nothing and get zero per-item results)."""
    c = compiled(prog, opts)
    ins = [device_tensor(x, a.dtype) for x, a in zip(pi, prog.p_avals())]
    ins += [device_tensor(x, a.dtype) for x, a in zip(bc, prog.b_avals())]
    for x, a in zip(ins[:prog.nP], prog.p_avals()):
        if tuple(x.shape) != (N,) + tuple(a.shape):
            raise ValueError(f"tallymap_amd: per-item operand of shape {tuple(x.shape)}, expected {(N,) + a.shape}")
    for x, a in zip(ins[prog.nP:], prog.b_avals()):
        if tuple(x.shape) != tuple(a.shape):
            raise ValueError(f"tallymap_amd: broadcast operand of shape {tuple(x.shape)}, expected {a.shape}")
    if getattr(prog, "spawn", None) is not None:
        if n_active is not None:
            raise ValueError("tallymap: n_active with spawn is not supported")
        return _run_spawn(c, prog, ins, N)
    if n_active is None:
        res = launch(c, ins, N)
    else:
        n = int(n_active)
        if not 0 <= n <= N:
            raise ValueError(f"tallymap: n_active={n} outside [0, N={N}]")
        res = _alloc(c, N)
        for r in c.layout.r_ys:                    # (the skipped items' per-item results: zero)
            res[r - c.layout.n_in][n:].zero_()
        _queue(c, ins, res, N, c.layout.n_zero, c.layout.flags, n_main=n)
    L = c.layout
    base = L.n_in
    tallies = [res[L.r_out[k] - base] for k in prog.out_tallies]
    stats = res[L.r_stats - base]
    ys = [res[r - base] for r in L.r_ys]
    ntr = res[L.r_ctl - base][2:3].view(__import__("torch").int32)[0] if prog.trunc is not None else None
    recs, rcount = {}, []
    for ri in getattr(L, "records", None) or []:
        recs[ri["name"]] = {f: res[rr - base] for f, rr in ri["fields"].items()}
        b, w = ri["r_ctr"]
        rcount.append(res[b - base].view(__import__("torch").int64)[w])
    return Outputs(tallies, stats, ys, ntr, recs, rcount)


def _run_spawn(c, prog, ins, N):
    """a spawning program, generation by generation (the reference's one-launch ticket ring, backends/kernel/
    kernel.py:1006-1040, made a host loop of ordinary launches: no wave ever waits for another).  Generation 0 runs
    the N items with tm_zero; each launch's children (their per-item operands in the Q-row buffers of the layout,
    the ticket counter in ctl words 32-33) are the next launch's items, without tm_zero, so the tallies and stats
    accumulate; tickets past Q are dropped children.  The loop ends at the first generation that spawns nothing
    (one device-to-host read of ctl per generation); the host then writes stats spawned / children_dropped /
    children_truncated and tm_post runs once (a dropped or truncated child poisons the float tallies there).

    The tree adjoint's recording forward (prog.spawn_mode 'record': children also store their parent and ordinal)
    puts every generation in canonical order -- the children of item i at off[i] .. off[i] + count[i] - 1, off the
    exclusive prefix sum of the items' spawn counts -- and keeps it: Outputs.generations = [(per-item operands,
    off int32[n], n)] from the roots down, or None when a child was dropped (the tree is incomplete), and
    Outputs.gen_counts = per generation, the items' Records counts (prog.counts; kept also after a drop)."""
    import torch
    L = c.layout
    base = L.n_in
    Q = int(prog.spawn)
    nP = prog.nP
    rec = getattr(prog, "spawn_mode", None) == "record"
    if not rec:
        return _run_spawn_device(c, prog, ins, N)
    outs = _alloc(c, N)
    ctl = outs[L.r_ctl - base].view(torch.int32)
    cur = [outs[r - base] for r in L.r_q]          # the buffers the last launch's children were written to
    spare, ys_scr = None, None
    _queue(c, ins, outs, N, L.n_zero, 0)
    spawned = dropped = 0
    ntr_roots = None
    gens, ops, n_cur = [], list(ins[:nP]), N      # (the operands and size of the generation just launched)
    gcounts = []
    while True:
        w = ctl.cpu().numpy().view(np.uint32)
        if ntr_roots is None:
            ntr_roots = int(w[2])
        cnt = int(w[32]) | (int(w[33]) << 32)
        if rec and prog.counts:                        # (the launch's per-item results: outs, or the scratch)
            src = (lambda r: outs[r - base]) if not gcounts else (lambda r: ys_scr[r])
            gcounts.append([src(L.r_ys[j])[:n_cur].clone() for j in prog.counts])
        if rec and gens is not None:
            counts = (outs[L.r_ys[prog.qcount] - base] if not gens else ys_scr[L.r_ys[prog.qcount]])[:n_cur]
            off = U.exclusive_scan(counts)             # (each item's first child, in canonical order)
            gens.append((ops, off.to(torch.int32), n_cur))
        if cnt == 0:
            break
        n = min(cnt, Q)
        spawned += n
        dropped += cnt - n
        if cnt > Q:
            gens = None                                # a dropped child: no complete tree to differentiate
        if spare is None:
            spare = [torch.empty_like(t) for t in cur]
            ys_scr = {r: torch.empty((Q,) + tuple(outs[r - base].shape[1:]), dtype=outs[r - base].dtype,
                                     device="cuda") for r in L.r_ys}
        if rec and gens is not None:                   # the children in canonical (parent, ordinal) order
            ops = []
            for t in cur[:nP]:
                z = torch.empty((n,) + tuple(t.shape[1:]), dtype=t.dtype, device="cuda")
                U.tree_scatter(off, cur[nP], cur[nP + 1], t, z, n)
                ops.append(z)
        else:
            ops = cur[:nP]
        ctl[K.SHARD0:L.n_claim].zero_()                # the item claim counters
        ctl[32:34].zero_()                             # the ticket counter
        gen = list(outs)
        for r, t in zip(L.r_q, spare):
            gen[r - base] = t
        for r, t in ys_scr.items():                    # (a child's own per-item result is discarded)
            gen[r - base] = t
        _queue(c, list(ops) + list(ins[nP:]), gen, n, 0, 0)
        n_cur = n
        cur, spare = spare, cur
    big = 2 ** 31 - 1
    ctr = int(w[2]) - ntr_roots
    outs[L.r_stats - base][0:3].copy_(torch.tensor([min(spawned, big), min(dropped, big), ctr], dtype=torch.int32))
    _queue(c, ins, outs, 0, 0, L.flags)
    tallies = [outs[L.r_out[k] - base] for k in prog.out_tallies]
    ys = [outs[r - base] for r in L.r_ys]
    ntr = torch.tensor(ntr_roots, dtype=torch.int32, device="cuda") if prog.trunc is not None else None
    o = Outputs(tallies, outs[L.r_stats - base], ys, ntr, {}, [])
    o.generations = gens if rec else None
    o.gen_counts = gcounts if rec else None
    return o


def _aux(c, name, bufs, n_items, grid=1, block=64, stream=None):
    import ctypes

    import torch
    arr = (ctypes.c_void_p * len(bufs))(*[t.data_ptr() for t in bufs])
    s = stream if stream is not None else raw_stream()
    Cm.check(Cm.lib().tm_launch_aux(c.id, name.encode(), ctypes.c_void_p(s), arr, len(bufs), n_items, grid, block))


def _run_spawn_device(c, prog, ins, N):
    """a spawning forward (or jvp) program whose generations are sized on the device: after each launch tm_qnext
    turns the ticket count into the next generation's item count (and the spawned / dropped / truncated stats), and
    the next launch (flags bit 4) reads it.  The counters are cleared and the stats written on the device: the host
    only reads one 8-byte count per generation, to stop, and it queues a generation before it waits for the count of
    the one before, so the device does not wait for the host; the one queued past the last finds no items and its
    workgroups return at once.  (The shower gradient at 262,144 roots, 7 generations: 0.83 ms with the host's read
    between a generation and the next, of which the kernels took 0.4.)  The children of one launch are the next
    one's per-item operands, in two buffers that alternate."""
    import torch
    L = c.layout
    base = L.n_in
    Q = int(prog.spawn)
    nP = prog.nP
    outs = _alloc(c, N)
    ctl = outs[L.r_ctl - base].view(torch.int32)
    cur = [outs[r - base] for r in L.r_q]
    spare = [torch.empty_like(t) for t in cur]
    ys_scr = {r: torch.empty((Q,) + tuple(outs[r - base].shape[1:]), dtype=outs[r - base].dtype, device="cuda")
              for r in L.r_ys}
    _queue(c, ins, outs, N, L.n_zero, 0)
    _aux(c, "tm_qnext", list(ins) + list(outs), 1)
    def generation():
        """queue the next generation and the read of its successor's item count -> (the pinned count, its event)."""
        nonlocal cur, spare
        gen = list(outs)
        for r, t in zip(L.r_q, spare):
            gen[r - base] = t
        for r, t in ys_scr.items():                    # (a child's own per-item result is discarded)
            gen[r - base] = t
        _queue(c, list(cur[:nP]) + list(ins[nP:]), gen, Q, 0, 4)
        _aux(c, "tm_qnext", list(cur[:nP]) + list(ins[nP:]) + gen, 0)
        cur, spare = spare, cur
        n = torch.empty(1, dtype=torch.int64, pin_memory=True)
        n.copy_(ctl[40:42].view(torch.int64), non_blocking=True)
        e = torch.cuda.Event()
        e.record()
        return n, e
    ahead = generation() if N > 0 else None
    while ahead is not None:
        (n, e), ahead = ahead, generation()
        e.synchronize()
        if int(n) == 0:
            break
    _queue(c, ins, outs, 0, 0, L.flags)
    tallies = [outs[L.r_out[k] - base] for k in prog.out_tallies]
    ys = [outs[r - base] for r in L.r_ys]
    ntr = ctl[48] if prog.trunc is not None else None
    o = Outputs(tallies, outs[L.r_stats - base], ys, ntr, {}, [])
    o.generations = None
    o.gen_counts = None
    return o


def run_generations(prog, gens, bc, opts):
    """an ordinary (not spawning) program over known generations -- gens = [(per-item operands, n)] -- as one
    accumulating launch sequence: tm_zero before the first, tm_post after the last (the fill pass of Records with
    spawn).  -> Outputs (per-item results of the first generation)."""
    import torch
    c = compiled(prog, opts)
    L = c.layout
    base = L.n_in
    if getattr(L, "aux", None):
        raise Cm.BackendError("internal: run_generations of a program with auxiliary passes")
    b_ins = [device_tensor(x, a.dtype) for x, a in zip(bc, prog.b_avals())]
    nmax = max(n for _, n in gens)
    outs = _alloc(c, nmax)
    for g, (ops, n) in enumerate(gens):
        ins = [device_tensor(x, a.dtype) for x, a in zip(ops, prog.p_avals())]
        if g:
            outs[L.r_ctl - base].view(torch.int32)[K.SHARD0:L.n_claim].zero_()     # (the item claim counters, per launch)
        _queue(c, ins + b_ins, outs, n, L.n_zero if g == 0 else 0, 0)
    _queue(c, [device_tensor(x, a.dtype) for x, a in zip(gens[0][0], prog.p_avals())] + b_ins, outs, 0, 0, L.flags)
    tallies = [outs[L.r_out[k] - base] for k in prog.out_tallies]
    ys = [outs[r - base][:gens[0][1]] for r in L.r_ys]
    ntr = outs[L.r_ctl - base][2:3].view(torch.int32)[0] if prog.trunc is not None else None
    return Outputs(tallies, outs[L.r_stats - base], ys, ntr, {}, [])


_LANES = {}


def _lanes(c, N):
    """the lanes tm_launch starts for c at N items: min(ceil(N / block), CUs x blocks per CU) x block.  A program with
    steps computed ahead may start more (tm_spread): nothing of it is sized by its lanes."""
    if c.layout.spread:
        raise Cm.BackendError("internal: buffers sized by the lanes of a launch that spreads")
    r = _LANES.get(c.id)
    if r is None:
        r = _LANES[c.id] = kernel_info(c)["resident_threads"]
    return min(-(-int(N) // c.block) * c.block, r)


def kernel_info(c):
    """tm_kernel_info of a compiled program: registers, private bytes, LDS bytes, blocks per CU, resident threads,
    CUs, max threads per block, persistent grid."""
    import ctypes
    out = (ctypes.c_longlong * 8)()
    Cm.check(Cm.lib().tm_kernel_info(c.id, c.block, out))
    keys = ("regs", "private_bytes", "lds_bytes", "blocks_per_cu", "resident_threads", "cus", "max_threads", "grid")
    return dict(zip(keys, [int(v) for v in out]))


def prebuild(entries, n=64):
    """compile (through hipRTC, no GPU needed) the forward and adjoint modules of each (name, config) in
    `entries` (config = dict(item, outputs, in_axes, max_steps); a config whose outputs are sized by N appears once
    per N) into the package's code-object cache -> [(name, tag, key)].  The operand shapes come from the config's
    input generator at `n` items (per-item shapes do not depend on N): configs.<name>_inputs, or the config's own
    `inputs` (returning (args, extra)); a config with `argnum` is differentiated w.r.t. that broadcast argument
    alone, others w.r.t. every differentiable argument and every broadcast one."""
    from .. import _api
    from .. import _core as C
    from .._api import build_program
    from .. import configs as CF
    done = []
    for name, cfg in entries:
        if cfg.get("queue"):
            continue                 # (a spawning call's programs are compiled when first run)
        args = cfg["inputs"](n)[0] if "inputs" in cfg else getattr(CF, f"{name}_inputs")(n)
        axes = cfg["in_axes"]
        pav = [C.AVal(np.shape(a)[1:], np.asarray(a).dtype) for a, x in zip(args, axes) if x == 0]
        bav = [C.AVal(np.shape(a), np.asarray(a).dtype) for a, x in zip(args, axes) if x is None]
        prog, _ = build_program(cfg["item"], cfg["outputs"], axes, pav, bav, cfg.get("max_steps"))
        src, _ = K.build(prog, block=K.BLOCK, schedule="step", refill=1)
        Cm.code_object(src, name=f"tm_{prog.tag}.hip", store_pkg=True)
        done.append((name, prog.tag, Cm._key(src)[:16]))
        from . import reverse as R
        if "argnum" in cfg:
            wrts = ([((), (sum(1 for x in axes[:cfg["argnum"]] if x is None),))] if cfg["argnum"] is not None
                    else [])
        else:
            wp, wb = R.default_wrt(prog)
            wrts = [(wp, wb), ((), wb)]
        for wrt in wrts:
            adj = R.adjoint_program(prog, wrt)
            pl = R.plan(adj)
            if any(pl.sweep):            # the tape adjoint: its count and reverse programs (and the count program
                from . import tape as T  # that keeps the forward's outputs: vjp's and value_and_grad's forward)
                tp = T.programs(adj, pl)
                progs = [tp.count, tp.reverse, T.programs(adj, pl, keep=True).count]
                lanes = sum(max(1, bav[i].size) for i in wrt[1])
                if not wrt[0] and 0 < lanes <= _api.TANGENT_MAX:
                    # grad_mode='auto' differentiates a few broadcast elements by tangent lanes: the jvp program
                    progs.append(_api._jvp_prog(prog, (False,) * len(pav),
                                                tuple(i in wrt[1] for i in range(len(bav))), lanes, wide=True))
            else:
                progs = [R.forward_only_program(adj, pl), R.forward_only_program(adj, pl, keep=True)]
            for q in progs:
                src, _ = K.build(q, block=K.BLOCK, schedule="step", refill=1)
                Cm.code_object(src, name=f"tm_{q.tag}.hip", store_pkg=True)
                done.append((name, q.tag + str(wrt), Cm._key(src)[:16]))
    return done


def compiled_adjoint(adj, opts):
    """the registered adjoint kernel of `adj` (a reverse.Adjoint) under opts."""
    from . import reverse as R
    from . import replay as RP
    block = int(opts.get("block", K.BLOCK))
    ck = int(opts.get("rev_checkpoints", R.C_DEFAULT) or R.C_DEFAULT)
    sched = opts.get("rev_schedule", "step")
    tape = int(opts.get("rev_tape", RP.TAPE) or RP.TAPE)
    rrefill = int(opts.get("rev_refill", RP.REFILL))
    if sched not in ("step", "item"):
        raise ValueError(f"tallymap_amd: rev_schedule must be 'tape', 'step' or 'item', got {sched!r}")
    key = (adj.digest(), block, "adjoint", sched, ck if sched == "item" else (tape, rrefill))
    with _LOCK:
        hit = _KERNELS.get(key)
        if hit is not None:
            _KERNELS.move_to_end(key)
            return hit
    if sched == "step":
        src, L = RP.build(adj, block=block, tape=tape, refill=rrefill)
    else:
        src, L = R.build(adj, block=block, ckpt=ck)
    img = Cm.code_object(src, name=f"tm_{adj.tag}.hip")
    kid = int(Cm._key(src)[:15], 16)
    Cm.check(Cm.lib().tm_register(kid, img, len(img), f"{adj.tag} {adj.where}".encode()))
    c = Compiled(kid, L, block, src, adj.tag)
    with _LOCK:
        _KERNELS[key] = c
        while len(_KERNELS) > KERNEL_CACHE:
            _KERNELS.popitem(last=False)
    return c


def _forward_outputs(prog, c, res, ys):
    """the forward's Outputs read from a value_and_grad launch of c (whose tally slots < prog.nT are the forward's,
    ys its per-item results)."""
    import torch
    L = c.layout
    base = L.n_in
    tallies = [res[L.r_out[k] - base] for k in prog.out_tallies]
    ntr = res[L.r_ctl - base][2:3].view(torch.int32)[0] if prog.trunc is not None else None
    return Outputs(tallies, res[L.r_stats - base], list(ys), ntr, {}, [])


def needs_sweep(prog, wrt):
    """True when the adjoint of prog w.r.t. wrt needs the reverse sweep of its loop (a carry's cotangent flows
    backward through the steps: the tape adjoint), False when the forward-only adjoint applies."""
    return any(_adjoint(prog, wrt)[1].sweep)


def _adjoint(prog, wrt):
    """(reverse.Adjoint, reverse.Plan) of prog w.r.t. wrt, cached."""
    from . import reverse as R
    if getattr(prog, "records", ()):
        raise Cm.BackendError("tallymap_amd: reverse mode through a program with Records outputs is not supported by "
                              "this backend yet (forward mode, jvp / jacfwd, is)")
    key = (prog.digest(), tuple(tuple(w) for w in wrt))
    hit = _ADJ.get(key)
    if hit is None:
        adj = R.adjoint_program(prog, wrt)
        hit = _ADJ[key] = (adj, R.plan(adj))
    return hit


def _tape_programs(adj, pl, opts, keep):
    from . import tape as T
    rres = opts.get("rev_residual")
    tkey = adj.digest() + ("|vg" if keep else "") + f"|{rres}"
    tp = _TAPE.get(tkey)
    if tp is None:
        tp = _TAPE[tkey] = T.programs(adj, pl, keep=keep, residual=rres)
    return tp


def _active(N_all, n_active):
    if n_active is None:
        return N_all
    N = int(n_active)
    if not 0 <= N <= N_all:
        raise ValueError(f"tallymap: n_active={N} outside [0, N={N_all}]")
    return N


def _pad_items(xs, N, N_all):
    """per-item results over the first N items -> over N_all (zeros after)."""
    import torch
    if N == N_all:
        return xs
    full = []
    for g in xs:
        z = torch.zeros((N_all,) + tuple(g.shape[1:]), dtype=g.dtype, device=g.device)
        z[:N] = g
        full.append(z)
    return full


@dataclasses.dataclass
class Taped:
    """the tape adjoint's forward half, kept for its reverse launch: the count launch's tape and per-item results
    ([K, the final stored state] + the truncation flag) over the first N of N_all items."""
    tp: object
    tape: object
    cap: object
    hand: list
    N: int
    N_all: int
    key: tuple


def _tape_count(prog, adj, pl, pi_t, bc_t, N, N_all, opts, keep):
    """the count launch over the first N items -> (Taped, the forward's Outputs when keep, else None)."""
    import torch

    from . import tape as T
    tp = _tape_programs(adj, pl, opts, keep)
    cap = T.tape_cap(N, tp.Wp, opts.get("rev_tape"), tp.Wck, tp.block)
    need = 4 * max(1, N * (cap * tp.Wp + tp.Wck))
    free = torch.cuda.mem_get_info()[0]
    if need > free:
        # (cap has a floor of T.CAP_MIN slots, so at very large N the tape can exceed the nominal budget)
        raise Cm.BackendError(f"tallymap_amd: the reverse-mode tape needs {need / 2 ** 30:.1f} GiB ({N} items x "
                              f"{cap} slots of {4 * tp.Wp} bytes) but {free / 2 ** 30:.1f} GiB are free; call with "
                              "fewer items (n_active, or several calls), a smaller rev_tape, or "
                              "rev_schedule='item' (in-lane checkpoints, no tape)")
    ck = (torch.cuda.current_device(), cap)
    capt = _CAPS.get(ck)
    if capt is None:         # (a read-only operand, made once: a new one per call is a pageable copy that waits for
        capt = _CAPS[ck] = torch.tensor(cap, dtype=torch.int32, device="cuda")     # the stream to drain)
    tape = torch.empty((max(1, N * (cap * tp.Wp + tp.Wck)),), dtype=torch.uint32, device="cuda")
    # the loop with its states taped -> K, the final state (and with keep, the forward's own outputs)
    c1 = compiled(tp.count, opts)
    r1 = launch(c1, pi_t + bc_t + [capt], N, tape=tape)
    hand = [r1[r - c1.layout.n_in] for r in c1.layout.r_ys]
    nh = 1 + tp.n_fin
    fo = None
    if keep:
        fo = _forward_outputs(prog, c1, r1, hand[nh:])
        fo.ys = _pad_items(fo.ys, N, N_all)
        hand = hand[:nh] + ([hand[tp.count.trunc]] if prog.trunc is not None else [])
    return Taped(tp, tape, capt, hand, N, N_all, (adj.digest(), N)), fo


def record(prog, wrt, pi, bc, N, opts, n_active=None):
    """vjp's forward as the tape adjoint's count launch: -> (Taped, the forward's Outputs), or None where the
    adjoint is not the tape schedule's (the forward-only adjoint, another rev_schedule, Records outputs): the
    caller then runs the plain forward and the whole adjoint at pullback time.  run_vjp(..., taped=) then launches
    the reverse program alone.  The tape stays allocated while the Taped object lives."""
    if getattr(prog, "records", ()) or getattr(prog, "spawn", None) is not None:
        return None
    if opts.get("rev_schedule", "tape") != "tape" or not opts.get("rev_record", True):
        return None
    adj, pl = _adjoint(prog, wrt)
    if not any(pl.sweep):
        return None
    N_all = N
    N = _active(N_all, n_active)
    pi_t = [device_tensor(x, a.dtype)[:N] for x, a in zip(pi, prog.p_avals())]
    bc_t = [device_tensor(x, a.dtype) for x, a in zip(bc, prog.b_avals())]
    return _tape_count(prog, adj, pl, pi_t, bc_t, N, N_all, opts, True)


def run_vjp(prog, wrt, pi, bc, N, ct_tallies, ct_ys, opts, n_active=None, forward=False, taped=None):
    """the replay adjoint of prog: cotangents of the per-item operands wrt[0] ([N, ...] each) and the broadcast
    operands wrt[1] (exact float32 sums), given the cotangents of the float tallies (ct_tallies[slot], missing ->
    0) and of the float per-item results (ct_ys[j], missing -> 0).  -> (g_pi list, g_bc list, n_truncated).
    When no loop carry needs a reverse sweep (an accumulator carry, c' = c + d, does not: reverse.Plan.accum) the
    adjoint is an ordinary item program (reverse.forward_only_program) run by the forward template (step refill);
    otherwise the adjoint opts['rev_schedule'] names: 'tape' (the default, backend/tape.py: the count and reverse
    launches of the forward template), 'step' (replay.build: one kernel, step refill over a tape) or 'item'
    (reverse.build: in-lane checkpoints).  With n_active
    only the first n_active items run (the adjoint launches over them alone); the others get zero cotangents and
    add nothing to the broadcast ones, as they emitted nothing in the forward.
    forward: value_and_grad -- the launches that replay the forward (the forward-only adjoint; the tape adjoint's
    count program) also return the forward's outputs, so no separate forward launch is needed: -> (g_pi, g_bc,
    n_truncated, Outputs of the forward).
    taped: a record() of the same program, operands and n_active -- the count launch already ran (as the forward
    call), only the reverse launch runs."""
    import torch

    adj, pl = _adjoint(prog, wrt)
    yav = prog.y_avals()
    wide = [prog.tallies[k].name for k in (ct_tallies or {}) if prog.tallies[k].dtype == np.float64]
    wide += [f"per-item result {j}" for j in (ct_ys or {}) if yav[j].dtype == np.float64]
    if wide:
        raise Cm.BackendError(f"tallymap_amd: reverse mode through float64 outputs ({', '.join(wide)}) is not "
                              "supported by this backend (float32 outputs and per-item results only)")
    N_all = N
    N = _active(N_all, n_active)
    pi_t = [device_tensor(x, a.dtype)[:N] for x, a in zip(pi, prog.p_avals())]
    cy_t = []
    for j in pl.fy:
        x = ct_ys.get(j) if ct_ys else None
        cy_t.append(device_tensor(x, yav[j].dtype)[:N] if x is not None
                    else torch.zeros((N,) + tuple(yav[j].shape), dtype=torch.float32, device="cuda"))
    bc_t = [device_tensor(x, a.dtype) for x, a in zip(bc, prog.b_avals())]
    ct_t = []
    for k in pl.ft:
        s = prog.tallies[k]
        x = ct_tallies.get(k) if ct_tallies else None
        if x is None:
            ct_t.append(torch.zeros((s.S,), dtype=torch.float32, device="cuda"))
        elif isinstance(x, (int, float, np.floating, np.integer)):
            ct_t.append(torch.full((s.S,), float(x), dtype=torch.float32, device="cuda"))
        else:
            ct_t.append(device_tensor(np.broadcast_to(np.asarray(x, np.float32), s.shape) if not hasattr(x, "device")
                                      else x, np.float32).reshape(-1))
    ins_p, ins_b = pi_t + cy_t, bc_t + ct_t
    fo = None
    if taped is not None and (taped.key != (adj.digest(), N) or taped.N_all != N_all):
        raise ValueError("tallymap_amd: a recorded tape of another program, operands or n_active")
    if not any(pl.sweep):
        fkey = adj.digest() + ("|vg" if forward else "")
        q = _FWD_ONLY.get(fkey)
        if q is None:
            from . import reverse as R
            q = _FWD_ONLY[fkey] = R.forward_only_program(adj, pl, keep=forward)
        c = compiled(q, opts)
        res = launch(c, ins_p + ins_b, N)
        L = c.layout
        base = L.n_in
        nT = prog.nT
        g_bc = [res[L.r_out[nT + jj] - base].reshape(prog.b_avals()[j].shape) for jj, j in enumerate(adj.wrt_bc)]
        ys = [res[r - base] for r in L.r_ys]
        g_pi = ys[:len(adj.wrt_pi)]
        if forward:
            fo = _forward_outputs(prog, c, res, _pad_items(ys[len(adj.wrt_pi):], N, N_all))
    elif opts.get("rev_schedule", "tape") == "tape":
        if taped is None:
            taped, fo = _tape_count(prog, adj, pl, pi_t, bc_t, N, N_all, opts, forward)
        tp = taped.tp
        # reverse: POST's VJP from the final state, the steps' VJPs newest first from the tape, PRE's VJP -> the
        # cotangents
        c = compiled(tp.reverse, opts)
        res = launch(c, ins_p + taped.hand + ins_b + [taped.cap], N, tape=taped.tape)
        L = c.layout
        base = L.n_in
        g_bc = [res[L.r_out[k] - base].reshape(prog.b_avals()[j].shape)
                for k, j in zip(tp.reverse.out_tallies, adj.wrt_bc)]
        g_pi = [res[r - base] for r in L.r_ys[:len(adj.wrt_pi)]]
    else:
        if forward:
            raise ValueError("tallymap_amd: value_and_grad in one pass runs the default (tape) replay schedule")
        c = compiled_adjoint(adj, opts)
        res = launch(c, ins_p + ins_b, N)
        L = c.layout
        base = L.n_in
        g_bc = [res[L.r_out[j] - base] for j in adj.wrt_bc]
        g_pi = [res[r - base] for r in L.r_ys[:len(adj.wrt_pi)]]
    ntr = res[L.r_ctl - base][2:3].view(torch.int32)[0] if prog.trunc is not None else None
    g_pi = _pad_items(g_pi, N, N_all)
    if forward:
        return g_pi, g_bc, ntr, fo
    return g_pi, g_bc, ntr


_FWD_ONLY = {}
_CAPS = {}                  # (device, tape slots per item) -> the int32 operand of the tape programs
_TAPE = {}                  # adjoint digest -> tape.TapePrograms
_ADJ = {}                   # (program digest, wrt) -> (reverse.Adjoint, reverse.Plan)
