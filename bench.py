"""Benchmark: items/s of the tallymap hot path (forward + replay gradient) on one MI355X.

Workload: BASELINE config 2, the 1-D random walk (C2) at N = 4,194,304 items, inputs resident in HBM.  One step is
the forward's outputs (occupancy and wall tallies, per-item trip counts, truncation flags) plus the gradient
d sum(tallies) / d drift (exact float32), through tm.value_and_grad on torch's current stream: C2's adjoint needs no
reverse sweep, and the forward-only adjoint replays the whole forward anyway, so one fused launch returns both;
`value` = N / (time per step).  The same quantities from two launches (the forward call, then tm.grad) are timed
beside it (fwd_ms, grad_ms, two_launch_items_per_s).

roofline: the dominant kernel's algorithmic HBM bytes per launch (per item: x0 4 B + key 8 B read, trip count 4 B +
truncation flag 1 B written = 17 B, for the fused launch as for the forward; the separate gradient launch: 12 B
read + 1 B written = 13 B) over its average launch duration (HIP events on the launch stream), against MI355X's
8 TB/s.  The path is VALU-bound (threefry, erf_inv in double), not HBM-bound: the fraction is reported as measured,
and valu_roofline puts the same launch against the VALU issue rates measured live on this GPU (backend/valu.py).  traffic: FETCH_SIZE + WRITE_SIZE per dispatch from
rocprofv3 counter runs of this bench, scaled by what the same counters read on a plain copy of known size
(--copy-probe); the recorded measurement at the default N unless --traffic-bytes gives another.
cpu_baseline: the oracle (the C/OpenMP restatement of the reference's CPU kernel backend) on the host's cores, on a
bounded sample of the same workload (the first items of the same inputs), forward + gradient, items/s.
configs: the other BASELINE configs at their own sizes (C1 10,000; C3, C4 4,194,304; C5 1,048,576), the forward call
and the gradient call timed the same way (the gradient by tangent lanes where grad_mode 'auto' takes them, C3 and C5,
with the replay adjoint's call beside it: grad_reverse_ms, and for C5 its count and reverse launches), each with the
oracle on a bounded sample beside it.
atomics / emit_roofline: the atomic adds/s of the patterns the kernels issue (backend/atomics.py; MI355X publishes no
atomic peak), and C2's forward emit rate against the peak of the LDS u64 adds its constant emits are counted with.
published: the reference's own benchmark problems (random walk, transport, walk on spheres, ODE ensemble;
tallymap_amd/problems.py) at the sizes of its published L40S kernel-backend timings, forward and loss gradient, the
published times beside them as cross-hardware context (the ratios are not like-for-like speedups).
"""
import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0
FWD_BYTES_PER_ITEM = 17
GRAD_BYTES_PER_ITEM = 13
# Counter-derived figures per launch at N = 4,194,304, each keyed by the machine code it was measured on (16 hex
# digits of sha256 over the code object's .text and .rodata: the instructions and kernel descriptors, whatever else
# of the source -- an unused device helper -- changed).  traffic: HBM bytes,
# FETCH_SIZE x 1.99992 + WRITE_SIZE x 1.000 (KiB), the factors those counters read on a plain 1 GiB device copy in the
# same runs (profiles/c2_random_walk_traffic.md); valu_insts: wave64 VALU instructions (SQ_INSTS_VALU) and
# valu_classes: the gfx950 SQ_INSTS_VALU_<class> counts of the same launch (profiles/c2_random_walk_sq_counters.md).
# A kernel whose machine code differs from the one measured reports null with the reason, so a changed kernel never
# carries a stale counter.
# (the SQ_INSTS_VALU_<class> counters bench.py reads, in the order the figures below list them)
VALU_CLASSES = ("INT32", "INT64", "ADD_F32", "MUL_F32", "FMA_F32", "TRANS_F32", "ADD_F64", "MUL_F64", "FMA_F64",
                "TRANS_F64", "CVT")


def _classes(*counts):
    return {"SQ_INSTS_VALU_" + c: float(n) for c, n in zip(VALU_CLASSES, counts)}


MEASURED = {"fused": {"code": "5e98387efe596d3b", "traffic": 82_543_940, "valu_insts": 6.1959e+09,
                       "valu_classes": _classes(1.835e+09, 4.835e+07, 1.404e+08, 8.638e+07, 0, 0,
                                                1.673e+08, 1.184e+08, 5.370e+08, 5.173e+06, 1.405e+08)},
            "forward": {"code": "1cdc3db81d2bc00d", "traffic": 83_894_085, "valu_insts": 6.1294e+09,
                        "valu_classes": _classes(1.836e+09, 4.838e+07, 1.404e+08, 8.639e+07, 0, 0,
                                                 1.674e+08, 1.185e+08, 5.371e+08, 5.173e+06, 1.405e+08)},
            "gradient": {"code": "47f260042cd43e9e", "traffic": 62_469_443, "valu_insts": 5.8878e+09,
                         "valu_classes": _classes(1.739e+09, 4.389e+07, 1.406e+08, 5.412e+07, 0, 0,
                                                  1.675e+08, 1.186e+08, 5.375e+08, 5.173e+06, 1.082e+08)}}


def code_keys(f, dev):
    """{fused, forward, gradient: the machine-code key (16 hex digits of sha256 over the code object's .text and
    .rodata: compile.machine_key) of the kernel that launch runs} for the mapped call f, its value_and_grad and its
    gradient w.r.t. argument 2 (each run once before, so all are compiled)."""
    from tallymap_amd import backend as B
    from tallymap_amd.backend import compile as Cm

    def mkey(q):
        return Cm.machine_key(Cm.code_object(B.compiled(q, f._opts).src))
    prog = f._prepare(dev)[0]
    keys = {"fused": None, "forward": mkey(prog), "gradient": None}
    for (dg, _), (adj, _) in list(B._ADJ.items()):
        if dg != prog.digest():
            continue
        for kind, suffix in (("gradient", ""), ("fused", "|vg")):
            q = B._FWD_ONLY.get(adj.digest() + suffix)
            tp = B._TAPE.get(adj.digest() + suffix + "|None")
            q = q if q is not None else (tp.reverse if tp is not None else None)
            if q is not None:
                keys[kind] = mkey(q)
    return keys


def vg_kernel(f, dev):
    """the compiled kernel of f's value_and_grad w.r.t. argument 2 (the forward-only adjoint keeping the forward)."""
    from tallymap_amd import backend as B
    prog = f._prepare(dev)[0]
    for (dg, _), (adj, _) in list(B._ADJ.items()):
        if dg == prog.digest() and B._FWD_ONLY.get(adj.digest() + "|vg") is not None:
            return B.compiled(B._FWD_ONLY[adj.digest() + "|vg"], f._opts)
    raise RuntimeError("bench: value_and_grad's kernel is not compiled")


def measured(kind, field, key, n):
    """(the recorded counter figure, None) when it was measured on this code object at this N, else (None, reason)."""
    m = MEASURED[kind]
    if n != 4_194_304:
        return None, f"measured at N = 4,194,304 only (this run: N = {n})"
    if m["code"] is None or m[field] is None:
        return None, "not measured"
    if m["code"] != key:
        return None, f"stale: measured on machine code {m['code']}, this run's {kind} kernel is {key}"
    return m[field], None


def valu_roofline(kind, key, n, ms):
    """the resource that binds C2's kernels: VALU issue (the HBM roofline is the contract's; the kernel reads 17 B
    and runs ~405 steps of ~210 VALU instructions per item).  peak: the fastest VALU issue rate measured live on this
    GPU (backend/valu.py: 32-bit integer and fp32 add / mul, xor), every pattern's rate beside it; achieved: the
    launch's SQ_INSTS_VALU over its duration.  issue_bound_ms: the shortest time the chip can issue that launch's
    instructions in, each SQ_INSTS_VALU_<class> count over the fastest measured rate of the instructions that class
    counts and the unclassed remainder (logic, rotations, selects, moves) at the fastest of its rates
    (valu.issue_bound); issue_bound_upper_ms prices every class at its slowest (INT32 at v_add3_u32's, the
    remainder at the slowest unclassed pattern's); issue_frac = issue_bound / time."""
    from tallymap_amd.backend import valu
    rates = valu.peaks()
    top = max(rates, key=rates.get)
    peak = rates[top]
    d = {"bound": "valu", "peak": peak, "unit": "wave64 VALU instructions/s",
         "peak_source": f"measured here: {top}, the fastest of the patterns, on every SIMD with 8 independent "
                        "chains per wave (backend/valu.py)",
         "rates": rates}
    vinsts, why = measured(kind, "valu_insts", key, n)
    if vinsts is None:
        d["null"] = why
        return d
    t = ms * 1e-3
    d.update(achieved=vinsts / t, frac=vinsts / t / peak, insts_per_launch=vinsts)
    classes, why = measured(kind, "valu_classes", key, n)
    if classes is None:
        d["issue_null"] = why
        return d
    lo, hi, parts = valu.issue_bound({"SQ_INSTS_VALU": vinsts, **classes}, rates)
    d.update(issue_bound_ms=lo * 1e3, issue_bound_upper_ms=hi * 1e3, issue_frac=lo / t, issue_frac_upper=hi / t,
             issue_parts_ms={c: [v[0] * 1e3, v[1] * 1e3] for c, v in parts.items()}, classes_per_launch=classes)
    return d


def host_info():
    """the host's CPU model and C library (the oracle calls its libm: glibc's bits are the CPU target's)."""
    import ctypes
    import platform
    model = platform.processor() or "unknown"
    try:
        with open("/proc/cpuinfo") as fh:
            for ln in fh:
                if ln.startswith("model name"):
                    model = ln.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    try:
        libc = ctypes.CDLL("libc.so.6")
        libc.gnu_get_libc_version.restype = ctypes.c_char_p
        glibc = libc.gnu_get_libc_version().decode()
    except (OSError, AttributeError):
        glibc = "-".join(platform.libc_ver())
    return model, glibc


def cpu_baseline(x0, keys, drift, max_steps, target_s=10.0):
    """the oracle on a bounded sample: forward + forward-mode gradient, items/s (and each of the two alone)."""
    import oracle as O
    O.build()
    threads = O.max_threads()
    n = 8192
    while True:
        t0 = time.perf_counter()
        O.c2_fwd(x0[:n], keys[:n], drift, max_steps=max_steps, shadow=False, per_item=True)
        t1 = time.perf_counter()
        O.c2_grad(x0[:n], keys[:n], drift, np.ones(128, np.float32), np.ones(2, np.float32), max_steps=max_steps)
        t2 = time.perf_counter()
        dt = t2 - t0
        if dt * 4 > target_s or n * 2 > x0.size:
            break
        n = min(x0.size, max(n * 2, int(n * target_s / max(dt, 1e-3) / 2)))
    model, glibc = host_info()
    return dict(value=n / dt, unit="items/s", cores=threads, kind="port",
                fwd_items_per_s=n / (t1 - t0), grad_items_per_s=n / (t2 - t1),
                sample=f"first {n} of the N=4,194,304 C2 items, forward + gradient (drift), {dt:.2f} s wall "
                       f"on {threads} OpenMP threads",
                cpu_model=model, glibc=glibc,
                build="oracle/Makefile: gcc -O3 -march=x86-64-v3 -ffp-contract=off -fopenmp, built in the build "
                      "container; the GPU box runs the same binary",
                gradient="forward-mode dual numbers in double (the oracle's c2_grad, ~0.9 of the forward's time): "
                         "not the reference CPU backend's checkpointed replay, whose forward-only activity analysis "
                         "keeps x active and runs a count and a replay pass, at least as much work")


def _cfg_runs(name, n, dev_inputs, mode="auto"):
    """(forward call, gradient call, mapped f) closures of config `name` on device inputs under grad_mode `mode`:
    the gradient of each config as BASELINE states it (C1 theta, C3 mu_a, C4 a: of the sum of the float tallies;
    C5 A: of the summed final energy, whose cotangent (sin theta, omega) comes from the forward's final states: a
    vjp and its pullback).  With the replay adjoint C5's gradient call is the count launch (the forward, taping the
    states) and the reverse launch; by tangent lanes (grad_mode 'auto' for a scalar A) it is one jvp launch and a
    contraction."""
    import torch

    import tallymap_amd as tm
    from tallymap_amd import configs
    cfg = configs.SIZED[name](n) if name in configs.SIZED else configs.CONFIGS[name]
    f = tm.vmap(cfg["item"], outputs=cfg["outputs"], in_axes=cfg["in_axes"], max_steps=cfg["max_steps"],
                **dict(cfg.get("opts", {}), grad_mode=mode))
    argn = {"c1": 2, "c3": 1, "c4": 3}
    if name in argn:
        g = tm.grad(f, argnums=argn[name])
        return (lambda: f(*dev_inputs)), (lambda: g(*dev_inputs)), f

    def grad(ev=None):
        res, pull = tm.vjp(f, *dev_inputs, argnums=3)
        st = res.outputs["state"]
        if ev is not None:
            ev.record(torch.cuda.current_stream())
        return pull({"state": torch.stack([torch.sin(st[:, 0]), st[:, 1]], 1)})
    return (lambda: f(*dev_inputs)), grad, f


def _timed(fn, steps, warmup):
    """mean ms of fn() over `steps` calls after `warmup`, HIP events on torch's current stream around each call."""
    import torch
    for _ in range(warmup):
        fn()
    torch.cuda.synchronize()
    stream = torch.cuda.current_stream()
    evs = [[torch.cuda.Event(enable_timing=True) for _ in range(2)] for _ in range(steps)]
    r = None
    for e in evs:
        e[0].record(stream)
        r = fn()
        e[1].record(stream)
    torch.cuda.synchronize()
    return float(np.mean([e[0].elapsed_time(e[1]) for e in evs])), r


def _cpu_sample(name, inputs, target_s):
    """the oracle's forward + gradient of config `name` on the first items of `inputs`, grown until the pair takes
    about target_s / 4 s -> (items/s, n, seconds)."""
    import oracle as O
    from tallymap_amd import configs
    O.build()
    n = 2048
    N = len(inputs[0])
    while True:
        sl = [x[:n] if np.ndim(x) else x for x in inputs]
        t0 = time.perf_counter()
        if name == "c1":
            O.c1_fwd(*sl, shadow=False)
            O.c1_grad(*sl, np.ones(16, np.float32))
        elif name == "c3":
            O.c3_fwd(*sl, shadow=False, per_item=False)
            O.c3_grad(*sl, np.ones((64, 64), np.float32))
        elif name == "c4":
            ids = np.arange(n, dtype=np.int32)
            O.c4_fwd(sl[0], sl[1], ids, sl[3], shadow=False, per_item=False)
            O.c4_grad(sl[0], sl[1], ids, sl[3], np.ones((256, 256), np.float32), np.ones((n, 1), np.float32))
        else:
            ids = np.arange(n, dtype=np.int32)
            r = O.c5_fwd(sl[0], sl[1], ids, sl[3], shadow=False, per_item=False)
            O.c5_grad(sl[0], sl[1], ids, sl[3], configs.c5_energy_ct(r.tallies["state"]))
        dt = time.perf_counter() - t0
        if dt * 4 > target_s or n >= N:
            return n / dt, n, dt
        n = min(N, max(n * 2, int(n * target_s / max(dt, 1e-3) / 4)))


def _records_walker(t, x, key, theta):
    """the quickstart walker writing a Records output: (bin, theta (1 - x)) per step instead of a histogram add."""
    from tallymap_amd import lax
    from tallymap_amd import numpy as jnp
    from tallymap_amd import random as R

    def body(c):
        k, x, t = c
        u = R.uniform(R.fold_in(key, k))
        b = (x * 16.0).astype(jnp.int32)
        t = t.append("steps", {"bin": b, "w": theta * (1.0 - x)}, when=b < 16)
        return k + 1, x * (0.5 + 0.5 * u), t
    k, x, t = lax.while_loop(lambda c: c[1] > 0.05, body, (0, x, t))
    return t, k


def bench_records(steps, warmup):
    """Records throughput: C1's walker over 4,194,304 items appending one record per step (about 33M records,
    capacity 2^26) -- the one-pass launch plus the canonicalisation passes, HIP events on torch's current stream."""
    import torch

    import tallymap_amd as tm
    from tallymap_amd import configs
    n = 4_194_304
    xs, keys, theta = configs.c1_inputs(n)
    dev = [torch.from_numpy(xs).cuda(), torch.from_numpy(keys).cuda(), torch.tensor(theta).cuda()]
    f = tm.vmap(_records_walker, outputs={"steps": tm.Records({"bin": np.int32, "w": np.float32}, capacity=1 << 26)},
                in_axes=(0, 0, None), max_steps=100)
    for _ in range(warmup):
        f(*dev)
    torch.cuda.synchronize()
    stream = torch.cuda.current_stream()
    evs = [[torch.cuda.Event(enable_timing=True) for _ in range(2)] for _ in range(steps)]
    for e in evs:
        e[0].record(stream)
        r = f(*dev)
        e[1].record(stream)
    torch.cuda.synchronize()
    ms = float(np.mean([e[0].elapsed_time(e[1]) for e in evs]))
    nrec = int(r.stats["appended"]["steps"].item())
    drop, ntr = int(r.stats["records_dropped"]["steps"].item()), int(r.stats["n_truncated"].item())
    if drop or ntr:
        raise RuntimeError(f"records bench: {nrec} records, {drop} dropped, {ntr} truncated items")
    print("bench: records done", file=sys.stderr, flush=True)
    return {"n_items": n, "records": nrec, "capacity": 1 << 26, "ms": ms, "records_per_s": nrec / (ms * 1e-3),
            "items_per_s": n / (ms * 1e-3)}


SHOWER_NZ, SHOWER_DEPTH = 16, 6


def _shower_particle(t, p, theta):
    """a branching shower (the reference's examples/shower_toy.py workload, with a uniform step length): a particle
    deposits theta[0] of its energy per step along z and, with probability 0.35 per step below generation 6,
    splits off a child with theta[1] x U(0.5, 1) of what is left."""
    from tallymap_amd import lax
    from tallymap_amd import numpy as jnp
    from tallymap_amd import random as R

    def body(c):
        s, n, t = c
        k = R.fold_in(s["key"], n)
        u = R.uniform(k, (3,))
        z = s["z"] + u[0] * 0.5
        dep = s["E"] * theta[0]
        t = t.add("dep", jnp.clip(jnp.floor(z * 2.0).astype(jnp.int32), 0, SHOWER_NZ - 1), dep)
        split = (u[1] < 0.35) & (s["g"] < SHOWER_DEPTH)
        ec = (s["E"] - dep) * theta[1] * (0.5 + 0.5 * u[2])
        t = t.spawn(dict(E=ec, z=z, key=R.fold_in(k, 1), g=s["g"] + 1), when=split)
        e = s["E"] - dep - jnp.where(split, ec, 0.0)
        return dict(E=e, z=z, key=s["key"], g=s["g"]), n + 1, t
    s, n, t = lax.while_loop(lambda c: (c[0]["E"] > 1e-3) & (c[1] < 40), body, (p, 0, t))
    return t.add("count", s["g"], 1)


def bench_spawn(steps, warmup):
    """spawn throughput: the shower from 1,048,576 roots (about 67M particles in 7 generations, Queue 2^25): one
    call is a launch per generation, each sized on the device from the previous one's tickets (the host reads the
    next generation's size after each to know when the tree ends); timed with HIP events on torch's current stream
    around the whole call (the host's generation loop included).  Then the gradient w.r.t. theta, timed the same
    way: by tangent lanes (the default for theta's two elements: one forward through the generations with two
    tangent lanes) and by the tree adjoint (grad_mode='reverse': the recording forward, a count and a reverse
    launch per generation); the two agree within 1e-4."""
    import torch

    import tallymap_amd as tm
    from tallymap_amd import random as R
    n = 1 << 20
    roots = dict(E=torch.linspace(1.0, 2.0, n, dtype=torch.float32, device="cuda"),
                 z=torch.zeros(n, dtype=torch.float32, device="cuda"),
                 key=torch.from_numpy(R._host_split(np.array([0, 7], np.uint32), n).view(np.int32)).cuda()
                 .view(torch.uint32), g=torch.zeros(n, dtype=torch.int32, device="cuda"))
    theta = torch.tensor([0.2, 0.6], dtype=torch.float32, device="cuda")
    f = tm.vmap(_shower_particle, outputs={"dep": tm.Sum((SHOWER_NZ,)), "count": tm.Sum((SHOWER_NZ,), np.int32)},
                in_axes=(0, None), spawn=tm.Queue(1 << 25))
    for _ in range(warmup):
        f(roots, theta)
    torch.cuda.synchronize()
    stream = torch.cuda.current_stream()
    evs = [[torch.cuda.Event(enable_timing=True) for _ in range(2)] for _ in range(steps)]
    for e in evs:
        e[0].record(stream)
        r = f(roots, theta)
        e[1].record(stream)
    torch.cuda.synchronize()
    ms = float(np.mean([e[0].elapsed_time(e[1]) for e in evs]))
    sp, dr = int(r.stats["spawned"].item()), int(r.stats["children_dropped"].item())
    count = r.outputs["count"].cpu().numpy()
    if dr or int(count.sum()) != n + sp:
        raise RuntimeError(f"spawn bench: {sp} spawned, {dr} dropped, {int(count.sum())} particles counted")
    gens = int(np.count_nonzero(count))
    # d <w, dep> / d theta: by default (grad_mode 'auto', theta's 2 elements) tangent lanes -- one forward through
    # the generations, the children carrying their parents' tangents; and the tree adjoint (grad_mode 'reverse':
    # the recording forward, then a count and a reverse launch per generation, deepest first)
    w = torch.linspace(1.0, 2.0, SHOWER_NZ, dtype=torch.float32, device="cuda")
    fr = tm.vmap(_shower_particle, outputs={"dep": tm.Sum((SHOWER_NZ,)), "count": tm.Sum((SHOWER_NZ,), np.int32)},
                 in_axes=(0, None), spawn=tm.Queue(1 << 25), grad_mode="reverse")
    gms, grs = {}, {}
    for mode, fm in (("auto", f), ("reverse", fr)):
        g = tm.grad(fm, weights={"dep": w}, argnums=1)
        g(roots, theta)
        torch.cuda.synchronize()
        gev = [[torch.cuda.Event(enable_timing=True) for _ in range(2)] for _ in range(steps)]
        for e in gev:
            e[0].record(stream)
            gr = g(roots, theta)
            e[1].record(stream)
        torch.cuda.synchronize()
        gms[mode] = float(np.mean([e[0].elapsed_time(e[1]) for e in gev]))
        grs[mode] = gr
        if not bool(torch.isfinite(gr).all()):
            raise RuntimeError(f"spawn bench: {mode} gradient {gr.tolist()}")
    rel = float(((grs["auto"].double() - grs["reverse"].double()).abs() / grs["reverse"].double().abs()).max())
    if not rel <= 1e-4:
        raise RuntimeError(f"spawn bench: lanes {grs['auto'].tolist()} vs tree adjoint {grs['reverse'].tolist()}")
    print("bench: spawn done", file=sys.stderr, flush=True)
    return {"roots": n, "children": sp, "generations": gens, "queue": 1 << 25, "ms": ms,
            "particles_per_s": (n + sp) / (ms * 1e-3), "grad_ms": gms["auto"], "grad_by": "tangent lanes",
            "grad_particles_per_s": (n + sp) / (gms["auto"] * 1e-3), "grad_tree_adjoint_ms": gms["reverse"],
            "grad_tree_adjoint_particles_per_s": (n + sp) / (gms["reverse"] * 1e-3),
            "grad_lanes_vs_tree_adjoint_max_rel": rel}


def bench_configs(steps, warmup, with_cpu):
    """items/s of configs 1, 3, 4, 5 at their BASELINE sizes: the forward call and the gradient call, each timed
    with HIP events on torch's current stream (mean of `steps` after `warmup`); items_per_s = N / (forward +
    gradient).  Where the default (grad_mode 'auto') differentiates by a tangent lane (C1's theta, C3's mu_a, C5's
    A: a scalar through a loop carry), the replay adjoint's gradient call is timed beside it (grad_mode
    'reverse'; C5: its count and reverse launches).  jvp: one fused primal + tangent launch; value_and_grad (C1,
    C3, C4).  The oracle on a bounded sample beside each."""
    import torch

    import tallymap_amd as tm
    from tallymap_amd import _api, configs
    out = {}
    sizes = {"c1": 10_000, "c3": 4_194_304, "c4": 4_194_304, "c5": 1_048_576}
    pos_of = {"c1": 2, "c3": 1, "c4": 3, "c5": 3}
    for name, n in sizes.items():
        inputs = getattr(configs, f"{name}_inputs")(n)
        dev = [torch.from_numpy(np.ascontiguousarray(x)).cuda() if np.ndim(x) else torch.tensor(x).cuda()
               for x in inputs]
        fwd, grad, f = _cfg_runs(name, n, dev)
        fwd_ms, r = _timed(fwd, steps, warmup)
        grad_ms, _ = _timed(grad, steps, warmup)
        assert int(r.stats["n_truncated"].item()) == 0
        pos = pos_of[name]
        m = f._sized(dev, None)
        prog, _, _, _, _, axes = m._prepare(dev)
        lanes = _api._tangent_plan(m, prog, dev, axes, pos) is not None
        d = {"n_items": n, "max_steps": (configs.SIZED[name](n) if name in configs.SIZED
                                         else configs.CONFIGS[name])["max_steps"],
             "items_per_s": n / ((fwd_ms + grad_ms) * 1e-3), "fwd_ms": fwd_ms, "grad_ms": grad_ms,
             "grad_by": "tangent lanes (grad_mode auto)" if lanes else "replay adjoint",
             "fwd_items_per_s": n / (fwd_ms * 1e-3), "grad_items_per_s": n / (grad_ms * 1e-3),
             "mean_trip_count": float(r.per_item.double().mean().item()),
             "max_trip_count": int(r.per_item.max().item())}
        if lanes:
            _, rgrad, _ = _cfg_runs(name, n, dev, mode="reverse")
            d["grad_reverse_ms"], _ = _timed(rgrad, steps, warmup)
            if name == "c5":
                # the replay adjoint's two launches: vjp's forward (the count launch, taping the states) and the
                # pullback (the reverse launch)
                evs = [[torch.cuda.Event(enable_timing=True) for _ in range(3)] for _ in range(steps)]
                stream = torch.cuda.current_stream()
                for e in evs:
                    e[0].record(stream)
                    rgrad(e[1])
                    e[2].record(stream)
                torch.cuda.synchronize()
                d["reverse_count_ms"] = float(np.mean([e[0].elapsed_time(e[1]) for e in evs]))
                d["reverse_pullback_ms"] = float(np.mean([e[1].elapsed_time(e[2]) for e in evs]))
        # forward mode: one fused primal + tangent launch, tangent 1 on the gradient's broadcast parameter
        tans = tuple(torch.ones((), dtype=torch.float32, device="cuda") if i == pos else None
                     for i in range(len(dev)))
        d["jvp_ms"], _ = _timed(lambda: tm.jvp(f, dev, tans), steps, warmup)
        d["jvp_items_per_s"] = n / (d["jvp_ms"] * 1e-3)
        # value_and_grad: the forward's outputs from the gradient's own launches (one for C1's forward-only
        # adjoint or a tangent lane, the count + reverse pair for the tape adjoint)
        if name in ("c1", "c3", "c4"):
            vg = tm.value_and_grad(f, argnums=pos)
            d["vg_ms"], (rv, _) = _timed(lambda: vg(*dev), steps, warmup)
            assert np.array_equal(rv.per_item.cpu().numpy(), r.per_item.cpu().numpy())
            d["vg_items_per_s"] = n / (d["vg_ms"] * 1e-3)
        else:
            d["vg_ms"] = None
            d["vg_note"] = "C5's cotangent (sin theta, omega) is a function of the forward's final states"
        if with_cpu:
            v, m_, dt = _cpu_sample(name, inputs, 8.0)
            d["cpu_items_per_s"] = v
            d["cpu_sample"] = f"first {m_} items, forward + gradient, {dt:.2f} s"
        out[name] = d
        print(f"bench: {name} done ({fwd_ms + grad_ms:.1f} ms per fwd+grad)", file=sys.stderr, flush=True)
    return out


def bench_published(steps, warmup):
    """the reference's own benchmark problems (tallymap_amd/problems.py, from benchmarks/vs_jax/problems/) at the
    size and divergence level of its published L40S kernel-backend rows: the forward call and the gradient of the
    problem's loss w.r.t. theta (the forward call, the loss's cotangent of the tally from its result, the adjoint),
    each timed with HIP events on torch's current stream around the whole call, median of `steps` after `warmup`;
    the published times beside them (jax.jit wall time per call, median of >= 7, on an NVIDIA L40S).  Each mode the
    reference publishes for a problem is timed: fwd, grad (the vjp of the loss: by default tangent lanes where a
    loop carry needs the reverse sweep or the call spawns and theta has at most 8 elements, else the replay adjoint;
    grad_reverse: the replay adjoint -- the tree adjoint for the shower -- always), jvp (a unit tangent on theta) and jacfwd of the loss (a forward-mode lane per element
    of theta)."""
    import torch

    import tallymap_amd as tm
    from tallymap_amd import problems as P
    out = {}
    stream = torch.cuda.current_stream()
    for name, p in P.PROBLEMS.items():
        n = p["n"]
        args, extra = p["inputs"](n)
        dev = [{k: torch.from_numpy(np.ascontiguousarray(v)).cuda() for k, v in x.items()} if isinstance(x, dict)
               else torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in args]
        # the losses' constant arrays resident on the device, as a jitted loss holds them (a host array would be
        # copied on every call, and a pageable copy waits for the stream)
        extra = {k: torch.from_numpy(np.ascontiguousarray(v)).cuda() if isinstance(v, np.ndarray) else v
                 for k, v in extra.items()}
        f = P.mapped(name)
        pub = p["published"]
        runs = {"fwd": lambda: f(*dev)}
        if "grad_ms" in pub:
            def grad(f=f):
                res, pull = tm.vjp(f, *dev, argnums=p["argnum"])
                return pull(p["ct"](res.outputs, n, extra))
            runs["grad"] = grad
            # the replay adjoint (the tree adjoint for the shower) beside the default, which takes tangent lanes
            # for these few-element parameters wherever a loop carry needs the reverse sweep or the call spawns
            runs["grad_reverse"] = lambda fr=P.mapped(name, grad_mode="reverse"): grad(fr)
        if "jvp_ms" in pub:
            tan = tuple(torch.ones_like(x) if i == p["argnum"] else None for i, x in enumerate(dev))
            runs["jvp"] = lambda: tm.jvp(f, dev, tan)
        if "jacfwd_ms" in pub:
            jf = tm.jacfwd(f, argnums=p["argnum"], with_primal=True)

            def jacfwd():
                # jax.jacfwd of the loss: d tally / d theta (one launch: a lane per element of theta, the primal
                # beside them), contracted with the loss's derivative at the primal tally
                jac, prim = jf(*dev)
                ct = p["ct"](prim.outputs, n, extra)
                a = p["argnum"]
                return sum((ct[k].reshape(ct[k].shape + (1,)) * jac[k][a]).reshape(-1, jac[k][a].shape[-1]).sum(0)
                           for k in ct)
            runs["jacfwd"] = jacfwd

        def timed(fn):
            for _ in range(warmup):
                fn()
            torch.cuda.synchronize()
            evs = [[torch.cuda.Event(enable_timing=True) for _ in range(2)] for _ in range(steps)]
            for e in evs:
                e[0].record(stream)
                fn()
                e[1].record(stream)
            torch.cuda.synchronize()
            return float(np.median([e[0].elapsed_time(e[1]) for e in evs]))
        r = runs["fwd"]()
        d = {"n_items": n, "truncated": int(r.stats["n_truncated"].item()), "l40s_source": pub["source"]}
        if r.per_item is not None:
            trips = (r.per_item[-1] if isinstance(r.per_item, (tuple, list)) else r.per_item).double()
            d["mean_trips"], d["max_trips"] = float(trips.mean().item()), int(trips.max().item())
        if "spawned" in r.stats:
            d["children"] = int(r.stats["spawned"].item())
        for mode, fn in runs.items():
            d[f"{mode}_ms"] = timed(fn)
            if f"{mode}_ms" in pub:
                d[f"l40s_{mode}_ms"] = pub[f"{mode}_ms"]
                d[f"{mode}_l40s_over_mi355x_cross_hardware"] = pub[f"{mode}_ms"] / d[f"{mode}_ms"]
        d["l40s_note"] = ("cross-hardware context, not a like-for-like speedup: the published times are the "
                          "reference's jax.jit wall time per call on an NVIDIA L40S; ours are HIP-event times on "
                          "MI355X")
        out[name] = d
        times = ", ".join("%s %.3f ms" % (m, d[m + "_ms"]) for m in runs)
        print(f"bench: published {name} done ({times})", file=sys.stderr, flush=True)
    return out


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--n", type=int, default=4_194_304)
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline")
    ap.add_argument("--headline-only", action="store_true", help="skip the configs 1, 3, 4, 5 and atomics sections")
    ap.add_argument("--copy-probe", type=int, default=0, metavar="BYTES",
                    help="run one plain device copy of BYTES first (its FETCH_SIZE / WRITE_SIZE under rocprofv3 "
                         "calibrate the traffic counters)")
    ap.add_argument("--traffic-bytes", type=float, default=None,
                    help="HBM bytes per dominant-kernel launch (default: the rocprofv3 measurement of this kernel at "
                         "the default N, null at other N)")
    ap.add_argument("--no-valu-rates", action="store_true",
                    help="skip the live VALU issue-rate measurement (counter passes: its kernels are also named "
                         "tm_main)")
    ap.add_argument("--section", choices=("configs", "records", "spawn", "published"), default=None,
                    help="run only this section and print its JSON object (for profiling one workload)")
    a = ap.parse_args()
    if a.copy_probe:
        import torch
        src = torch.ones(a.copy_probe // 4, dtype=torch.float32, device="cuda")
        dst = torch.empty_like(src)
        torch.cuda.synchronize()
        dst.copy_(src)
        torch.cuda.synchronize()
        del src, dst
    if a.section:
        steps = max(3, a.steps // 4)
        run = {"configs": lambda: bench_configs(steps, 1, not a.no_cpu), "records": lambda: bench_records(steps, 1),
               "spawn": lambda: bench_spawn(steps, 1), "published": lambda: bench_published(max(7, steps), 2)}[a.section]
        print(json.dumps({a.section: run()}))
        return
    if a.gpus != 1:
        print(f"bench.py: this build runs on one GPU only (got --gpus {a.gpus}): items shard contiguously over "
              "GPUs with one all-reduce of the tallies, which is designed but not built", file=sys.stderr)
        sys.exit(2)
    import torch

    import tallymap_amd as tm
    from tallymap_amd import backend as B
    from tallymap_amd import configs
    cfg = configs.C2
    x0, keys, drift = configs.c2_inputs(a.n)
    dev = [torch.from_numpy(x0).cuda(), torch.from_numpy(keys).cuda(), torch.tensor(drift).cuda()]
    f = tm.vmap(cfg["item"], outputs=cfg["outputs"], in_axes=cfg["in_axes"], max_steps=cfg["max_steps"])
    g = tm.grad(f, argnums=2)
    vg = tm.value_and_grad(f, argnums=2)
    stream = torch.cuda.current_stream()

    def step(ev=None):
        if ev:
            ev[0].record(stream)
        r, gr = vg(*dev)
        if ev:
            ev[1].record(stream)
        return r, gr

    def two(ev):
        ev[0].record(stream)
        r = f(*dev)
        ev[1].record(stream)
        gr = g(*dev)
        ev[2].record(stream)
        return r, gr
    for _ in range(a.warmup):
        step()
    torch.cuda.synchronize()
    evs = [[torch.cuda.Event(enable_timing=True) for _ in range(2)] for _ in range(a.steps)]
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for i in range(a.steps):
        r, gr = step(evs[i])
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    fused_ms = float(np.mean([e[0].elapsed_time(e[1]) for e in evs]))
    ms = wall * 1e3 / a.steps
    N = a.n
    # sanity: the step computed what it should (no truncation, every item absorbed once, zero gradient)
    assert int(r.stats["n_truncated"].item()) == 0
    assert abs(float(r.outputs["wall"].sum().item()) - N) <= 1e-5 * N
    assert float(gr.item()) == 0.0
    # the same quantities from two launches (outside the timed region above)
    two([torch.cuda.Event(enable_timing=True) for _ in range(3)])
    ev2 = [[torch.cuda.Event(enable_timing=True) for _ in range(3)] for _ in range(max(3, a.steps // 2))]
    torch.cuda.synchronize()
    for e in ev2:
        r2, gr2 = two(e)
    torch.cuda.synchronize()
    fwd_ms = float(np.mean([e[0].elapsed_time(e[1]) for e in ev2]))
    grad_ms = float(np.mean([e[1].elapsed_time(e[2]) for e in ev2]))
    assert float(gr2.item()) == 0.0
    assert np.array_equal(r2.per_item.cpu().numpy(), r.per_item.cpu().numpy())
    dom, dom_ms, bpi = "fused", fused_ms, FWD_BYTES_PER_ITEM
    achieved = bpi * N / (dom_ms * 1e-3) / 1e9
    pi = B.compiled(f._prepare(dev)[0], f._opts)
    info = B.kernel_info(pi)
    ckeys = code_keys(f, dev)
    traffic, t_why = (a.traffic_bytes, None) if a.traffic_bytes is not None else \
        measured(dom, "traffic", ckeys[dom], N)
    out = {
        "metric": "items/s fwd+grad at N=4,194,304 (C2 random walk)",
        "value": N / (ms * 1e-3),
        "unit": "items/s",
        "n_gpus": 1,
        "steps": a.steps,
        "warmup": a.warmup,
        "ms_per_step": ms,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic (seeded threefry keys, x0 ~ U(0.2, 0.8))",
        "config": {"workload": "C2: 1-D random walk, N=4,194,304, forward outputs + replay gradient w.r.t. drift "
                               "per step (tm.value_and_grad: one fused launch)",
                   "n_items": N, "max_steps": cfg["max_steps"], "parallelism": "single GPU"},
        "fused_ms": fused_ms,
        "two_launch_items_per_s": N / ((fwd_ms + grad_ms) * 1e-3),
        "fwd_items_per_s": N / (fwd_ms * 1e-3),
        "grad_items_per_s": N / (grad_ms * 1e-3),
        "fwd_ms": fwd_ms,
        "grad_ms": grad_ms,
        "mean_trip_count": float(r.per_item.double().mean().item()),
        "kernel": {"name": "tm_fused (value_and_grad)", **B.kernel_info(vg_kernel(f, dev))},
        "forward_kernel": {"name": "tm_main (forward)", **info},
        "code_objects": ckeys,
        "roofline": {"bound": "hbm", "achieved": achieved, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": achieved / HBM_PEAK_GBS, "traffic": traffic,
                     "algorithmic_bytes_per_launch": bpi * N,
                     "binding_resource": "VALU issue, not HBM: the kernel moves 17 B per item and runs ~405 "
                                         "steps of ~210 VALU instructions per item; its bound and fraction are "
                                         "valu_roofline's"},
        "valu_roofline": valu_roofline(dom, ckeys[dom], N, dom_ms) if not a.no_valu_rates else None,
    }
    if t_why:
        out["roofline"]["traffic_null"] = t_why
    if not a.no_cpu:
        out["cpu_baseline"] = cpu_baseline(x0, keys, drift, cfg["max_steps"])
    if not a.headline_only:
        # the atomic peaks MI355X does not publish, measured; C2's emits add the constant 1.0 to its privatised
        # occupancy (128 bins) and wall (2 bins) tallies, one per kept step and one per item, which the kernel
        # counts with LDS u64 adds (the flush adds count x 1.0): their peak is lds_u64_128's
        from tallymap_amd.backend import atomics
        peaks = {p: atomics.run(p) for p in atomics.PATTERNS}
        emits = float(r.outputs["occ"].double().sum().item() + r.outputs["wall"].double().sum().item())
        rate = emits / (fwd_ms * 1e-3)
        out["atomics"] = {p: {"adds_per_s": v["adds_per_s"], "exact": v["exact"]} for p, v in peaks.items()}
        out["emit_roofline"] = {"kernel": "tm_main (forward)", "emits_per_launch": emits, "achieved": rate,
                                "peak": peaks["lds_u64_128"]["adds_per_s"], "unit": "LDS u64 atomic adds/s",
                                "frac": rate / peaks["lds_u64_128"]["adds_per_s"],
                                "f32_peak": peaks["lds_f32_128"]["adds_per_s"]}
        print("bench: atomics done", file=sys.stderr, flush=True)
        out["configs"] = bench_configs(max(3, a.steps // 4), 1, not a.no_cpu)
        out["records"] = bench_records(max(3, a.steps // 4), 1)
        out["spawn"] = bench_spawn(max(3, a.steps // 4), 1)
        out["published"] = bench_published(7, 2)
    print(json.dumps(out))


if __name__ == "__main__":
    main()
