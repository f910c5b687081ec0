"""The performance cases: calls a user of this package makes, through its public entry points.

A case is one program (`kind`), one way of calling it (`mode`) and a number of items:

  quickstart   the quickstart walker, 16 bins: short items, one histogram add per step
  walk         the 1-D random walk with absorbing walls: hundreds of steps per item, a heavy tail of lengths
  slab         photon transport in a slab, a 64 x 64 deposit map
  disk         walk on spheres in the unit disk: a score per walker and a 256 x 256 map
  pendulum     driven pendulums, adaptive Dormand-Prince 5(4), the final state per item
  random_walk  the decaying-weight walker, 64 bins, several adds of computed values per item
  transport    packets in a disk, 32 sensors, one add per item
  spheres      walk on spheres for Poisson's equation in the unit square, 64 evaluation points
  ode          forced Van der Pol oscillators, Bogacki-Shampine 3(2), 32 groups
  barrier      up-and-out call paths, 252 daily steps
  gillespie    Schloegl reaction paths, thousands of events per item
  shower       a branching shower through a spawn queue
  records      the quickstart walker appending one record per step

  forward         the mapped call
  fixed_point     the mapped call with an order-independent (fixed-point) sum
  value_and_grad  outputs and gradient w.r.t. the broadcast parameter
  reverse         the same with the reproducible replay gradient
  loss_grad       vjp, then the pullback of a loss of the outputs (what a fit runs)
  items_grad      vjp w.r.t. per-item arguments (initial values), then the pullback
  jacfwd          the Jacobian of the outputs w.r.t. the broadcast parameters

The programs are the package's own configurations and problems; their inputs are drawn on the GPU from the case's
seed, with the distributions those configurations use."""
import math

import numpy as np
import torch

import tallymap_amd as tm
from tallymap_amd import configs, lax, problems, random
from tallymap_amd import numpy as jnp

MODES = {"quickstart": ("forward", "value_and_grad", "fixed_point", "items_grad"),
         "walk": ("forward", "value_and_grad"),
         "slab": ("forward", "value_and_grad", "reverse"),
         "disk": ("forward", "value_and_grad"),
         "pendulum": ("forward", "loss_grad"),
         "random_walk": ("forward", "loss_grad", "jacfwd"),
         "transport": ("forward", "loss_grad"),
         "spheres": ("forward", "jacfwd"),
         "ode": ("forward", "loss_grad", "items_grad"),
         "barrier": ("forward", "loss_grad"),
         "gillespie": ("forward",),
         "shower": ("forward", "loss_grad"),
         "records": ("forward",)}
# the items of a drawn case: from a few wavefronts to the sizes the benchmark runs each program at, fewer for the
# programs whose items take hundreds or thousands of steps
LARGEST = {"walk": 2_097_152, "pendulum": 524_288, "ode": 524_288, "barrier": 2_097_152, "gillespie": 131_072,
           "shower": 262_144}
# per item, mean steps and the arithmetic operations of a step (random bits, libm polynomials and updates counted
# from the programs: a threefry2x32 hash 75, a float32 transcendental 20)
STEPS = {"quickstart": (8.0, 165), "walk": (406.0, 210), "slab": (10.2, 520), "disk": (9.15, 215),
         "pendulum": (254.5, 430), "random_walk": (25.5, 170), "transport": (16.1, 330), "spheres": (8.8, 480),
         "ode": (227.4, 190), "barrier": (221.0, 230), "gillespie": (1916.0, 290), "shower": (33.0, 330),
         "records": (8.0, 165)}


def listed():
    """Twelve calls from the smallest to the largest."""
    return [
        # a script's first try of a program: launches and latency are everything
        {"name": "quickstart_1k", "kind": "quickstart", "mode": "forward", "n": 1000},
        # the quickstart as published: outputs and gradient of 10,000 walkers
        {"name": "quickstart_grad_10k", "kind": "quickstart", "mode": "value_and_grad", "n": 10_000},
        # pricing at an interactive size: fewer paths than the chip has lanes, 252 dependent steps each
        {"name": "barrier_4k", "kind": "barrier", "mode": "forward", "n": 4096},
        # an ordinary odd-sized ensemble of long walks: the longest item is ten times the mean
        {"name": "walk_50k", "kind": "walk", "mode": "forward", "n": 50_021},
        # initial-value sensitivities of an ODE ensemble: the taped replay adjoint (forward, then backward)
        {"name": "ode_items_grad_65k", "kind": "ode", "mode": "items_grad", "n": 65_537},
        # the reproducible gradient of photon transport: the adjoint's tape and its reverse launch
        {"name": "slab_reverse_500k", "kind": "slab", "mode": "reverse", "n": 500_009},
        # final-energy gradient of a pendulum ensemble: arithmetic of a high-order integrator with tangents
        {"name": "pendulum_grad_260k", "kind": "pendulum", "mode": "loss_grad", "n": 262_144},
        # a spawning cascade and its gradient, generation by generation
        {"name": "shower_grad_260k", "kind": "shower", "mode": "loss_grad", "n": 262_144},
        # per-step event records of 1.5M walkers, in canonical order
        {"name": "records_1500k", "kind": "records", "mode": "forward", "n": 1_500_007},
        # one iteration of a fit at the benchmark's size: loss gradient of a histogram
        {"name": "random_walk_grad_4m", "kind": "random_walk", "mode": "loss_grad", "n": 4_194_304},
        # many short walks into large outputs: a row per walker and a 256 x 256 map
        {"name": "disk_grad_4m", "kind": "disk", "mode": "value_and_grad", "n": 4_194_304},
        # the headline workload: forward and gradient of 4M long walks
        {"name": "walk_grad_4m", "kind": "walk", "mode": "value_and_grad", "n": 4_194_304},
    ]


def draw(rng):
    """A program, a mode of it, and a size spread over the logarithm of its range."""
    kind = rng.choice(sorted(MODES))
    n = int(math.exp(rng.uniform(math.log(700.0), math.log(float(LARGEST.get(kind, 4_194_304))))))
    return {"kind": kind, "mode": rng.choice(MODES[kind]), "n": n}


# ---------------------------------------------------------------------------------------------------- inputs
def _inputs(case, seed):
    """(per-item and broadcast arguments, what the loss needs) on the GPU, from the seed."""
    kind, n = case["kind"], case["n"]
    g = torch.Generator(device="cuda").manual_seed(seed)

    def u(lo, hi, *shape):
        return torch.rand(shape, generator=g, device="cuda", dtype=torch.float64).mul_(hi - lo).add_(lo)

    def f(x):
        return torch.as_tensor(x, dtype=torch.float32, device="cuda").contiguous()
    keys = torch.randint(-2 ** 31, 2 ** 31, (n, 2), generator=g, device="cuda", dtype=torch.int32).view(torch.uint32)
    ids = torch.arange(n, device="cuda", dtype=torch.int32)
    if kind in ("quickstart", "records"):
        return (f(u(0.1, 0.99, n)), keys, f(2.0)), {"w": f(u(0.5, 1.5, 16))}
    if kind == "walk":
        return (f(u(0.2, 0.8, n)), keys, f(1e-3)), {}
    if kind == "slab":
        return (keys, f(0.1)), {}
    if kind in ("disk", "transport"):
        r, a = u(0.0, 1.0, n).sqrt_() * (0.95 if kind == "disk" else 0.5), u(0.0, 2.0 * math.pi, n)
        p = f(torch.stack([r * a.cos(), r * a.sin()], 1))
        if kind == "disk":
            return (p, keys, ids, f(0.75)), {}
        return ((p, keys, f([0.2, 0.5]), f(0.8 + 0.2 * np.cos(np.arange(problems.TR_NS)))),
                {"tgt": f(u(5.0, 30.0, problems.TR_NS))})
    if kind == "pendulum":
        return (f(u(-math.pi, math.pi, n)), f(u(-2.0, 2.0, n)), ids, f(1.2)), {}
    if kind == "random_walk":
        return (keys, f(u(0.60, 0.95, n)), f([1.0, 0.5, 0.25])), {"wq": f(u(0.5, 1.5, problems.RW_NB))}
    if kind == "spheres":
        return (f(u(0.02, 0.98, n, 2)), ids % problems.WS_M, keys, f([1.0, 4.0, 0.3, 0.5, 2.0])), {}
    if kind == "ode":
        y0 = torch.stack([u(-2.0, 2.0, n), u(-1.0, 1.0, n)], 1)
        return (f(y0), f(u(math.log(0.5), math.log(6.0), n).exp_()), ids % problems.OD_G, f([1.0, 0.05, 0.3])), {
            "w": f(u(0.5, 1.5, problems.OD_G))}
    if kind == "barrier":
        return (keys, f([0.25, 0.03, 100.0]), f(np.linspace(0.8, 1.2, problems.BA_NK))), {
            "w": f(u(1.0, 2.0, problems.BA_NK))}
    if kind == "gillespie":
        x0 = torch.randint(100, 501, (n,), generator=g, device="cuda", dtype=torch.int32)
        return (x0, keys, f([3.0e-7, 1.0e-4, 1.0e-3, 3.5])), {}
    z = torch.zeros(n, device="cuda", dtype=torch.int32)          # shower
    return (dict(E=f(u(1.0, 2.0, n)), z=f(torch.zeros(n, device="cuda")), key=keys, g=z, n=z.clone(), did=z.clone()),
            f([0.2, 0.6])), {"wz": f(u(0.5, 1.5, problems.SH_NZ))}


def _record_item(t, x, key, theta):
    """The quickstart walker writing (bin, weight) per step."""
    def body(c):
        k, x, t = c
        u = random.uniform(random.fold_in(key, k))
        t = t.append("steps", dict(bin=(x * configs.NB).astype(jnp.int32), w=theta * (1.0 - x)))
        return k + 1, x * (0.5 + 0.5 * u), t
    k, x, t = lax.while_loop(lambda c: c[1] > 0.05, body, (0, x, t))
    return t, k


PROBLEM = {"spheres": "walk_on_spheres", "ode": "ode_ensemble"}


def _mapped(case):
    """The mapped call of a case, as a program builds it once."""
    kind, n = case["kind"], case["n"]
    if kind == "records":
        return tm.vmap(_record_item, outputs={"steps": tm.Records({"bin": np.int32, "w": np.float32}, capacity=9 * n)},
                       in_axes=(0, 0, None), max_steps=100)
    if kind == "shower":
        p = problems.PROBLEMS[kind]
        return tm.vmap(p["item"], outputs=p["outputs"], in_axes=p["in_axes"], spawn=tm.Queue(n))
    if kind in ("quickstart", "walk", "slab", "disk", "pendulum"):
        c = {"quickstart": configs.C1, "walk": configs.C2, "slab": configs.C3}.get(kind) or (
            configs.c4_config(n) if kind == "disk" else configs.c5_config(n))
        outs, opts = c["outputs"], dict(c.get("opts", {}))
        if case["mode"] == "fixed_point":
            outs = {"hist": tm.Sum((configs.NB,), fixed_point=True)}
        if case["mode"] == "reverse":
            opts["grad_mode"] = "reverse"
        return tm.vmap(c["item"], outputs=outs, in_axes=c["in_axes"], max_steps=c["max_steps"], **opts)
    return problems.mapped(PROBLEM.get(kind, kind))


ARGNUM = {"quickstart": 2, "walk": 2, "slab": 1, "disk": 3, "pendulum": 3, "random_walk": 2, "transport": 2,
          "spheres": 3, "ode": 3, "barrier": 1, "shower": 1}


def prepare(case, seed):
    args, extra = _inputs(case, seed)
    f = _mapped(case)
    call = None
    if case["mode"] in ("value_and_grad", "reverse"):
        call = tm.value_and_grad(f, argnums=ARGNUM[case["kind"]])
    elif case["mode"] == "jacfwd":
        call = tm.jacfwd(f, argnums=ARGNUM[case["kind"]], with_primal=True)
    return {"case": case, "args": args, "extra": extra, "f": f, "call": call}


# ------------------------------------------------------------------------------------------------------ runs
def _cotangent(case, outputs, extra):
    """The derivative of the case's loss at the outputs, on the device."""
    kind, n = case["kind"], case["n"]
    if kind == "pendulum":             # the summed final energy omega^2 / 2 + 1 - cos(theta)
        s = outputs["state"]
        return {"state": torch.stack([torch.sin(s[:, 0]), s[:, 1]], 1)}
    if kind == "quickstart":
        return {"hist": extra["w"]}
    return problems.PROBLEMS[PROBLEM.get(kind, kind)]["ct"](outputs, n, extra)


def _result(r):
    out = {"outputs": r.outputs, "dropped": r.stats["dropped_emits"], "truncated": r.stats["n_truncated"]}
    if r.per_item is not None:
        out["per_item"] = r.per_item
    return out


def run(state):
    case, args, mode = state["case"], state["args"], state["case"]["mode"]
    if mode in ("forward", "fixed_point"):
        return _result(state["f"](*args))
    if mode in ("loss_grad", "items_grad"):
        argnums = ARGNUM[case["kind"]] if mode == "loss_grad" else 0
        res, pullback = tm.vjp(state["f"], *args, argnums=argnums)
        return dict(_result(res), grad=pullback(_cotangent(case, res.outputs, state["extra"])))
    if mode == "jacfwd":
        jac, res = state["call"](*args)
        return dict(_result(res), jac=jac)
    res, grad = state["call"](*args)
    return dict(_result(res), grad=grad)


# ------------------------------------------------------------------------------------------- work, tolerance
# bytes per item: operands read and per-item results written (truncation flag included where there is a cap)
ITEM_BYTES = {"quickstart": 12 + 5, "walk": 12 + 5, "slab": 8 + 5, "disk": 20 + 9, "pendulum": 12 + 13,
              "random_walk": 12 + 4, "transport": 16 + 4, "spheres": 20 + 4, "ode": 16 + 4, "barrier": 8 + 8,
              "gillespie": 12 + 8, "shower": 28, "records": 12 + 5}
BINS = {"quickstart": 16, "walk": 130, "slab": 4096, "disk": 65536, "random_walk": 64, "transport": 32, "spheres": 64,
        "ode": 32, "barrier": 9, "gillespie": 33, "shower": 16}
# arithmetic of a differentiated call relative to the forward's: what the derivative itself needs (nothing for the
# histogram of a walk whose bins do not move, a lane's multiplies for the others)
GRAD = {"walk": 0.02, "disk": 0.05, "quickstart": 0.05, "slab": 0.15, "pendulum": 0.4, "random_walk": 0.1,
        "transport": 0.05, "spheres": 0.1, "ode": 0.8, "barrier": 0.1, "shower": 0.15}


def work(case):
    kind, n, mode = case["kind"], case["n"], case["mode"]
    steps, ops = STEPS[kind]
    nbytes = n * ITEM_BYTES[kind] + 4 * BINS.get(kind, 0)
    flops = n * steps * ops
    if kind == "records":
        nbytes += 8 * 9 * n                       # the whole output, its unused part zero
    if mode == "items_grad":
        nbytes += n * (8 if kind == "ode" else 4)
    if mode not in ("forward", "fixed_point"):
        flops *= 1.0 + GRAD[kind]
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Whole values are the same.  A float32 sum depends on the order of its adds: two runs of one build differ by
    up to 1.6e-6 (2-norm, over the programs and sizes here), a sum in float64 from either by as much; records are
    copies."""
    return {"rel": 1e-7} if case["kind"] == "records" else {"rel": 1e-5}


# ----------------------------------------------------------------------------------------------------- exact
# The same programs in torch: float64 arithmetic on the same float32 uniform draws, all live items one step at a
# time.  A quantity differentiated in forward mode carries its tangents in dual tensors.
def _hash(k0, k1, c1):
    """threefry2x32 with counter (0, c1) on int64 tensors holding 32-bit words."""
    m = 0xFFFFFFFF
    ks = (k0, k1, k0 ^ k1 ^ 0x1BD11BDA)
    a, b = ks[0], (ks[1] + c1) & m
    for g in range(5):
        for r in ((13, 15, 26, 6), (17, 29, 16, 24))[g & 1]:
            a = (a + b) & m
            b = (((b << r) | (b >> (32 - r))) & m) ^ a
        a, b = (a + ks[(g + 1) % 3]) & m, (b + ks[(g + 2) % 3] + g + 1) & m
    return a, b


def _uniform(keys, k, count=1):
    """uniform(fold_in(key, k), (count,)): float32 draws, held in float64."""
    a, b = _hash(keys[:, 0], keys[:, 1], k)
    out = []
    for i in range(count):
        p, q = _hash(a, b, i)
        out.append(((p ^ q) >> 9).double() * 2.0 ** -23)
    return out


def _loop(state, alive, body):
    """while alive(state): state = body(state), item by item: live items are kept dense, finished ones put back."""
    final = [x.clone() for x in state]
    index = torch.arange(state[0].shape[0], device="cuda")
    while index.numel():
        live = alive(state)
        if not bool(live.all()):
            for whole, x in zip(final, state):
                whole[index[~live]] = x[~live]
            index = index[live]
            state = [x[live] for x in state]
            if not index.numel():
                break
        state = body(state)
    return final


def _bins(total, bin_, value):
    """total[..., bin] += value; a bin outside is dropped.  value: [lanes, items]."""
    ok = (bin_ >= 0) & (bin_ < total.shape[-1])
    return total.index_add_(-1, bin_[ok], value[..., ok].to(total.dtype))


def _trunc(x):
    return x.trunc().long()
H = 1e-30                    # the complex step: an imaginary perturbation this small differentiates exactly


def _re(x):
    return x.real if x.is_complex() else x


def _normal(keys, k):
    lo = np.nextafter(np.float32(-1.0), np.float32(0.0))
    u = _uniform(keys, k)[0].float() * float(np.float32(1.0) - lo) + float(lo)
    return math.sqrt(2.0) * torch.erfinv(u.double())


def _sim_quickstart(case, args, sums, n):
    def body(s):
        x, keys, k, i = s
        b, v = _trunc(_re(x) * configs.NB), args[2] * (1.0 - x)
        _bins(sums["hist"], b, v)
        if "items" in sums:
            sums["items"].index_add_(0, i, v * sums["w"][b])
        return [x * (0.5 + 0.5 * _uniform(keys, k)[0]), keys, k + 1, i]
    ids = torch.arange(n, device="cuda")
    _loop([args[0], args[1], torch.zeros_like(ids), ids], lambda s: _re(s[0]) > 0.05, body)


def _sim_walk(case, args, sums, n):
    def body(s):
        x, keys, k = s
        _bins(sums["occ"], _trunc(_re(x) * 128), torch.ones_like(x))
        return [x + (args[2] + 0.02 * _normal(keys, k)), keys, k + 1]
    x = _loop([args[0].to(args[2].dtype), args[1], torch.zeros(n, device="cuda", dtype=torch.long)],
              lambda s: (_re(s[0]) >= 0.0) & (_re(s[0]) <= 1.0), body)[0]
    _bins(sums["wall"], (_re(x) > 1.0).long(), torch.ones_like(x))


def _sim_slab(case, args, sums, n):
    mu_a, g = args[1], configs.C3_G
    mu_t = mu_a + configs.C3_MU_S

    def body(s):
        p, d, w, keys, k = s
        u = _uniform(keys, k, 4)
        p = p + (-torch.log(1.0 - u[0]) / mu_t)[:, None] * d
        z, r = _re(p[:, 2]), _re(p[:, :2]).square().sum(1).sqrt()
        esc = (z < 0.0) | (z > configs.C3_DEPTH)
        nb = configs.C3_NB
        iz, ir = _trunc(z * (nb / configs.C3_DEPTH)), _trunc(r * (nb / configs.C3_DEPTH))
        _bins(sums["absorbed"], torch.where(esc | (iz >= nb) | (ir >= nb), -1, iz * nb + ir), w * (mu_a / mu_t))
        w = w * (configs.C3_MU_S / mu_t)
        tmp = (1.0 - g * g) / (1.0 - g + 2.0 * g * u[1])
        cost = (1.0 + g * g - tmp * tmp) / (2.0 * g)
        sint = (1.0 - cost * cost).clamp(min=0.0).sqrt()
        cp, sp = torch.cos(2.0 * math.pi * u[2]), torch.sin(2.0 * math.pi * u[2])
        ux, uy, uz = d.unbind(1)
        temp = (1.0 - uz * uz).clamp(min=0.0).sqrt()
        near = uz.abs() > 0.99999
        den = torch.where(near, 1.0, temp)
        d = torch.stack([torch.where(near, sint * cp, sint * (ux * uz * cp - uy * sp) / den + ux * cost),
                         torch.where(near, sint * sp, sint * (uy * uz * cp + ux * sp) / den + uy * cost),
                         torch.where(near, torch.sign(uz) * cost, -sint * cp * temp + uz * cost)], 1)
        w = torch.where(_re(w) < 0.01, torch.where(u[3] < 0.1, w * 10.0, 0.0 * w), w)
        return [p, d, torch.where(esc, 0.0 * w, w), keys, k + 1]
    d = torch.zeros(n, 3, device="cuda", dtype=torch.float64)
    p, w = d.to(mu_a.dtype), torch.ones(n, device="cuda", dtype=mu_a.dtype)
    d = d.clone()
    d[:, 2] = 1.0
    _loop([p, d, w, args[0], torch.zeros(n, device="cuda", dtype=torch.long)], lambda s: _re(s[2]) > 0.0, body)


def _sim_disk(case, args, sums, n):
    def body(s):
        p, keys, k = s
        phi = 2.0 * math.pi * _uniform(keys, k)[0]
        return [p + (1.0 - p.norm(dim=1))[:, None] * torch.stack([phi.cos(), phi.sin()], 1), keys, k + 1]
    p = _loop([args[0], args[1], torch.zeros(n, device="cuda", dtype=torch.long)],
              lambda s: 1.0 - s[0].norm(dim=1) >= configs.C4_EPS, body)[0]
    score = args[3] * torch.sin(3.0 * torch.atan2(p[:, 1], p[:, 0]))
    sums["walker"] = score[:, None]
    i = _trunc((args[0] + 1.0) * (configs.C4_NB / 2.0))
    _bins(sums["grid"], i[:, 0] * configs.C4_NB + i[:, 1], score)


def _sim_pendulum(case, args, sums, n):
    A, a, b, e = args[3], configs.DP_A, configs.DP_B, configs.DP_E

    def rhs(t, y):
        return torch.stack([y[:, 1], -configs.C5_DAMP * y[:, 1] - torch.sin(y[:, 0])
                            + A * torch.cos(configs.C5_WD * t)], 1)

    def body(s):
        t, y, f0, h = s
        h = torch.minimum(h, configs.C5_T1 - t)
        ks, hh = [f0], h[:, None]
        for row, c in zip(a, configs.DP_C + (1.0,)):
            ks.append(rhs(t + c * h, y + hh * sum(w * q for w, q in zip(row, ks))))
        k = [ks[0]] + ks[2:6]
        y5 = y + hh * sum(w * q for w, q in zip(b, k))
        k.append(rhs(t + h, y5))
        scale = configs.C5_ATOL + configs.C5_RTOL * torch.maximum(y.abs(), y5.abs())
        q = hh * sum(w * x for w, x in zip(e, k)) / scale
        err = (q.square().sum(1) * 0.5).sqrt()
        ok = err <= 1.0
        return [torch.where(ok, t + h, t), torch.where(ok[:, None], y5, y), torch.where(ok[:, None], k[5], f0),
                h * (0.9 * err ** -0.2).clamp(0.2, 10.0)]
    y = torch.stack([args[0], args[1]], 1)
    t = torch.zeros(n, device="cuda", dtype=torch.float64)
    sums["state"] = _loop([t, y, rhs(t, y), t + configs.C5_H0], lambda s: s[0] < configs.C5_T1, body)[1]


def _sim_random_walk(case, args, sums, n):
    th = args[2]

    def body(s):
        w, decay, keys, k = s
        u = _uniform(keys, k)[0]
        _bins(sums["hist"], _trunc(u * problems.RW_NB), w * th[0] + th[1] * u + th[2] * w * w)
        return [w * decay, decay, keys, k + 1]
    w = torch.ones(n, device="cuda", dtype=torch.float64)
    _loop([w, args[1], args[0], torch.zeros(n, device="cuda", dtype=torch.long)],
          lambda s: s[0] > problems.RW_WMIN, body)


def _sim_transport(case, args, sums, n):
    th, eff = args[2], args[3]

    def body(s):
        p, d, w, keys, k, _ = s
        u = _uniform(keys, k, 2)
        fl = -torch.log1p(-u[0]) * th[0]
        p, phi = p + fl[:, None] * d, 2.0 * math.pi * u[1]
        return [p, torch.stack([phi.cos(), phi.sin()], 1), w * torch.exp(-th[1] * fl), keys, k + 1,
                _re(p).square().sum(1) >= 1.0]
    w = torch.ones(n, device="cuda", dtype=th.dtype)
    d = torch.zeros(n, 2, device="cuda", dtype=torch.float64)
    d[:, 0] = 1.0
    p, _, w, _, _, esc = _loop([args[0].to(th.dtype), d, w, args[1], torch.zeros(n, device="cuda", dtype=torch.long),
                                torch.zeros(n, device="cuda", dtype=torch.bool)],
                               lambda s: ~s[5] & (_re(s[2]) > problems.TR_WMIN), body)
    angle = torch.atan2(_re(p[:, 1]), _re(p[:, 0])) + math.pi
    i = _trunc(angle * (problems.TR_NS / (2.0 * math.pi))) % problems.TR_NS
    _bins(sums["Q"], torch.where(esc, i, -1), w * eff[i])


def _sim_spheres(case, args, sums, n):
    th = args[3]

    def sdf(x):
        return torch.minimum(x, 1.0 - x).amin(1)

    def body(s):
        x, acc, keys, k = s
        R, u = sdf(x), _uniform(keys, k, 3)
        a, a2 = 2.0 * math.pi * u[1], 2.0 * math.pi * u[2]
        y = x + (R * u[0].sqrt())[:, None] * torch.stack([a.cos(), a.sin()], 1)
        f = th[0] * torch.exp(-th[1] * (y - 0.5).square().sum(1))
        acc = acc + 0.5 * R * R * (-0.5 * torch.log(u[0].clamp(min=1e-20))) * f
        return [x + R[:, None] * torch.stack([a2.cos(), a2.sin()], 1), acc, keys, k + 1]
    x, acc, _, _ = _loop([args[0], torch.zeros(n, device="cuda", dtype=th.dtype), args[2],
                          torch.zeros(n, device="cuda", dtype=torch.long)], lambda s: sdf(s[0]) > problems.WS_EPS, body)
    i = torch.stack([x[:, 0], 1.0 - x[:, 0], x[:, 1], 1.0 - x[:, 1]], 1).argmin(1)
    bx = torch.where(i == 0, 0.0, torch.where(i == 1, 1.0, x[:, 0]))
    by = torch.where(i == 2, 0.0, torch.where(i == 3, 1.0, x[:, 1]))
    _bins(sums["u"], args[1], acc + (th[2] + th[3] * torch.cos(th[4] * math.pi * (bx + by))))


def _sim_ode(case, args, sums, n):
    th = args[3]

    def rhs(t, y, mu):
        return torch.stack([y[:, 1], mu * th[0] * (1.0 - y[:, 0] * y[:, 0]) * y[:, 1] - y[:, 0] - th[1] * y[:, 1]
                            + th[2] * torch.sin(2.0 * t)], 1)

    def body(s):
        t, y, h, mu = s
        h = torch.minimum(h, problems.OD_T - t)
        hh = h[:, None]
        k1 = rhs(t, y, mu)
        k2 = rhs(t + 0.5 * h, y + 0.5 * hh * k1, mu)
        k3 = rhs(t + 0.75 * h, y + 0.75 * hh * k2, mu)
        yn = y + hh * (2.0 / 9.0 * k1 + 1.0 / 3.0 * k2 + 4.0 / 9.0 * k3)
        k4 = rhs(t + h, yn, mu)
        e = (2.0 / 9.0 - 7.0 / 24.0) * k1 + (1.0 / 3.0 - 0.25) * k2 + (4.0 / 9.0 - 1.0 / 3.0) * k3 - 0.125 * k4
        scale = problems.OD_ATOL + problems.OD_RTOL * torch.maximum(_re(y).abs(), _re(yn).abs())
        err = ((hh * _re(e)).abs() / scale).amax(1)
        ok = err <= 1.0
        fac = (0.9 * err.clamp(min=1e-10) ** (-1.0 / 3.0)).clamp(0.2, 5.0)
        return [torch.where(ok, t + h, t), torch.where(ok[:, None], yn, y), (h * fac).clamp(min=1e-7), mu]
    t = torch.zeros(n, device="cuda", dtype=torch.float64)
    y0 = args[0] if args[0].is_complex() or not th.is_complex() else args[0].to(th.dtype)
    y = _loop([t, y0, t + 1e-2, args[1]], lambda s: s[0] < problems.OD_T, body)[1]
    o = torch.tanh(y[:, 0]) + 0.5 * y[:, 1] * torch.exp(-0.1 * y[:, 1] * y[:, 1])
    _bins(sums["obs"], args[2], o)
    sums["items"] = o


def _sim_barrier(case, args, sums, n):
    th, strikes, dt = args[1], args[2], problems.BA_DT

    def body(s):
        S, keys, k, _ = s
        S = S * torch.exp((th[1] - 0.5 * th[0] * th[0]) * dt + th[0] * problems.BA_SQDT * _normal(keys, k))
        return [S, keys, k + 1, _re(S) < problems.BA_BAR * _re(th)[2]]
    S, _, _, alive = _loop([th[2].expand(n).clone(), args[0], torch.zeros(n, device="cuda", dtype=torch.long),
                            torch.ones(n, device="cuda", dtype=torch.bool)],
                           lambda s: (s[2] < problems.BA_KSTEPS) & s[3], body)
    gain = S[:, None] - strikes * th[2]
    pay = torch.exp(-th[1] * problems.BA_T) * torch.where(_re(gain) > 0, gain, 0.0 * gain) * alive[:, None]
    sums["price"] += pay.sum(0)
    sums["ko"] += (~alive).double().sum()
    sums["pay"] = pay[:, problems.BA_NK // 2]


def _sim_gillespie(case, args, sums, n):
    c = args[2]

    def body(s):
        t, x, keys, k = s
        a = torch.stack([c[0] * problems.GI_A * x * (x - 1.0) * 0.5, c[1] * x * (x - 1.0) * (x - 2.0) / 6.0,
                         (c[2] * problems.GI_B).expand(x.shape[0]), c[3] * x], 1).clamp(min=0.0)
        a0, u = a.sum(1), _uniform(keys, k, 2)
        r = ((u[1] * a0)[:, None] > a.cumsum(1)).sum(1).clamp(0, 3)
        return [t - torch.log(u[0].clamp(min=1e-20)) / a0.clamp(min=1e-20),
                (x + 1.0 - 2.0 * (r & 1)).clamp(0.0, 2000.0), keys, k + 1]
    x = _loop([torch.zeros(n, device="cuda", dtype=torch.float64), args[0].double(), args[1],
               torch.zeros(n, device="cuda", dtype=torch.long)], lambda s: s[0] < problems.GI_T, body)[1]
    b = _trunc(x * (problems.GI_NB / problems.GI_XMAX)).clamp(0, problems.GI_NB - 1)
    _bins(sums["hist"], b, torch.ones_like(x))
    sums["mean"] += x.sum()


def _sim_shower(case, args, sums, n):
    roots, th = args
    queue = [(roots["E"].to(th.dtype), roots["z"], roots["key"], roots["g"])]

    def body(s):
        E, z, keys, g, k, did = s
        a, b = _hash(keys[:, 0], keys[:, 1], k)
        here = torch.stack([a, b], 1)
        u = [((p ^ q) >> 9).double() * 2.0 ** -23 for p, q in (_hash(a, b, i) for i in range(3))]
        z = z - torch.log1p(-u[0]) * 0.5
        dep = E * th[0]
        split = (u[1] < problems.SH_PSPLIT) & (g < problems.SH_DEPTH) & ~did & (_re(E) > problems.SH_EMIN)
        ec = (E - dep) * th[1] * (0.5 + 0.5 * u[2])
        _bins(sums["dep"], torch.floor(z * 2.0).long().clamp(0, problems.SH_NZ - 1), dep)
        if bool(split.any()):
            h = here[split]
            queue.append((ec[split], z[split], torch.stack(_hash(h[:, 0], h[:, 1], 1), 1), g[split] + 1))
        return [E - dep - torch.where(split, ec, 0.0 * ec), z, keys, g, k + 1, did | split]
    while queue:
        parts = list(zip(*queue))
        E, z, keys, g = (torch.cat(p) for p in parts)
        queue.clear()
        zero = torch.zeros(E.shape[0], device="cuda", dtype=torch.long)
        _loop([E, z, keys, g, zero, zero.bool()],
              lambda s: (_re(s[0]) > problems.SH_EMIN) & (s[4] < problems.SH_KMAX), body)


SHAPES = {"quickstart": {"hist": (16,)}, "walk": {"occ": (128,), "wall": (2,)}, "slab": {"absorbed": (4096,)},
          "disk": {"grid": (65536,)}, "pendulum": {}, "random_walk": {"hist": (problems.RW_NB,)},
          "transport": {"Q": (problems.TR_NS,)}, "spheres": {"u": (problems.WS_M,)}, "ode": {"obs": (problems.OD_G,)},
          "barrier": {"price": (problems.BA_NK,), "ko": (1,)}, "gillespie": {"hist": (problems.GI_NB,), "mean": (1,)},
          "shower": {"dep": (problems.SH_NZ,)}}
# (larger calls would take minutes item by item)
EXACT_ITEMS = {"walk": 120_000, "gillespie": 20_000}


def exact(case, seed):
    """The float outputs of run() in float64; None for whole numbers, for records (a rounding that adds one record
    moves all that follow) and for the pendulums' gradient (some of them are chaotic)."""
    kind, n, mode = case["kind"], case["n"], case["mode"]
    if kind == "records" or n > EXACT_ITEMS.get(kind, 1 << 30):
        return None
    args, extra = _inputs(case, seed)

    def wide(a):
        if isinstance(a, dict):
            return {k: wide(v) for k, v in a.items()}
        if a.dtype == torch.uint32:
            return a.view(torch.int32).long() & 0xFFFFFFFF
        return a.double() if a.dtype == torch.float32 else a.long()
    args = [wide(a) for a in args]
    extra = {k: v.double() for k, v in extra.items()}

    def simulate(perturbed=None, element=None):
        a = list(args)
        dt = torch.float64
        if perturbed is not None:
            dt = torch.complex128
            x = a[perturbed].to(dt)
            if element is None:
                x = x + 1j * H
            else:
                x = x.clone()
                x[element] += 1j * H
            a[perturbed] = x
        sums = {k: torch.zeros(s, device="cuda", dtype=dt) for k, s in SHAPES[kind].items()}
        if kind == "quickstart" and mode == "items_grad":
            sums.update(items=torch.zeros(n, device="cuda", dtype=dt), w=extra["w"])
        globals()["_sim_" + kind](case, a, sums, n)
        return sums
    sums = simulate()
    names = set(SHAPES[kind]) | ({"walker"} if kind == "disk" else {"state"} if kind == "pendulum" else set())
    shape = {"absorbed": (64, 64), "grid": (256, 256)}
    out = {"outputs": {k: sums[k].reshape(shape.get(k, sums[k].shape)) for k in names}}
    if kind == "barrier":
        out["per_item"] = [sums["pay"], None]
    if mode in ("forward", "fixed_point") or kind == "pendulum":
        return out
    if mode == "items_grad":
        ct = _cotangent(case, out["outputs"], extra)
        if kind == "quickstart":
            out["grad"] = simulate(0)["items"].imag / H
        else:
            out["grad"] = torch.stack([simulate(0, (slice(None), j))["items"].imag / H * ct["obs"][args[2]]
                                       for j in range(2)], 1)
        return out
    arg = args[ARGNUM[kind]]
    places = [None] if arg.dim() == 0 else range(arg.shape[0])
    tangents = [simulate(ARGNUM[kind], p) for p in places]
    if mode == "jacfwd":
        out["jac"] = {k: {ARGNUM[kind]: torch.stack([t[k].imag / H for t in tangents], -1)} for k in names}
        return out
    ct = {k: 1.0 for k in names} if mode != "loss_grad" else _cotangent(case, out["outputs"], extra)
    total = [sum((t[k].imag / H * ct[k]).sum() for k in ct) for t in tangents]
    out["grad"] = total[0] if arg.dim() == 0 else torch.stack(total)
    return out
