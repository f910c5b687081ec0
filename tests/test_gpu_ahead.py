"""Steps computed ahead by idle lanes (backend/ahead.py: the tail loop's groups of 1 .. 64 lanes per item) give the
plain loop's results: per-item results and integer sums bitwise, exact sums bitwise, dropped emits and truncations
counted once per item."""
import numpy as np
import pytest

import tallymap_amd as tm
from tallymap_amd import configs, lax, problems, random
from tallymap_amd import numpy as jnp

import test_ahead

pytestmark = pytest.mark.gpu
# from one item (64 lanes) over the group sizes' edges to more items than a workgroup and than 2 workgroups per CU
SIZES = (1, 3, 4, 5, 16, 17, 64, 65, 129, 255, 257, 1000, 4099, 131_073)


def _pair(f_of, args_of, n):
    import torch
    args = args_of(n)
    a, b = f_of(dict())(*args), f_of(dict(compact=0))(*args)
    for x, y in zip(tm_leaves(a.per_item), tm_leaves(b.per_item)):
        assert torch.equal(x, y), n
    assert torch.equal(a.truncated, b.truncated)
    for k in a.stats:
        assert int(a.stats[k].item()) == int(b.stats[k].item()), (n, k)
    for k in a.outputs:
        assert torch.equal(a.outputs[k], b.outputs[k]), (n, k)


def tm_leaves(x):
    if x is None:
        return []
    return [z for y in x for z in tm_leaves(y)] if isinstance(x, (tuple, list)) else [x]


def _exact(outputs):
    return {k: tm.Sum(v.shape, fixed_point=True) for k, v in outputs.items()}


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("name", ["c1", "c2", "c3"])
def test_configs_match_the_plain_loop(name, n):
    cfg = getattr(configs, name.upper())
    if name != "c1" and n > 5000:
        n = 20_011
    print("case:", name, n, flush=True)
    _pair(lambda o: tm.vmap(cfg["item"], outputs=_exact(cfg["outputs"]), in_axes=cfg["in_axes"],
                            max_steps=cfg["max_steps"], **o), getattr(configs, name + "_inputs"), n)


@pytest.mark.parametrize("n", [1, 7, 64, 300, 5003])
@pytest.mark.parametrize("name", ["transport", "walk_on_spheres", "barrier", "gillespie", "random_walk"])
def test_problems_match_the_plain_loop(name, n):
    p = problems.PROBLEMS[name]
    print("case:", name, n, flush=True)
    _pair(lambda o: tm.vmap(p["item"], outputs=_exact(p["outputs"]), in_axes=p["in_axes"], **o),
          lambda n: p["inputs"](n)[0], n)


@pytest.mark.parametrize("opts", [dict(block=64), dict(block=192), dict(compact=1), dict(post_batch=64), dict(refill=5)],
                         ids=str)
def test_options_match_the_plain_loop(opts):
    for n in (1, 9, 100, 1000):
        print("case:", opts, n, flush=True)
        _pair(lambda o: tm.vmap(configs.c2_item, outputs=_exact(configs.C2["outputs"]), in_axes=(0, 0, None),
                                max_steps=65_536, **dict(opts, **o)), configs.c2_inputs, n)


def test_truncation_and_dropped_emits_are_counted_once():
    """a cap that falls inside a group's round, and bins past the tally's end."""
    def item(t, x, key):
        def body(c):
            k, x, t = c
            u = random.uniform(random.fold_in(key, k))
            t = t.add("n", (u * 10.0).astype(jnp.int32), np.int32(1))
            return k + 2, x * (0.9 + 0.1 * u), t
        k, x, t = lax.while_loop(lambda c: c[1] > 0.05, body, (np.int32(3), x, t))
        return t, (k, x)
    for cap in (5, 37, 1000):
        for n in (1, 50, 700):
            print("case: cap", cap, "n", n, flush=True)
            _pair(lambda o: tm.vmap(item, outputs={"n": tm.Sum((7,), dtype=np.int32)}, in_axes=(0, 0), max_steps=cap,
                                    **o),
                  lambda n: (np.linspace(0.1, 5.0, n).astype(np.float32), random.split(random.PRNGKey(1), n)), n)


@pytest.mark.parametrize("n", [1, 33, 900])
def test_taped_gradient_matches_the_plain_loop(n):
    """the tape adjoint's count launch (its tape rows written by one lane of a group)."""
    import torch
    args = configs.c1_inputs(n)
    w = np.linspace(0.5, 1.5, 16).astype(np.float32)
    got = []
    for o in (dict(), dict(compact=0)):
        f = tm.vmap(configs.c1_item, outputs=configs.C1["outputs"], in_axes=(0, 0, None), max_steps=100, **o)
        got.append(tm.grad(f, {"hist": w}, argnums=(0, 2))(*args))
    assert torch.equal(got[0][0], got[1][0])
    assert torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("n", [1, 5, 64, 300, 3000])
def test_spawning_program_matches_the_plain_loop(n):
    """the shower: the same tree (children spawned once per item, by one lane of its group), the same exact deposits."""
    import torch
    p = problems.PROBLEMS["shower"]
    args = p["inputs"](n)[0]
    got = [tm.vmap(p["item"], outputs=_exact(p["outputs"]), in_axes=p["in_axes"], spawn=tm.Queue(max(n, 64)), **o)(*args)
           for o in (dict(), dict(compact=0))]
    for k in got[0].stats:
        assert int(got[0].stats[k].item()) == int(got[1].stats[k].item()), k
    assert torch.equal(got[0].outputs["dep"], got[1].outputs["dep"])


def _host_steps(oracle, name, steps, x, keys):
    """test_ahead's items in numpy float32, step by step -> (steps, the final x) of each item."""
    f = np.float32
    out = []
    for i, x in enumerate(x):
        k, x = 0, f(x)
        while (k < steps) if name != "condition" else (np.ceil(-np.log2(x)) < 12):
            u = f(oracle.uniform(oracle.fold_in(keys[i], k)))
            if name == "condition":
                x = x * (f(0.5) + f(0.5) * u)
            else:
                trips = {"up": 20 - k, "shift": (20 - k).bit_length(), "branch": 0 if k % 2 else 20 - k,
                         "levels": 1 << k, "literal": 100}[name]
                v = u
                for _ in range(trips):
                    v = v * f(0.75) + u
                x = x * (f(0.5) + f(0.125) * u) + v
            k += 1
        out.append((k, x))
    return np.array([k for k, _ in out], np.int32), np.array([x for _, x in out], np.float32)


@pytest.mark.parametrize("name", list(test_ahead.LOOPS) + ["condition"])
def test_steps_with_loops_of_their_own(oracle, name):
    """loops that end for the steps an item takes and not for those after its last: the plain loop's results, and the
    host's for the first items."""
    steps = test_ahead.LOOPS.get(name)
    item = test_ahead.condition_item if name == "condition" else test_ahead.loop_item(name, steps)
    for n in (1, 6, 70, 700):
        print("case:", name, n, flush=True)
        _pair(lambda o: tm.vmap(item, outputs={"h": tm.Sum((4,), dtype=np.int32)}, in_axes=(0, 0), **o),
              test_ahead._walk_args, n)
    x, keys = test_ahead._walk_args(6)
    r = tm.vmap(item, outputs={"h": tm.Sum((4,), dtype=np.int32)}, in_axes=(0, 0))(x, keys)
    k, y = _host_steps(oracle, name, steps, x, keys)
    assert np.array_equal(r.per_item[0].cpu().numpy(), k)
    assert np.array_equal(r.per_item[1].cpu().numpy(), y)


@pytest.mark.parametrize("n", [1, 40, 1000, 9001])
def test_a_spread_launchs_float_sums_round_once(oracle, n):
    """the sums of up to 512 workgroups into a float32 bin: the float64 sum of the emitted values (each one of them
    representable, positive: float64's own roundings are far below) rounded once to float32, also for a constant, in
    a register-held, a float64 and a float32 LDS tally."""
    sizes = {"one": 1, "few": 5, "many": 1500}

    def item(t, key):
        def body(c):
            k, t = c
            u = random.uniform(random.fold_in(key, k), minval=0.25, maxval=1.75)
            for name, S in sizes.items():
                t = t.add(name, k % S, u)
            return k + 1, t.add("c", 0, 0.1)
        return lax.while_loop(lambda c: c[0] < 4, body, (np.int32(0), t))[1]
    keys = np.asarray(random.split(random.PRNGKey(5), n))
    r = tm.vmap(item, outputs={**{k: tm.Sum((S,)) for k, S in sizes.items()}, "c": tm.Sum((1,))}, in_axes=(0,))(keys)
    u = np.array([[oracle.uniform(oracle.fold_in(key, k), 0.25, 1.75) for k in range(4)] for key in keys], np.float64)
    want = {k: np.bincount(np.arange(4) % S, weights=u.sum(0), minlength=S) for k, S in sizes.items()}
    want["c"] = np.array([4 * n * float(np.float32(0.1))])
    for k, w in want.items():
        got = r.outputs[k].cpu().numpy().astype(np.float64)
        # (the float32 LDS bins: a rounding per add within a workgroup, at most 16 items' there)
        slack = 2.0 ** -24 * (16 if k == "many" else 1) + 1e-12
        assert np.all(np.abs(got - w) <= slack * w), (n, k, got[:5], w[:5])
