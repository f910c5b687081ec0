"""tm_launch_noalloc against tm_launch through the C ABI: the same program, the same inputs, the scratch buffers
(exact words, counters) in the library's per-device array instead of caller allocations.  Outputs must be bitwise
equal -- exact tallies are order independent, trip counts and flags are integers -- on two calls in a row, the
second with fewer items (the array keeps the first call's contents: tm_zero must clear what has to start at zero).
After its first call on a device (module load, array address resolved) the entry allocates nothing: device free
memory is unchanged across a call made directly through ctypes on preallocated outputs.  The file's name sorts
last, so `pytest -m gpu` runs it after every other test; it must also pass on its own in a fresh process
(`pytest tests/test_zz_no_alloc.py`)."""
import ctypes

import numpy as np
import pytest

from tallymap_amd import _core as CO
from tallymap_amd import backend as B
from tallymap_amd import configs
from tallymap_amd._api import Sum, build_program
from tallymap_amd.backend import compile as Cm

pytestmark = pytest.mark.gpu


def _prog(cfg, args, exact):
    outs = {k: Sum(v.shape, fixed_point=True) if exact else v for k, v in cfg["outputs"].items()}
    axes = cfg["in_axes"]
    pav = [CO.AVal(np.shape(a)[1:], np.asarray(a).dtype) for a, x in zip(args, axes) if x == 0]
    bav = [CO.AVal(np.shape(a), np.asarray(a).dtype) for a, x in zip(args, axes) if x is None]
    return build_program(cfg["item"], outs, axes, pav, bav, cfg["max_steps"])[0]


def _ins(args, axes):
    pi = [B.device_tensor(a, np.asarray(a).dtype) for a, x in zip(args, axes) if x == 0]
    bc = [B.device_tensor(a, np.asarray(a).dtype) for a, x in zip(args, axes) if x is None]
    return pi + bc


def _pair(c, args, axes, N):
    import torch
    ins = _ins(args, axes)
    ref = B.launch(c, ins, N)
    got = B.launch_noalloc(c, ins, N)
    torch.cuda.synchronize()
    scr = set(c.layout.scratch)
    n = 0
    for j, (r, g) in enumerate(zip(ref, got)):
        if c.layout.n_in + j in scr:
            assert g is None
            continue
        assert g is not None
        a, b = r.cpu().numpy(), g.cpu().numpy()
        assert a.shape == b.shape
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), f"result {j} differs"
        n += 1
    return n


@pytest.mark.parametrize("name,n1,n2", [("c1", 10_000, 3_000), ("c3", 65_536, 8_192)])
def test_noalloc_matches_tm_launch(name, n1, n2):
    cfg = getattr(configs, name.upper())
    args = getattr(configs, f"{name}_inputs")(n1)
    prog = _prog(cfg, args, exact=True)
    c = B.compiled(prog, {})
    assert c.layout.scratch
    for N in (n1, n2):
        print(f"case: {name} exact tallies, N={N}: tm_launch vs tm_launch_noalloc", flush=True)
        a = [np.asarray(x)[:N] if ax == 0 else x for x, ax in zip(args, cfg["in_axes"])]
        assert _pair(c, a, cfg["in_axes"], N) >= 3


def test_noalloc_refuses_oversized_scratch():
    import torch
    cfg = configs.C1
    args = configs.c1_inputs(1024)
    c = B.compiled(_prog(cfg, args, exact=True), {})
    ins = _ins(args, cfg["in_axes"])
    outs = B._alloc(c, 1024)
    bufs = [t.data_ptr() for t in ins] + [t.data_ptr() for t in outs]
    arr = (ctypes.c_void_p * len(bufs))(*bufs)
    sl = (ctypes.c_int * 1)(c.layout.scratch[0])
    nb = (ctypes.c_longlong * 1)((32 << 20) + 1)
    lib = Cm.lib()
    rc = lib.tm_launch_noalloc(c.id, None, arr, len(bufs), sl, nb, 1, c.layout.n_zero, c.layout.flags, 1024,
                               c.block)
    assert rc != 0 and b"no-alloc array" in lib.tm_last_error()
    torch.cuda.synchronize()


def test_noalloc_allocates_nothing_after_the_first_call():
    """the entry point itself, through ctypes, on outputs allocated beforehand: a warm-up call, then a call across
    which the device's free memory (hipMemGetInfo) does not move and whose outputs equal the warm-up's bitwise."""
    import torch
    cfg = configs.C1
    N = 10_000
    args = configs.c1_inputs(N)
    c = B.compiled(_prog(cfg, args, exact=True), {})
    L = c.layout
    ins = _ins(args, cfg["in_axes"])
    outs = B._alloc(c, N)
    scr = list(L.scratch)
    nbytes = [outs[r - L.n_in].numel() * outs[r - L.n_in].element_size() for r in scr]
    bufs = [t.data_ptr() for t in ins] + [0 if (L.n_in + j) in scr else t.data_ptr() for j, t in enumerate(outs)]
    arr = (ctypes.c_void_p * len(bufs))(*bufs)
    sl = (ctypes.c_int * len(scr))(*scr)
    nb = (ctypes.c_longlong * len(scr))(*nbytes)
    lib = Cm.lib()
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)

    def call():
        rc = lib.tm_launch_noalloc(c.id, s, arr, len(bufs), sl, nb, len(scr), L.n_zero, L.flags, N, c.block)
        assert rc == 0, lib.tm_last_error()
        torch.cuda.synchronize()
        return [outs[r - L.n_in].cpu().numpy().copy() for r in list(L.r_out.values()) + list(L.r_ys)]
    print("case: C1 exact tallies, N=10000: tm_launch_noalloc allocation check", flush=True)
    first = call()
    free0 = torch.cuda.mem_get_info()[0]
    second = call()
    free1 = torch.cuda.mem_get_info()[0]
    assert free1 == free0, (free0, free1)
    for a, b in zip(first, second):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8))


@pytest.mark.parametrize("name, flags", [("c1", 2), ("random_walk", 8)])
def test_noalloc_plain_sums_in_a_graph(name, flags):
    """plain float32 sums of a spread launch (its float64 sums are in a ctl of the caller's, read by tm_post: of the
    program's own, or launched for them alone) and of one that does not spread, captured and replayed with eager work
    between the replays: the eager launch's results."""
    import torch

    from tallymap_amd import problems
    cfg = configs.C1 if name == "c1" else dict(problems.PROBLEMS[name], max_steps=None)
    N = 400_000
    args = configs.c1_inputs(N) if name == "c1" else cfg["inputs"](N)[0]
    c = B.compiled(_prog(cfg, args, exact=False), {})
    L = c.layout
    assert L.flags == flags and L.spread > 0 and L.r_ctl not in L.scratch
    for n in (3_000, N):
        print("case:", name, n, flush=True)
        ins = _ins([np.asarray(a)[:n] if ax == 0 else a for a, ax in zip(args, cfg["in_axes"])], cfg["in_axes"])
        ref = B.launch(c, ins, n)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            got = B.launch_noalloc(c, ins, n)
        for _ in range(3):
            g.replay()
            torch.cuda.synchronize()
            for r in L.r_out.values():
                a, b = got[r - L.n_in].double(), ref[r - L.n_in].double()
                assert bool((b > 0).any()) and torch.allclose(a, b, rtol=2e-6, atol=0.0), (n, a, b)
            for r in L.r_ys:
                assert torch.equal(got[r - L.n_in], ref[r - L.n_in]), n
            B.launch(c, ins, n)
            torch.cuda.synchronize()
