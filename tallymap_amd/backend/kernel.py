"""One HIP module per item program: tm_zero, tm_main (the persistent item loop) and tm_post (readout / poison).

Buffers (one by-value struct of pointers, TmParams; the item count is a kernel argument, so one code object serves
every N):
    inputs  [per-item operands][broadcast operands]
    results [sum tallies][exact scratch of each exact tally][ctl u32][stats i32[5]] | [per-item results]
The first group of results (up to stats) is zeroed by tm_zero before tm_main runs: the reference's n_zero
(reference backends/kernel/kernel.py:565-591, shim.cc:215-218).  ctl holds the count of truncated items
(word 2), the claim counters of the item ranges and, where steps are computed ahead, float64 sums of the privatised
float32 tallies, which tm_post rounds into them.

tm_main is the hand-written CDNA4 loop (reference kernel.py:812-838 is the CUDA one it replaces):
  * a persistent grid (256 CUs x achieved occupancy), block BLOCK = 256 (4 wave64s);
  * step-granular refill (the reference's schedule='step', kernel.py:239-295, 469-563): each loop iteration, the
    lanes of a wave whose item has finished are counted with one ballot and take the next items of the chunk the
    wave holds (mbcnt gives each idle lane its rank); a chunk is claimed with one atomic on the counter of an item
    range, of which there are 64.  A lane then runs its item's `pre`, and every live lane runs one (cond, body)
    step or, when the predicate fails, `post` and writes its per-item results.  A lane never waits for its wave's
    longest item; lanes left without an item compute the draws of other lanes' coming steps (backend/ahead.py);
  * small tallies privatised in LDS (up to LDS_BYTES per block), flushed once at exit with device atomics;
    larger ones take the global atomic directly;
  * dropped emits and truncations counted in registers, one atomic per lane at exit.
Programs without exactly one top-level while loop run the item schedule (a lane runs its whole item per claim).
"""
import dataclasses
import re

import numpy as np

from .. import _core as C
from .codegen import Emitter, Val, VTally, assign_carries, ctype, lit
from . import ahead as Ahead
from . import simplify

BLOCK = 256
LDS_BYTES = 32768          # privatised tallies per block (MI355X: 160 KB LDS per CU)
LDS_F64 = 8192             # of those, float32 sums held as float64 in LDS take up to this many bytes (8 per bin):
                           # ds_add_f64 runs ~8x faster than ds_add_f32 on gfx950 (a wave64 add occupies a CU's LDS
                           # for ~6 cycles against 194 -- 2,048 workgroups x 256 x 512 adds onto 64 random bins:
                           # 0.167 ms, 0.13 of it the address arithmetic, against 1.335 -- whatever the bins and
                           # conflicts), and a float32 value or a sum of them is never a float64 subnormal, so the
                           # compare-and-swap path of tm_ladd_f32 goes too.  Larger tallies keep float32: at 8 bytes a
                           # 4,096-bin map takes a workgroup per CU from the loop, and there the adds are not the bound
LDS_MAX = 160 << 10        # bytes of LDS a workgroup may have (gfx950)
LDS_COPIES = 256           # a float64 or count bin of a tally of S bins has up to 16 copies in LDS, S x copies at most
                           # this (8-byte words); a lane adds to copy lane % copies and the flush sums them.  Lanes of
                           # a wave that add to one address take turns: ds_add_f64 cycles per wave64 add and CU (the
                           # probe above, ~18 of them address arithmetic) 392 onto one bin, 111 onto 2, 45 onto 8, 31
                           # onto 16, 24 onto 64; with 16 copies 18-19 onto 1, 8 or 16 bins, with 4 copies 21 onto 64.
                           # All copies of a program together take at most LDS_F64 bytes: an unrolled loop over a
                           # table of 84 weights is 84 counters of 16 bins, 11 KB at one copy and 170 at 16
REG_BINS = 2               # privatised tallies of at most this many bins accumulate in each lane's registers
XW = 9                     # int64 words per exact bin (tm_device.h TM_XW: weights 2^(32 j))
CHUNK = 64
RESERVE = 4                # chunks a wave reserves per claim while far from the end (short items)
CLAIM_NS = 20_000          # reserve when a chunk lasted less than this many ns
SHARDS = 64                # item ranges with a claim counter each (one per lane of the wave that looks for items left)
SHARD0 = 64                # ctl word of the first range's counter (u64), SHARD_WORDS words apart (256 bytes)
SHARD_WORDS = 64
IL_CHUNKS = 4              # chunks of a block, where the ranges are blocks dealt out in turn (tape programs)
RC_WORDS = SHARDS * SHARD_WORDS + 64    # u32 words of a Records output's counters: a u64 of slots claimed per segment of
                           # its raw slots (SHARD_WORDS apart), then (u64) the records appended and the launch's waves
RC_TOTAL = SHARDS * SHARD_WORDS // 2    # u64 index of the records appended among them
RB = 256                   # slots per Records batch (TM_RB in tm_device.h)
SPREAD = 16                # lanes per item a small launch of a program with steps computed ahead spreads to (the
                           # launcher's grid, the module's tm_spread)
COMPACT = 16               # iterations between the tail-phase repacks of a workgroup's live items
POST_BATCH = 2.0           # finished items wait for their POST until the wave's waiting lane-iterations reach this
                           # many times the (POST + refill) / step cost ratio x 64 (0: each item's POST at once) ...
POST_BATCH_MIN = 25        # ... when that wait is at least this long: below it the wave's per-step bookkeeping costs
                           # more than the shared passes save.  Measured: at 1.0 and 24, C2's 11 ran 2.5 % slower
                           # batched and C4's 37-42 16-20 % faster; at 2.0 the transport problem's 30 / 34 ran
                           # 12 % faster, C2's fused 24 0.5 % slower (so 25)
BCAST_REG = 16             # broadcast operands up to this many elements are loaded into registers
TABLE_MAX = 16384          # bytes: a larger broadcast array read by the item is copied into LDS once per workgroup
SPAWN_BLOCKS = 2           # workgroups per CU of a spawning program's item loop (the launcher's grid cap): the
                           # shower forward ran 9.18 / 9.07 / 8.92 / 8.66 / 8.38 / 8.26 / 8.02 ms at 8 / 7 / 6 / 5 /
                           # 4 / 3 / 2 per CU
LDS_TABLES = 0             # bytes of such tables per workgroup (the build option lds_tables; 0: none).  Off by
                           # default: staging C3's 16 KB cotangent table took its reverse launch from 4 to 3
                           # workgroups per CU and from 0.66 to 0.72 ms (a per-step L2 read was not its bound)


@dataclasses.dataclass
class Layout:
    n_in: int
    res: list              # (shape, dtype, per_item) per result buffer
    n_zero: int
    r_out: dict            # tally slot -> result index (absolute buffer index)
    r_ctl: int
    r_stats: int
    r_ys: list
    flags: int             # bit 1: launch tm_post; bit 3: launch it where the launch spread
    mode: str
    priv: list
    zero_words: list       # (buffer index, u32 words) zeroed by tm_zero
    records: list = dataclasses.field(default_factory=list)
    # per Records output: dict(name, capacity, r_ctr (its u64 record count: result index, word), fields {suffix:
    # canonical result index}), and aux: the passes (entry name, grid kind, block) run after tm_launch
    aux: list = dataclasses.field(default_factory=list)
    # spawn: the next generation's per-item operand buffers (result indices, one per per-item operand, Q rows)
    r_q: list = dataclasses.field(default_factory=list)
    # the buffers only the kernels read (exact / fixed-point words, ctl without float64 sums): what tm_launch_noalloc
    # may place itself
    scratch: list = dataclasses.field(default_factory=list)
    # u32 words of ctl up to the end of its claim counters (0: a program without them); float64 sums may follow
    n_claim: int = 0
    spread: int = 0        # the module's tm_spread (0: its launches do not spread)
    emitted: set = dataclasses.field(default_factory=set)      # the tally slots with an emit


def _split(jx):
    """-> (index of the only top-level while eqn that is not a static loop) or None.  A static-bound fori_loop or
    long scan (equation param static=True) is ordinary straight-line work of its step, as a scan is in JAX."""
    ws = [i for i, e in enumerate(jx.eqns) if e.prim == "while" and not e.params.get("static", False)]
    return ws[0] if len(ws) == 1 else None


def _staged_tables(jx, b0, bav, budget):
    """broadcast operand indices to copy into LDS (see build's lds_tables): arrays above BCAST_REG elements and at
    most TABLE_MAX bytes that the item reads, most-referenced first while the total fits `budget` bytes."""
    if budget <= 0:
        return []
    ids = {v.id: i for i, v in enumerate(jx.invars[b0:b0 + len(bav)])}
    refs = {}
    for e in C.walk_eqns(jx):
        for v in e.invars:
            if isinstance(v, C.Var) and v.id in ids:
                refs[ids[v.id]] = refs.get(ids[v.id], 0) + 1
    out = []
    for i in sorted(refs, key=lambda j: (-refs[j], j)):
        a = bav[i]
        nb = a.size * a.dtype.itemsize
        if a.size > BCAST_REG and nb <= TABLE_MAX and nb <= budget:
            out.append(i)
            budget -= nb
    return sorted(out)


def _used_vars(eqns, outvars):
    s = set()
    for e in eqns:
        for v in e.invars:
            if isinstance(v, C.Var):
                s.add(v.id)
        for sub in C.subjaxprs(e):
            s |= _free_vars(sub)
    for v in outvars:
        if isinstance(v, C.Var):
            s.add(v.id)
    return s


def _free_vars(jx):
    defined = {v.id for v in jx.invars}
    free = set()
    for e in jx.eqns:
        for v in e.invars:
            if isinstance(v, C.Var) and v.id not in defined:
                free.add(v.id)
        for o in e.outvars:
            defined.add(o.id)
    return free


_HEAVY = {"exp", "log", "sin", "cos", "tan", "atan", "atan2", "asin", "acos", "sinh", "cosh", "tanh", "asinh", "acosh",
          "atanh", "log1p", "expm1", "exp2", "log2", "pow", "erf", "erfc", "erf_inv", "lgamma", "cbrt", "logistic", "tallymap_sincos"}
_FREE = {"slice", "squeeze", "reshape", "broadcast_in_dim", "concatenate", "copy", "stop_gradient"}


def cost(eqns, loop=4):
    """a rough count of the VALU instructions one evaluation of `eqns` issues (static weights: a libm call 30, the
    threefry2x32 hash 72 per pair, a division or square root 8, an effect 6, other element operations 1; a nested
    loop counts `loop` trips; a cond its costliest branch that is not marked cold).  It sets how long finished items wait for their POST (build's post_batch)."""
    c = 0
    for e in eqns:
        n = max([1] + [max(1, o.aval.size) for o in e.outvars])
        p = e.prim
        if p == "while":
            c += loop * (cost(e.params["cond_jaxpr"].eqns, loop) + cost(e.params["body_jaxpr"].eqns, loop))
        elif p == "cond":          # (a branch marked cold -- rarely taken -- is left out)
            cold = set(e.params.get("cold", ()))
            brs = [b for i, b in enumerate(e.params["branches"]) if i not in cold] or list(e.params["branches"])
            c += 2 + max(cost(b.eqns, loop) for b in brs)
        elif p in _HEAVY:
            c += 30 * n * len(e.outvars)
        elif p == "threefry2x32":
            c += 72 * n
        elif p in ("div", "rem", "sqrt", "rsqrt"):
            c += 8 * n
        elif p.startswith("tallymap_"):
            c += 6
        elif p not in _FREE:
            c += n
    return c


def _records_passes(ri, r_rctr, r_out, r_cnt, r_rex, r_rbs, prog, bad):
    """the passes that move Records output j's raw records to their canonical slots (replacing the reference's
    _records.canon, _records.py:45-74): tm_rscan<j> (blocks of 1024 items: the exclusive prefix sum of the per-item counts within the block, and the
    block's total), tm_rtop<j> (one block: the exclusive prefix sum of the block totals), tm_rcanon<j> (every claimed
    raw slot with a key: record (i, k) to slot offset[i] + k; the slots past the last record zeroed; when `bad` -- a
    truncation or any Records output past its capacity (reference _api.py:745-755) -- every float field NaN and
    every integer field -1 instead)."""
    j, cap = ri["ctr"], ri["capacity"]
    cnt, rex, rbs = f"((const i32*)P.p[{r_cnt}])", f"((i64*)P.p[{r_rex}])", f"((i64*)P.p[{r_rbs}])"
    rc, S = f"((const u64*)P.p[{r_rctr}] + {RC_WORDS // 2 * j})", ri["segments"]
    nb = f"({-(-cap // RB)}ull + {rc}[{RC_TOTAL + 1}])"          # (raw_segment_slots, with the launch's waves)
    seg = (f"{cap}ull + {rc}[{RC_TOTAL + 1}] * {RB - 1}ull" if S == 1 else f"({nb} + {S - 1}ull) / {S}ull * {RB}ull")
    ki, kk = f"((i32*)P.p[{r_out[ri['ki']]}])", f"((const i32*)P.p[{r_out[ri['kk']]}])"
    scan = ("  for (int d = 1; d < 1024; d <<= 1) {\n"
            "    const i64 x = (int)threadIdx.x >= d ? tm_s[threadIdx.x - d] : 0;\n"
            "    __syncthreads();\n"
            "    tm_s[threadIdx.x] += x;\n"
            "    __syncthreads();\n"
            "  }\n")
    out = []
    out.append(f"extern \"C\" __global__ void __launch_bounds__(1024) tm_rscan{j}(const TmParams P, const i64 n_items) {{\n"
               "  __shared__ i64 tm_s[1024];\n"
               "  const i64 i = (i64)blockIdx.x * 1024 + threadIdx.x;\n"
               f"  const i64 c = i < n_items ? (i64){cnt}[i] : 0;\n"
               "  tm_s[threadIdx.x] = c;\n"
               "  __syncthreads();\n" + scan +
               f"  if (i < n_items) {rex}[i] = tm_s[threadIdx.x] - c;\n"
               f"  if (threadIdx.x == 1023) {rbs}[blockIdx.x] = tm_s[1023];\n}}")
    out.append(f"extern \"C\" __global__ void __launch_bounds__(1024) tm_rtop{j}(const TmParams P, const i64 n_items) {{\n"
               "  __shared__ i64 tm_s[1024];\n"
               "  const i64 nb = (n_items + 1023) / 1024;\n"
               "  i64 carry = 0;\n"
               "  for (i64 base = 0; base < nb; base += 1024) {\n"
               "    const i64 i = base + threadIdx.x;\n"
               f"    const i64 v = i < nb ? {rbs}[i] : 0;\n"
               "    tm_s[threadIdx.x] = v;\n"
               "    __syncthreads();\n" + scan.replace("\n  ", "\n    ").replace("  for", "    for", 1) +
               f"    if (i < nb) {rbs}[i] = carry + tm_s[threadIdx.x] - v;\n"
               "    carry += tm_s[1023];\n"
               "    __syncthreads();\n"
               "  }\n}")
    mv, fill, zero = [], [], []
    for f, (k, rr) in ri["fields"].items():
        ct = ctype(prog.tallies[k].dtype)
        mv.append(f"(({ct}*)P.p[{rr}])[dst] = ((const {ct}*)P.p[{r_out[k]}])[s];")
        zero.append(f"(({ct}*)P.p[{rr}])[s] = ({ct})0;")
        if prog.tallies[k].dtype in (C.F32, C.F64):
            fill.append(f"(({ct}*)P.p[{rr}])[s] = ({ct})__builtin_nan(\"\");")
        else:
            fill.append(f"(({ct}*)P.p[{rr}])[s] = ({ct})-1;")
    out.append(f"extern \"C\" __global__ void __launch_bounds__(256) tm_rcanon{j}(const TmParams P, const i64 n_items) {{\n"
               "  const i64 g = (i64)blockIdx.x * blockDim.x + threadIdx.x, st = (i64)gridDim.x * blockDim.x;\n"
               f"  if ({bad}) {{\n"
               f"    for (i64 s = g; s < {cap}; s += st) {{ {' '.join(fill)} }}\n"
               "    return;\n"
               "  }\n"
               f"  const i64 ntot = (i64){rc}[{RC_TOTAL}], seg = (i64)({seg});\n"
               # a segment's slots go to the workgroups of its index modulo the segments: on MI355X a workgroup's XCD is
               # its index % 8, the XCD whose waves wrote the segment and whose items' records it mostly holds
               f"  for (i64 q = blockIdx.x % {S}; q < {S}; q += gridDim.x) {{\n"
               f"    const i64 parts = gridDim.x >= {S}u ? (i64)((gridDim.x - q + {S - 1}) / {S}) : 1;\n"
               f"    const i64 part = gridDim.x >= {S}u ? (i64)(blockIdx.x / {S}u) : 0;\n"
               f"    const i64 n = (i64){rc}[q * {SHARD_WORDS // 2}] < seg ? (i64){rc}[q * {SHARD_WORDS // 2}] : seg;\n"
               "    for (i64 i = part * 256 + threadIdx.x; i < n; i += parts * 256) {\n"
               "      const i64 s = q * seg + i;\n"
               f"      const i32 key = {ki}[s];\n"
               "      if (key <= 0 || (i64)key > n_items) continue;\n"
               f"      const i32 cid = key - 1, k = {kk}[s];\n"
               f"      const i64 dst = {rex}[cid] + {rbs}[cid >> 10] + k;\n"
               f"      if (dst < 0 || dst >= {cap}) continue;\n"
               f"      {' '.join(mv)}\n"
               "    }\n"
               "  }\n"
               f"  for (i64 s = ntot + g; s < {cap}; s += st) {{ {' '.join(zero)} }}\n"
               "}")
    return "\n".join(out)


def raw_segments(capacity, direct):
    """segments a Records output's raw slots are split into, each with its own slot counter (1: the claims are of other
    sizes than a batch, or the slots come near 2^31)."""
    return 1 if direct or capacity > 2 ** 30 else SHARDS


def raw_segment_slots(capacity, waves, S):
    """the raw slots of a segment, for a launch of `waves` waves: room for every record of the capacity and one partly
    used batch per wave, in whole batches per segment."""
    if S == 1:
        return capacity + waves * (RB - 1)
    return RB * -(-(-(-capacity // RB) + waves) // S)


def exact_words(S):
    """u32 words of an exact tally's scratch: XW int64 words per bin, then one flag bit per bin."""
    return 2 * XW * S + (S + 31) // 32


def wide_words(S):
    """u32 words of a scaled fixed-point tally's scratch: per bin a u64 low word, then an i32 carry word per bin,
    then a u32 flag per bin (reference kernel.py:952-956)."""
    return 4 * S


def scratch_words(s):
    return exact_words(s.S) if s.exact else wide_words(s.S)


_IRANGE = {"int32": ("-2147483648.0", "2147483648.0", "tm_d2i32"), "uint32": ("0.0", "4294967296.0", "tm_d2u32"),
           "int64": ("-9223372036854775808.0", "9223372036854775808.0", "tm_d2i64"),
           "uint64": ("0.0", "18446744073709551616.0", "tm_d2u64")}


def _wide_readout(s, lo, cw, fl, out):
    """tm_post's readout of a scaled fixed-point tally (reference kernel.py:652-664): the exact total rounded once
    to double, times 1/scale, in the output dtype.  A total that does not fit is counted in fixed_point_overflow
    (unless the bin is already flagged); a float bin is NaN when flagged or too big, an integer one saturates."""
    v = f"tm_wide_f64({lo}[i], {cw}[i]) * {lit(1.0 / s.scale, np.float64)}"
    if s.dtype == C.F64:
        return (f"for (i64 i = g; i < {s.S}; i += st) {{ const double v = {v}; "
                f"const bool big = !(__builtin_fabs(v) <= 1.7976931348623157e308); "
                f"if (big && !{fl}[i]) atomicAdd(&TM_STATS[3], 1); "
                f"((double*){out})[i] = ({fl}[i] || big) ? __builtin_nan(\"\") : v; }}")
    lo_, hi_, cv = _IRANGE[s.dtype.name]
    ct = ctype(s.dtype)
    return (f"for (i64 i = g; i < {s.S}; i += st) {{ const double v = {v}; "
            f"if (!(v >= {lo_} && v < {hi_})) atomicAdd(&TM_STATS[3], 1); (({ct}*){out})[i] = ({ct}){cv}(v); }}")


_W64 = {"i64", "u64", "double"}


def _repack_code(decls, cap):
    """(pack lines, unpack lines, words per item) moving one item's loop state -- the declared carries and
    persistent values, and tm_item -- through the LDS pool tm_pool (column w of word w, row q)."""
    fields = []
    for d in decls:
        ct, nm = d.strip().rstrip(";").split()
        fields.append((ct, nm))
    fields.append(("i64", "tm_item"))
    pack, unpack = [], []
    w = 0
    for ct, nm in fields:
        if ct in _W64:
            pack.append(f"{{ const u64 b = __builtin_bit_cast(u64, {nm}); tm_pool[{w * cap}u + q] = (u32)b; "
                        f"tm_pool[{(w + 1) * cap}u + q] = (u32)(b >> 32); }}")
            unpack.append(f"{nm} = __builtin_bit_cast({ct}, (u64)tm_pool[{w * cap}u + q] | "
                          f"((u64)tm_pool[{(w + 1) * cap}u + q] << 32));")
            w += 2
        elif ct == "bool":
            pack.append(f"tm_pool[{w * cap}u + q] = (u32){nm};")
            unpack.append(f"{nm} = tm_pool[{w * cap}u + q] != 0u;")
            w += 1
        elif ct in ("float", "u32", "i32"):
            pack.append(f"tm_pool[{w * cap}u + q] = __builtin_bit_cast(u32, {nm});")
            unpack.append(f"{nm} = __builtin_bit_cast({ct}, tm_pool[{w * cap}u + q]);")
            w += 1
        else:                                      # 8- and 16-bit integers
            pack.append(f"tm_pool[{w * cap}u + q] = (u32){nm};")
            unpack.append(f"{nm} = ({ct})tm_pool[{w * cap}u + q];")
            w += 1
    return pack, unpack, w


def lds_bytes(src):
    """the bytes of the __shared__ arrays and scalars that `src` declares (one declaration a line)."""
    size = {"double": 8, "float": 4, "bool": 1}
    n = 0
    for ct, names in re.findall(r"__shared__ (\w+) ([^;]*);", src):
        b = size.get(ct) or int(ct[1:]) // 8
        for nm in names.split(","):
            m = re.search(r"\[(\d+)\]", nm)
            n += b * (int(m.group(1)) if m else 1)
    return n


def tally_lds_bytes(s):
    """the LDS bytes a privatised copy of tally spec s takes (exact: XW int64 words per bin; fixed point: an int64
    word, an int32 carry word; else the dtype's size): the kernel privatises tallies in slot order while their
    bytes fit LDS_BYTES."""
    return s.S * (8 * XW if s.exact else (12 if s.fixed else np.dtype(s.dtype).itemsize))


def build(prog, block=BLOCK, schedule="step", refill=1, chunk=CHUNK, compact=COMPACT, min_blocks=0,
          post_batch=POST_BATCH, lds_tables=LDS_TABLES, grid_cap=0, lean=False):
    """-> (HIP source, Layout) of prog's module.  chunk: items a wave claims with one atomic (their per-item operands
    are staged in LDS by one coalesced load, and idle lanes take them from there at step granularity).  compact:
    once every wave of a workgroup has drained the item queue, the waves meet every `compact` iterations and
    repack their live items densely onto the first waves (0: off; step schedule only).  min_blocks: workgroups per
    CU the compiler must leave registers for (as waves per SIMD in __launch_bounds__; 0: its own choice).
    post_batch (step schedule): an item whose loop condition fails waits, its lane idle, until the wave's waiting
    lane-iterations reach post_batch x 64 x (the POST's + a refill's cost) / (a step's cost), and then every
    waiting lane runs its POST at once and is refilled together: lanes that finish at different steps then
    share one pass through POST and the refill, where each finishing step cost the whole wave both.  With the
    queue drained, waiting items run their POST in the step they finish (0, or a wait below POST_BATCH_MIN:
    always so).
    lds_tables: bytes of broadcast tables (arrays above BCAST_REG elements, at most TABLE_MAX bytes each, that the
    item reads -- a cotangent tally read at a data-dependent bin in a reverse launch, a lookup table) copied into
    LDS at the workgroup's start, most-referenced first: every read of them, static or at a runtime index, is then
    an LDS load instead of a dependent global (L2) load in the step.  0: none.
    grid_cap: at most this many workgroups per CU in the item loop's persistent grid (the module's tm_grid_cap,
    which the launcher reads when it loads the module and takes as the occupancy when lower); 0: the occupancy.
    Fewer resident waves give each lane more items (a shorter tail) and a spawning loop's waves fewer concurrent
    claims and queue flushes, at the cost of latency hiding.
    lean: no copies of LDS bins and no float64 ones: what a program whose LDS would pass LDS_MAX with them is built
    as."""
    opts = dict(block=block, schedule=schedule, refill=refill, chunk=chunk, compact=compact, min_blocks=min_blocks,
                post_batch=post_batch, lds_tables=lds_tables, grid_cap=grid_cap)
    chunk = max(1, int(chunk))
    compact = max(0, int(compact))
    jx = simplify.drop_draw_clamp(prog.jaxpr)
    jx = simplify.cse(jx, _split(jx))
    jx = simplify.pair_sincos(jx, _split(jx))
    nT, nP, nB = prog.nT, prog.nP, prog.nB
    pav, bav = prog.p_avals(), prog.b_avals()
    yav = prog.y_avals()
    n_in = nP + nB
    res = []

    def result(shape, dt, per_item=False):
        res.append((tuple(shape), np.dtype(dt), per_item))
        return n_in + len(res) - 1
    outs = prog.out_tallies
    from .._tally import KI, KK, rkey
    raw = set()                # the Records outputs' raw tallies: sized per launch (capacity + the waves' batch
    for rn, _, _ in (getattr(prog, "records", ()) or ()):     # slack), never zeroed, stored to once per slot
        raw |= {k for k in outs if prog.tallies[k].name.startswith(rkey(rn, ""))}
    # appends inside a cond claim slots one point at a time (tm_rclaim_direct): such an output keeps one segment
    segs = {}
    for j, (rn, cap, _) in enumerate(getattr(prog, "records", ()) or ()):
        direct = any(x.prim == "tallymap_claim" and int(x.params["r"]) == j for e in C.walk_eqns(jx) if e.prim == "cond"
                     for b in C.subjaxprs(e) for x in C.walk_eqns(b))
        segs[rn] = raw_segments(int(cap), direct)

    def raw_of(k):
        """the Records output whose raw tally k is."""
        return next(rn for rn in segs if prog.tallies[k].name.startswith(rkey(rn, "")))
    r_out = {k: result(prog.tallies[k].shape, prog.tallies[k].dtype, ("rraw", segs[raw_of(k)]) if k in raw else False)
             for k in outs}
    r_scr = {k: result((scratch_words(prog.tallies[k]),), np.uint32) for k in outs
             if prog.tallies[k].exact or prog.tallies[k].fixed}
    recs = list(getattr(prog, "records", ()) or ())
    r_rctr = result((RC_WORDS * len(recs),), np.uint32) if recs else None
    rec_info = []
    for j, (rn, cap, _) in enumerate(recs):
        pre, keys = rkey(rn, ""), (rkey(rn, KI), rkey(rn, KK))
        fl = {}
        for k in outs:
            nm = prog.tallies[k].name
            if nm.startswith(pre) and nm not in keys:
                fl[nm[len(pre):]] = (k, result((cap,), prog.tallies[k].dtype))
        ks = [k for k in outs if prog.tallies[k].name in keys]
        rec_info.append(dict(name=rn, capacity=cap, ctr=j, fields=fl, ki=ks[0], kk=ks[1], count=prog.counts[j],
                             segments=segs[rn]))
    Q = getattr(prog, "spawn", None)
    # ctl: truncations (word 2), the claim counters of the item ranges (from word SHARD0); a spawning program's ticket counter sits at
    # words 32-33, on its own 128-byte line (two counters that every wave hits serialise on a shared line), and
    # tm_qnext's generation state after it: the next generation's item count (words 40-41), children spawned and
    # dropped so far (42-43, 44-45), the roots' truncations (word 48)
    n_ctl = SHARD0 + SHARDS * SHARD_WORDS
    r_ctl = result((n_ctl,), np.uint32)
    r_stats = result((5,), np.int32)
    n_zero = len(res)
    r_ys = [result(a.shape, a.dtype, per_item=True) for a in yav]
    # the queue's columns: the child's per-item operands, then (recording forward of the tree adjoint) its parent
    # (the item index) and its ordinal among the parent's children
    qav = list(pav) + ([C.AVal((), C.I32)] * 2 if getattr(prog, "spawn_mode", None) == "record" else [])
    r_q = [result((Q,) + tuple(a.shape), a.dtype) for a in qav] if Q is not None else []
    q_words, q_off = 0, []     # a child's operands as u32 words (the LDS staging layout)
    for a in qav:
        q_off.append(q_words)
        q_words += max(1, a.size) * (2 if a.dtype.itemsize == 8 else 1)
    # children staged per wave in LDS and flushed with one ticket claim per QS children (0: a claim per spawn point)
    QS = (128 if q_words <= 16 else 64 if q_words <= 48 else 0) if Q is not None else 0
    r_rex = result((), np.int64, per_item=True) if recs else None       # the Records scans' scratch (per item)
    r_rbs = result((), np.int64, per_item=True) if recs else None
    # the tape adjoint's programs (backend/tape.py): a u32 buffer of N x cap x Wp words (cap: an operand), written
    # by the count program's tape puts and read by the reverse program's gets; the caller allocates it
    tape_w = int(getattr(prog, "tape_words", 0) or 0)
    tape_ck = int(getattr(prog, "tape_ck_words", 0) or 0)     # (the residual tape's checkpoint after the slots)
    r_tape = result((tape_w,), np.uint32, per_item=("itape",)) if tape_w else None

    # ------------------------------------------------------------------------------- privatisation plan
    priv = []
    budget = LDS_BYTES
    for k in outs:
        s = prog.tallies[k]
        if k in raw:
            continue
        nbytes = tally_lds_bytes(s)
        if nbytes <= budget:
            budget -= nbytes
            priv.append(k)

    # the smallest privatised tallies (a wall tally's bins, say) accumulate in each lane's registers, one register
    # per bin, merged into the workgroup's copy once when the lane exits: no LDS atomic per emit.  (An exact tally
    # would take 2 x XW registers per bin in every lane -- measured slower on C5's reverse launch -- so it stays in
    # LDS.)
    # float32 sums accumulated as float64 in LDS (LDS_F64), rounded once per workgroup by the flush
    d64, left = set(), 0 if lean else LDS_F64
    for k in priv:
        s = prog.tallies[k]
        if s.dtype == C.F32 and not s.exact and not s.fixed and 8 * s.S <= left:
            left -= 8 * s.S
            d64.add(k)

    def copies(S, words):
        """LDS copies per bin of an 8-byte accumulator of S bins, while all of them fit `words`."""
        R = 16
        while R > 1 and (S * R > LDS_COPIES or S * R > words):
            R //= 2
        return R
    ncopy, room = {}, 0 if lean else LDS_F64 // 8
    for k in priv:
        s = prog.tallies[k]
        if k in d64 or (s.dtype == C.F64 and not s.fixed and not s.exact):
            ncopy[k] = copies(s.S, room)
            room -= s.S * ncopy[k] if ncopy[k] > 1 else 0

    def copy_of(ei, R):
        """the index of bin ei's copy for this lane."""
        return ei if R == 1 else f"{ei} * {R} + (threadIdx.x & {R - 1}u)"

    def sum_copies(nm, R):
        """the flush's total of bin i's copies (a C expression)."""
        return f"{nm}[i]" if R == 1 else "(" + " + ".join(f"{nm}[i * {R} + {q}]" for q in range(R)) + ")"
    rpriv = [k for k in priv if prog.tallies[k].S <= REG_BINS and not prog.tallies[k].fixed
             and not prog.tallies[k].exact and prog.tallies[k].dtype in (C.F32, C.I32, C.U32)]
    em = Emitter()
    counts = {}                 # (tally slot, f32 bits of a constant emitted value) -> (LDS u64 counter array, value)
    rcounts = {}                # the same, for a lane-register tally: -> (the lane's u32 counter names per bin, value)

    emitted = set()             # the slots an emit was written for (a tangent that is always zero has none)
    quiet = set(getattr(prog, "quiet_tallies", ()))
    lead = [False]              # emitting the update side of a group of lanes (tail loop)

    def emit_rule(em_, e, ins):
        t, idx, val = ins
        k = t.slot
        s = prog.tallies[k]
        if s.kind == "discard":
            return t
        emitted.add(k)
        ei = em_.bind(idx.el[0], np.int32, "ei")
        ok = em_.bind(f"(u32){ei} < {s.S}u", C.BOOL, "ok")
        if lead[0]:            # (a group of lanes holds the item: one of them emits)
            if k not in quiet:
                em_.line(f"tm_drop += (tm_lead && !{ok}) ? 1 : 0;")
            em_.open(f"if (tm_lead && {ok})")
        else:
            if k not in quiet:
                em_.line(f"tm_drop += {ok} ? 0 : 1;")
            em_.open(f"if ({ok})")
        v = val.el[0]
        lv = e.invars[2]
        if k in rpriv:
            bins = range(s.S)
            if (s.dtype == C.F32 and not s.exact and isinstance(lv, C.Lit) and np.isfinite(float(lv.val))
                    and float(lv.val) != 0.0):
                c = np.float32(lv.val)
                key = (k, int(c.view(np.uint32)))
                if key not in rcounts:
                    rcounts[key] = ([f"tm_rn{k}_{len(rcounts)}_{b}" for b in bins], c)
                names = rcounts[key][0]
                em_.line(" else ".join(f"if ({ei} == {b}) ++{names[b]};" if b < s.S - 1 else f"++{names[b]};"
                                       for b in bins))
            else:
                em_.line(" else ".join((f"if ({ei} == {b}) " if b < s.S - 1 else "") + f"tm_r{k}_{b} += {v};"
                                       for b in bins))
            em_.close()
            return t
        if (k in priv and s.dtype == C.F32 and not s.exact and isinstance(lv, C.Lit)
                and np.isfinite(float(lv.val)) and float(lv.val) != 0.0):
            # a constant f32 emit into a privatised tally: count it (integer LDS atomics run far faster than f32
            # ones on CDNA), the flush adds count x constant
            c = np.float32(lv.val)
            key = (k, int(c.view(np.uint32)))
            if key not in counts:
                counts[key] = (f"tm_cn{k}_{len(counts)}", c)
            em_.line(f"atomicAdd(&{counts[key][0]}[TM_CN{k}({ei})], 1ull);")
            em_.close()
            return t
        if s.exact:
            acc = f"tm_xsh{k}" if k in priv else f"((u64*)P.p[{r_scr[k]}])"
            fl = f"tm_xfl{k}" if k in priv else f"((u32*)P.p[{r_scr[k]}] + {2 * XW * s.S})"
            em_.line(f"if (tm_xemit(&{acc}[(i64){ei} * {XW}], {v})) atomicOr(&{fl}[{ei} >> 5], 1u << ({ei} & 31));")
        elif s.fixed:
            lo = f"tm_wsh{k}" if k in priv else f"((u64*)P.p[{r_scr[k]}])"
            cw = f"tm_wsc{k}" if k in priv else f"((i32*)P.p[{r_scr[k]}] + {2 * s.S})"
            em_.line(f"if (!tm_wemit(&{lo}[{ei}], &{cw}[{ei}], (double){v}, {lit(s.scale, np.float64)})) {{ "
                     f"atomicAdd(&TM_STATS[3], 1); ((u32*)P.p[{r_scr[k]}] + {3 * s.S})[{ei}] = 1u; }}")
        elif s.dtype == C.F32:
            if k in d64:
                em_.line(f"atomicAdd(&tm_sh{k}[{copy_of(ei, ncopy[k])}], (double){v});")
            elif k in priv:
                em_.line(f"tm_ladd_f32(&tm_sh{k}[{ei}], {v});")
            else:
                em_.line(f"tm_gadd_f32(&((float*)P.p[{r_out[k]}])[{ei}], {v});")
        elif s.dtype == C.F64:
            if k in priv:
                em_.line(f"tm_ladd_f64(&tm_sh{k}[{copy_of(ei, ncopy[k])}], {v});")
            else:
                em_.line(f"tm_gadd_f64(&((double*)P.p[{r_out[k]}])[{ei}], {v});")
        elif s.dtype in (C.I32, C.U32):
            ct = ctype(s.dtype)
            dst = f"tm_sh{k}" if k in priv else f"(({ct}*)P.p[{r_out[k]}])"
            em_.line(f"atomicAdd(&{dst}[{ei}], {v});")
        elif s.dtype in (C.I64, C.U64):
            dst = f"tm_sh{k}" if k in priv else f"((u64*)P.p[{r_out[k]}])"
            em_.line(f"tm_gadd_u64((u64*)&{dst}[{ei}], (u64){v});")
        else:
            raise NotImplementedError(f"sum output of dtype {s.dtype}")
        em_.close()
        return t
    em.hooks["tallymap_emit"] = emit_rule

    def emit_slot_rule(em_, e, ins):
        """an emit addressed by tally slot (params slot) rather than by a threaded tally value: the adjoint's sparse
        table-read cotangents, emitted where the read's step VJP runs."""
        emit_rule(em_, C.Eqn("tallymap_emit", [None] + list(e.invars), [], {}), [VTally(int(e.params["slot"]))] + ins)
        return []
    em.hooks["tallymap_emit_slot"] = emit_slot_rule

    def claim_rule(em_, e, ins):
        """a Records append's raw slot (tm_rclaim: the wave's batch), -1 when `when` is false.  Inside a cond
        branch, tm_rclaim_direct (a counter claim per wave at this point): the batch state passes between appends
        through plain LDS loads and first-lane stores, sound only where all the wave's lanes run the same code."""
        t, w, _ = ins
        j = int(e.params["r"])
        if em_.div:
            sl = em_.bind(f"(i32)tm_rclaim_direct((u64*)P.p[{r_rctr}] + {RC_WORDS // 2 * j}, "
                          f"(u64*)&tm_rcnt{j}[threadIdx.x >> 6], {w.el[0]}, tm_rawcap{j})", C.I32, "sl")
            return [t, Val([sl], (), C.I32)]
        sl = em_.bind(f"(i32)tm_rclaim<{rec_info[j]['segments']}, {SHARD_WORDS // 2}>((u64*)P.p[{r_rctr}] + "
                      f"{RC_WORDS // 2 * j}, &tm_rbase{j}[threadIdx.x >> 6], &tm_rleft{j}[threadIdx.x >> 6], "
                      f"&tm_rcnt{j}[threadIdx.x >> 6], &tm_rseg{j}[threadIdx.x >> 6], {w.el[0]}, tm_rawseg{j})",
                      C.I32, "sl")
        return [t, Val([sl], (), C.I32)]
    em.hooks["tallymap_claim"] = claim_rule

    def put_rule(em_, e, ins):
        """a Records field or key stored at its raw slot: a plain store, once per slot (a float adds +0.0 first,
        so -0.0 is stored as +0.0 like the reference's add into a zeroed buffer)."""
        t, idx, val = ins
        k = t.slot
        s = prog.tallies[k]
        ct = ctype(s.dtype)
        v = f"({val.el[0]} + ({ct})0)" if s.dtype in (C.F32, C.F64) else val.el[0]
        j = next(ri["ctr"] for ri in rec_info if s.name.startswith(rkey(ri["name"], "")))
        em_.line(f"if ((u64)(u32){idx.el[0]} < tm_rawcap{j}) (({ct}*)P.p[{r_out[k]}])[{idx.el[0]}] = {v};")
        return t
    em.hooks["tallymap_put"] = put_rule
    em.hooks["tallymap_item_index"] = lambda em_, e, ins: Val(["((i32)tm_item)"], (), C.I32)

    def _words_of(em_, v):
        """the u32 words of a value's elements (a 64-bit element: low word first)."""
        ws = []
        for el in v.el:
            ct = ctype(v.dtype)
            if v.dtype.itemsize == 8:
                b = em_.bind(f"__builtin_bit_cast(u64, ({ct})({el}))", C.U64, "tw")
                ws += [f"(u32){b}", f"(u32)({b} >> 32)"]
            elif ct in ("float", "i32", "u32"):
                ws.append(f"__builtin_bit_cast(u32, ({ct})({el}))")
            else:
                ws.append(f"(u32)({el})")
        return ws

    def tape_row(em_, k, cap, const, ck=False):
        """slot k of the item's tape row (a row: cap slots of tape_w words, then tape_ck words of checkpoint), or
        (ck) the row's checkpoint."""
        p = em_.fresh("tp")
        at = f"(u64)(u32)({cap}) * {tape_w}ull" if ck else f"(u64)(u32)({k}) * {tape_w}ull"
        em_.line(f"{const}u32* const {p} = ({const}u32*)P.p[{r_tape}] + (u64)tm_item * ((u64)(u32)({cap}) * "
                 f"{tape_w}ull + {tape_ck}ull) + {at};")
        return p

    def tape_put_rule(em_, e, ins):
        """leaves into slot k of the item's tape row when k < cap, or (ck) into the row's checkpoint when k == cap
        (whole 16- or 8-byte units)."""
        t, k, cap = ins[0], ins[1], ins[2]
        W, ck = int(e.params["words"]), bool(e.params.get("ck", False))
        ws = [w_ for v in ins[3:] for w_ in _words_of(em_, v)]
        ws += ["0u"] * (W - len(ws))
        em_.open(f"if ({'tm_lead && ' if lead[0] else ''}(u32)({k.el[0]}) {'==' if ck else '<'} (u32)({cap.el[0]}))")
        p = tape_row(em_, k.el[0], cap.el[0], "", ck)
        u = 4 if W % 4 == 0 else (2 if W % 2 == 0 else 1)
        for q in range(0, W, u):
            if u == 1:
                em_.line(f"{p}[{q}] = {ws[q]};")
            else:
                em_.line(f"*(tm_u32x{u}*)&{p}[{q}] = (tm_u32x{u}){{{', '.join(ws[q:q + u])}}};")
        em_.close()
        return t
    em.hooks["tallymap_tape_put"] = tape_put_rule

    def _vals_of(em_, words, avals):
        """the values of `avals` whose elements' u32 words are `words` (_words_of's order)."""
        outs, w_ = [], 0
        for a in avals:
            ct = ctype(a.dtype)
            els = []
            for _ in range(max(1, a.size)):
                if a.dtype.itemsize == 8:
                    els.append(em_.bind(f"__builtin_bit_cast({ct}, (u64)({words[w_]}) | ((u64)({words[w_ + 1]}) << 32))",
                                        a.dtype, "tg"))
                    w_ += 2
                elif ct in ("float", "i32", "u32"):
                    els.append(em_.bind(f"__builtin_bit_cast({ct}, (u32)({words[w_]}))", a.dtype, "tg"))
                    w_ += 1
                elif ct == "bool":
                    els.append(em_.bind(f"(({words[w_]}) != 0u)", a.dtype, "tg"))
                    w_ += 1
                else:
                    els.append(em_.bind(f"({ct})({words[w_]})", a.dtype, "tg"))
                    w_ += 1
            outs.append(Val(els, a.shape, a.dtype))
        return outs

    def tape_get_rule(em_, e, ins):
        """the leaves stored in slot j (< cap) of the item's tape row, or (ck) in its checkpoint."""
        j, cap = ins
        W, ck = int(e.params["words"]), bool(e.params.get("ck", False))
        p = tape_row(em_, j.el[0], cap.el[0], "const ", ck)
        words = []
        u = 4 if W % 4 == 0 else (2 if W % 2 == 0 else 1)
        for q in range(0, W, u):
            if u == 1:
                words.append(em_.bind(f"{p}[{q}]", C.U32, "tq"))
                continue
            v = em_.fresh("tq")
            em_.line(f"const tm_u32x{u} {v} = *(const tm_u32x{u}*)&{p}[{q}];")
            words += [f"{v}.{c}" for c in "xyzw"[:u]]
        return _vals_of(em_, words, [o.aval for o in e.outvars])
    em.hooks["tallymap_tape_get"] = tape_get_rule

    def spawn_rule(em_, e, ins):
        """a spawned child.  Staged (QS > 0): the spawning lanes write the child's operands as words into their
        wave's LDS staging rows (rank order after the wave's count); a wave whose rows would overflow first
        flushes them (_qflush_lines: one ticket claim for all of them, then rows stored to the next generation's
        buffer), and each wave flushes what is left when it exits.  Direct (QS = 0): one ticket claim per wave at
        this point (tm_qclaim) and the row stored at once.  Tickets past the capacity Q are not stored (the host
        counts them as dropped children).  A spawn inside a cond branch is always direct: the staging count passes
        between spawn points through LDS, and lanes of one wave in two branches run one branch after the other;
        the compiler, which reasons per lane, may merge the branches' trailing first-lane stores of the count into
        one after both, so the second branch would stage over the first's rows."""
        t, w, leaves = ins[0], ins[1], ins[2:]
        if Q is None or len(leaves) != len(qav):
            raise RuntimeError("internal: a spawn in a program without a queue of its per-item operands")
        when = f"(tm_lead && {w.el[0]})" if lead[0] else w.el[0]
        if not QS or em_.div:
            tq = em_.bind(f"tm_qclaim(tm_qctr, {when})", C.I64, "tq")
            em_.open(f"if ((u64){tq} < {int(Q)}ull)")
            for i, (lv, a) in enumerate(zip(leaves, qav)):
                ct, n = ctype(a.dtype), max(1, a.size)
                for el in range(n):
                    em_.line(f"(({ct}*)P.p[{r_q[i]}])[{tq} * {n} + {el}] = {lv.el[el]};")
            em_.close()
            return t
        wv = em_.bind(when, C.BOOL, "sw")
        m, nn, q = em_.fresh("sm"), em_.fresh("sn"), em_.fresh("sq")
        em_.line(f"const u64 {m} = tm_ballot({wv});")
        em_.open(f"if ({m} != 0ull)")
        em_.line(f"const u32 {nn} = (u32)__builtin_popcountll({m});")
        em_.line(f"u32 {q} = tm_qn[threadIdx.x >> 6];")
        em_.open(f"if ({q} + {nn} > {QS}u)")
        for ln in _qflush_lines(q):
            em_.line(ln)
        em_.line(f"{q} = 0u;")
        em_.close()
        em_.open(f"if ({wv})")
        d = em_.fresh("sd")
        em_.line(f"volatile u32* const {d} = tm_qs + ({q} + tm_rank({m})) * {q_words}u;")
        for i, (lv, a) in enumerate(zip(leaves, qav)):
            for el in range(max(1, a.size)):
                o = q_off[i] + el * (2 if a.dtype.itemsize == 8 else 1)
                v = lv.el[el]
                if a.dtype.itemsize == 8:
                    b = em_.bind(f"__builtin_bit_cast(u64, ({ctype(a.dtype)})({v}))", C.U64, "sb")
                    em_.line(f"{d}[{o}] = (u32){b}; {d}[{o + 1}] = (u32)({b} >> 32);")
                elif a.dtype.itemsize == 4:
                    em_.line(f"{d}[{o}] = __builtin_bit_cast(u32, ({ctype(a.dtype)})({v}));")
                else:
                    em_.line(f"{d}[{o}] = (u32)({v});")
        em_.close()
        em_.line("__builtin_amdgcn_wave_barrier();")
        em_.line(f"if (tm_lane() == (int)__builtin_ctzll(tm_ballot(true))) tm_qn[threadIdx.x >> 6] = {q} + {nn};")
        em_.close()
        return t

    def _qflush_lines(cnt):
        """store the wave's `cnt` staged children to the next generation's buffer with the lanes that are active:
        one ticket claim for all of them, the rows spread over the lanes."""
        rd = []
        for i, a in enumerate(qav):
            ct, n = ctype(a.dtype), max(1, a.size)
            for el in range(n):
                o = q_off[i] + el * (2 if a.dtype.itemsize == 8 else 1)
                if a.dtype.itemsize == 8:
                    v = f"__builtin_bit_cast({ct}, (u64)tm_fs[{o}] | ((u64)tm_fs[{o + 1}] << 32))"
                elif a.dtype.itemsize == 4:
                    v = f"__builtin_bit_cast({ct}, tm_fs[{o}])"
                elif a.dtype == C.BOOL:
                    v = f"(tm_fs[{o}] != 0u)"
                else:
                    v = f"({ct})tm_fs[{o}]"
                rd.append(f"      (({ct}*)P.p[{r_q[i]}])[tm_ft * {n} + {el}] = {v};")
        return ([ "{",
                 f"  const u64 tm_fb = tm_claim(tm_qctr, {cnt});",
                  "  const u64 tm_fa = tm_ballot(true);",
                  "  const u32 tm_fna = (u32)__builtin_popcountll(tm_fa);",
                  "  __builtin_amdgcn_wave_barrier();",
                 f"  for (u32 tm_fe = tm_rank(tm_fa); tm_fe < {cnt}; tm_fe += tm_fna) {{",
                  "    const u64 tm_ft = tm_fb + tm_fe;",
                 f"    if (tm_ft < {int(Q)}ull) {{",
                 f"      const volatile u32* const tm_fs = tm_qs + tm_fe * {q_words}u;"]
                + rd + ["    }", "  }", "  __builtin_amdgcn_wave_barrier();", "}"])
    em.hooks["tallymap_spawn"] = spawn_rule

    # --------------------------------------------------------------------------------- the item's code
    w = _split(jx) if schedule == "step" else None
    mode = "step" if w is not None else "item"
    tallies = [VTally(k) for k in range(nT)]
    staged = _staged_tables(jx, nT + nP, bav, int(lds_tables))
    bvals = []
    for i, a in enumerate(bav):
        ct = ctype(a.dtype)
        if i in staged:             # copied into LDS in the prologue, read there
            bvals.append(Val([f"tm_tab{i}[{e}]" for e in range(a.size)], a.shape, a.dtype, ptr=f"tm_tab{i}"))
        elif a.size > BCAST_REG:    # a larger broadcast array is read in place (and can be indexed dynamically)
            ptr = f"((const {ct}*)P.p[{nP + i}])"
            bvals.append(Val([f"{ptr}[{e}]" for e in range(a.size)], a.shape, a.dtype, ptr=ptr))
        else:
            bvals.append(Val([f"tm_b{i}_{e}" for e in range(max(1, a.size))], a.shape, a.dtype,
                             ptr=f"((const {ct}*)P.p[{nP + i}])"))

    # per-item operands of 4-byte elements are staged in LDS per wave chunk: word offsets within an item's record
    stage_off, W = {}, 0
    for i, a in enumerate(pav):
        if a.dtype.itemsize == 4:
            stage_off[i] = W
            W += max(1, a.size)

    def load_pi(i, a):
        ct = ctype(a.dtype)
        n = max(1, a.size)
        if i in stage_off:
            return Val([f"__builtin_bit_cast({ct}, tm_st[tm_loc * {W} + {stage_off[i] + e}])" for e in range(n)],
                       a.shape, a.dtype)
        return Val([f"(({'const ' + ct}*)P.p[{i}])[tm_item * {n} + {e}]" for e in range(n)], a.shape, a.dtype)

    decls, pre_lines, step_lines, post_lines, tail_lines, uni_lines = [], [], [], [], [], []
    pb_h, pl_ahead = 0, None

    def write_ys(vals, trunc_idx):
        lines = []
        for j, (v, a) in enumerate(zip(vals, yav)):
            ct = ctype(a.dtype)
            n = max(1, a.size)
            for e in range(n):
                lines.append(f"(({ct}*)P.p[{r_ys[j]}])[tm_item * {n} + {e}] = {v.el[e]};")
        if trunc_idx is not None:
            lines.append(f"if ({vals[trunc_idx].el[0]}) ++tm_ntr;")
        return lines

    if mode == "item":
        em.lines, em.ind = [], 4
        pis = []
        for i, a in enumerate(pav):
            lv = load_pi(i, a)
            pis.append(Val([em.bind(x, a.dtype, "x") for x in lv.el], a.shape, a.dtype))
        outv = em.run(jx, tallies + pis + bvals)
        for ln in write_ys(outv[nT:], prog.trunc):
            em.line(ln)
        pre_lines = em.lines
    else:
        we = jx.eqns[w]
        pre_e, post_e = jx.eqns[:w], jx.eqns[w + 1:]
        nc, nb = we.params["cond_nconsts"], we.params["body_nconsts"]
        ops = we.invars
        cc_v, bc_v, init_v = ops[:nc], ops[nc:nc + nb], ops[nc + nb:]
        post_used = _used_vars(post_e, jx.outvars)
        loop_used = {v.id for v in cc_v + bc_v if isinstance(v, C.Var)}
        bids = {v.id for v in jx.invars[nT + nP:]}
        # ---- pre: loads + pre eqns -> carries and persistent state
        em.lines, em.ind = [], 5
        env = {}
        for v, t in zip(jx.invars[:nT], tallies):
            env[v.id] = t
        for i, (v, a) in enumerate(zip(jx.invars[nT:nT + nP], pav)):
            lv = load_pi(i, a)
            env[v.id] = Val([em.bind(x, a.dtype, "x") for x in lv.el], a.shape, a.dtype)
        for v, bv in zip(jx.invars[nT + nP:], bvals):
            env[v.id] = bv
        # PRE values of broadcast operands alone are the same for every item: computed once per kernel, held as scalars
        # (no state per lane, nothing to repack), and their reciprocals taken there (tm_div_by)
        loads, uni = em.lines, set(bids)
        em.lines, em.ind = [], 1
        once = [el for a, bv in zip(bav, bvals) if a.dtype == C.F32 and a.size <= BCAST_REG for el in bv.el]
        for e in pre_e:
            if not Ahead.pure(e) or any(x.prim == "tallymap_item_index" for x in C.walk_eqns(C.Jaxpr([], [], [e]))) \
                    or not all(isinstance(v, C.Lit) or v.id in uni for v in e.invars) or any(
                    o.aval.dtype.itemsize != 4 or o.aval.size > BCAST_REG for o in e.outvars):
                continue
            outs_ = em.eqn(e, [em.value_of(env, x) for x in e.invars])
            for o, x in zip(e.outvars, outs_):
                names = []
                for el in x.el:
                    names.append(em.bind(f"__builtin_bit_cast({ctype(x.dtype)}, tm_bcast_first(__builtin_bit_cast(u32, "
                                         f"({ctype(x.dtype)})({el}))))", x.dtype, "un"))
                env[o.id] = Val(names, x.shape, x.dtype)
                uni.add(o.id)
                if x.dtype == C.F32:
                    once += names
        for i_, el in enumerate(once):
            nm = em.invariant[el] = f"tm_rc{i_}"
            em.line(f"const u64 {nm}u = __builtin_bit_cast(u64, 1.0 / (double){el});")
            em.line(f"const double {nm} = __builtin_bit_cast(double, (u64)tm_bcast_first((u32){nm}u) | "
                    f"((u64)tm_bcast_first((u32)({nm}u >> 32)) << 32));")
        uni_lines, bids = em.lines, uni
        em.lines, em.ind = loads, 5
        for e in pre_e:
            if all(o.id in uni for o in e.outvars) and e.outvars:
                continue
            vals = [em.value_of(env, x) for x in e.invars]
            for o, x in zip(e.outvars, em.eqn(e, vals)):
                env[o.id] = x
        # persistent values: defined before the loop (per-item inputs included), read by the loop or post
        state = {}
        need = (loop_used | post_used)
        cand = [v for v in jx.invars[nT:nT + nP]] + [o for e in pre_e for o in e.outvars]
        for v in cand:
            if v.id in need and v.id not in bids and not isinstance(env.get(v.id), VTally):
                x = env[v.id]
                names = []
                for j, el in enumerate(x.el):
                    nm = f"tm_s{len(state)}_{j}"
                    names.append(nm)
                    decls.append(f"  {ctype(x.dtype)} {nm};")
                    em.line(f"{nm} = {el};")
                state[v.id] = Val(names, x.shape, x.dtype)
        cars = []
        for j, (v, o) in enumerate(zip(init_v, we.outvars)):
            x = em.value_of(env, v)
            if isinstance(x, VTally):
                cars.append(x)
                continue
            names = []
            for e_, el in enumerate(x.el):
                nm = f"tm_c{j}_{e_}"
                names.append(nm)
                decls.append(f"  {ctype(o.aval.dtype)} {nm};")
                em.line(f"{nm} = {el};")
            cars.append(Val(names, o.aval.shape, o.aval.dtype))
        pre_lines = em.lines

        def sval(v):
            if isinstance(v, C.Lit):
                return em.value_of({}, v)
            if v.id in bids:
                return env[v.id]
            if v.id in state:
                return state[v.id]
            x = env.get(v.id)
            if isinstance(x, VTally):
                return x
            raise RuntimeError("internal: a loop operand is neither state nor broadcast")
        # the wait before POST, in lane-iterations (0: each item's POST in the step its condition fails)
        step_c = cost(we.params["cond_jaxpr"].eqns) + cost(we.params["body_jaxpr"].eqns)
        fin_c = cost(post_e) + cost(pre_e) + W + 16 + 2 * len(yav)
        pb_h = int(round(float(post_batch or 0) * 64 * fin_c / max(1, step_c)))
        if pb_h < POST_BATCH_MIN:
            pb_h = 0
        def post():
            """the item's POST and its per-item results."""
            penv = {}
            for v in jx.invars[:nT]:
                penv[v.id] = env[v.id]
            for i_ in bids:
                penv[i_] = env[i_]
            penv.update((i_, x) for i_, x in env.items() if isinstance(x, VTally))     # (emitted into by PRE)
            for vid, x in state.items():
                penv[vid] = x
            for o, c in zip(we.outvars, cars):
                penv[o.id] = c
            for e in post_e:
                vals = [em.value_of(penv, x) for x in e.invars]
                for o, x in zip(e.outvars, em.eqn(e, vals)):
                    penv[o.id] = x
            outv = [em.value_of(penv, v) for v in jx.outvars]
            for ln in write_ys(outv[nT:], prog.trunc):
                em.line(ln)

        def step(ind, deferred):
            """one step of a live lane: cond; body, or the item's end (deferred: its POST waits)."""
            em.lines, em.ind = [], ind
            pr = em.run(we.params["cond_jaxpr"], [sval(v) for v in cc_v] + cars)[0]
            em.open(f"if ({pr.el[0]})")
            bouts = em.run(we.params["body_jaxpr"], [sval(v) for v in bc_v] + cars)
            assign_carries(em, cars, bouts)
            em.close("} else {")
            em.ind += 1
            if not deferred:
                post()
            em.line("tm_live = false;")
            if deferred:
                em.line("tm_pend = true;")
            em.close()
            return em.lines
        step_lines = step(4, pb_h > 0)
        if pb_h:
            em.lines, em.ind = [], 7
            post()
            post_lines = em.lines
        def tail_ahead(pl):
            """a group's round in the tail loop (Ahead): lane tm_go of the group computes the values of the step
            tm_go ahead, then the group runs tm_g updates, update j on the values of its lane j."""
            bj, nb_ = we.params["body_jaxpr"], we.params["body_nconsts"]
            em.lines, em.ind = [], 4
            ins_ = [sval(v) for v in bc_v] + cars
            e_ = {v.id: x for v, x in zip(bj.invars, ins_)}
            for j, gain in pl.counters.items():
                v = bj.invars[nb_ + j]
                e_[v.id] = Val([em.bind(f"({ctype(v.aval.dtype)})((u32){cars[j].el[0]} + tm_go * {gain & 0xffffffff}u)",
                                        v.aval.dtype, "kg")], (), v.aval.dtype)
            for q in pl.ahead:
                for o, x in zip(q.outvars, em.eqn(q, [em.value_of(e_, v) for v in q.invars])):
                    e_[o.id] = x
            words = [w_ for v in pl.cut for w_ in _words_of(em, e_[v.id])]
            for i, w_ in enumerate(words):
                em.line(f"tm_h{i} = {w_};")
            head = em.lines
            em.lines, em.ind = [], 4
            lead[0] = True
            # (a straight-line condition on every lane, an item's end under a wave-uniform branch: one lane mask per
            # update.  One with a loop or a branch in it on live lanes alone: the others' state is unset)
            cj = we.params["cond_jaxpr"]
            if any(C.subjaxprs(q) for q in cj.eqns):
                em.line("bool tm_go_on = false;")
                em.open("if (tm_live)")
                em.line(f"tm_go_on = {em.run(cj, [sval(v) for v in cc_v] + cars)[0].el[0]};")
                em.close()
            else:
                pr = em.run(cj, [sval(v) for v in cc_v] + cars)[0]
                em.line(f"const bool tm_go_on = tm_live && {pr.el[0]};")
            em.open("if (tm_ballot(tm_live && !tm_go_on) != 0ull)")
            em.open("if (tm_live && !tm_go_on && tm_lead)")
            lead[0] = False
            post()
            lead[0] = True
            em.close()
            em.line("tm_live = tm_go_on;")
            em.close()
            em.open("if (tm_go_on)")
            e_ = {v.id: x for v, x in zip(bj.invars, ins_)}
            for v, x in zip(pl.cut, _vals_of(em, [f"tm_q{i}" for i in range(len(words))], [v.aval for v in pl.cut])):
                e_[v.id] = x
            for q in pl.update:
                for o, x in zip(q.outvars, em.eqn(q, [em.value_of(e_, v) for v in q.invars])):
                    e_[o.id] = x
            assign_carries(em, cars, [em.value_of(e_, v) for v in bj.outvars])
            lead[0] = False
            em.close()
            return head, em.lines, len(words)
        if compact:
            # (not with Records: their raw buffers are sized by the launch's lanes without the spread, _lanes)
            pl_ahead = Ahead.plan(we, lambda v: isinstance(v, C.Var) and isinstance(env.get(v.id), VTally), cost) \
                if not recs else None
            tail_lines = tail_ahead(pl_ahead) if pl_ahead is not None else step(5, False)

    # A small launch of a program with steps computed ahead spreads to up to 512 workgroups, each of which adds its sum
    # of a privatised float32 tally to the launch's: in float32 that many roundings lose what the float64 bins kept
    # (quickstart at 10,000 items, error against float64: 1.0e-7 in 40 workgroups, 3.1e-7 in 512).  Such a program sums
    # them in float64, and tm_post rounds once
    # (in ctl, past the claim counters: no pointer of their own through the step loop)
    wide, n_claim = {}, n_ctl
    for k in priv:
        s = prog.tallies[k]
        if pl_ahead and s.dtype == C.F32 and not s.exact and not s.fixed:
            wide[k] = n_ctl // 2
            n_ctl += 2 * s.S
    res[r_ctl - n_in] = ((n_ctl,), np.dtype(np.uint32), False)

    # ------------------------------------------------------------------------------------ assemble
    from . import compile as Cm
    src = [Cm.prelude(), f"struct TmParams {{ void* p[{n_in + len(res)}]; }};",
           f"#define TM_STATS ((i32*)P.p[{r_stats}])", f"#define TM_CTL ((u32*)P.p[{r_ctl}])",
           f"#define TM_BLOCK {block}u"]
    if pl_ahead:
        src.append(f"extern \"C\" __constant__ int tm_spread = {SPREAD};")
    if int(grid_cap) > 0:
        src.append(f"extern \"C\" __constant__ int tm_grid_cap = {int(grid_cap)};")
    zero_words = []
    for k in outs:
        s = prog.tallies[k]
        if k in raw:
            continue
        zero_words.append((r_out[k], s.S * np.dtype(s.dtype).itemsize // 4 if np.dtype(s.dtype).itemsize >= 4
                           else (s.S * np.dtype(s.dtype).itemsize + 3) // 4))
        if k in r_scr:
            zero_words.append((r_scr[k], scratch_words(s)))
    if recs:
        zero_words.append((r_rctr, RC_WORDS * len(recs)))
    zero_words += [(r_ctl, n_ctl), (r_stats, 5)]
    zl = []
    for b, nw in zero_words:
        zl.append(f"  for (i64 i = g; i < {nw}; i += s) ((u32*)P.p[{b}])[i] = 0u;")
    src.append("extern \"C\" __global__ void tm_zero(const TmParams P, const i64 n_items) {\n"
               "  const i64 g = (i64)blockIdx.x * blockDim.x + threadIdx.x, s = (i64)gridDim.x * blockDim.x;\n"
               + "\n".join(zl) + "\n}")
    # tm_post: exact readout, then the truncation poison of float tallies
    post = []
    flags = 0
    for k in outs:
        s = prog.tallies[k]
        if s.exact:
            words = f"((const u64*)P.p[{r_scr[k]}])"
            fl = f"((const u32*)P.p[{r_scr[k]}] + {2 * XW * s.S})"
            if s.dtype == C.F64:   # (a tangent's exact sum: not among the call's outputs, so none of its overflows)
                post.append(f"for (i64 i = g; i < {s.S}; i += st) ((double*)P.p[{r_out[k]}])[i] = "
                            f"(({fl}[i >> 5] >> (i & 31)) & 1u) != 0u ? __builtin_nan(\"\") : "
                            f"tm_xread_f64(&{words}[i * {XW}]);")
                continue
            post.append(f"for (i64 i = g; i < {s.S}; i += st) {{ bool bad = false; "
                        f"const float o = tm_xread(&{words}[i * {XW}], &bad); "
                        f"const bool f = (({fl}[i >> 5] >> (i & 31)) & 1u) != 0u; "
                        f"if (f || bad) atomicAdd(&TM_STATS[3], 1); "
                        f"((float*)P.p[{r_out[k]}])[i] = (f || bad) ? __builtin_nanf(\"\") : o; }}")
        elif s.fixed:
            post.append(_wide_readout(s, f"((const u64*)P.p[{r_scr[k]}])", f"((const i32*)P.p[{r_scr[k]}] + {2 * s.S})",
                                      f"((const u32*)P.p[{r_scr[k]}] + {3 * s.S})", f"P.p[{r_out[k]}]"))
        elif k in wide:
            post.append(f"for (i64 i = g; i < {s.S}; i += st) {{ float* const o = &((float*)P.p[{r_out[k]}])[i]; "
                        f"*o = (float)((double)*o + ((const double*)P.p[{r_ctl}])[{wide[k]} + i]); }}")
    poison = [k for k in outs if prog.tallies[k].dtype in (C.F32, C.F64) and k not in raw]
    bad = ["TM_CTL[2] != 0u"] if prog.trunc is not None else []
    # a Records output past its capacity poisons every float output of the call (reference _api.py:120-131)
    bad += [f"((const u64*)P.p[{r_rctr}])[{RC_WORDS // 2 * ri['ctr'] + RC_TOTAL}] > {ri['capacity']}ull"
            for ri in rec_info]
    if Q is not None:          # a dropped child (tm_qnext counts them from the generations' tickets)
        bad.append("TM_STATS[1] != 0")
    if bad and poison:
        # (the readout and the poison visit a bin from the same thread, in program order)
        post.append(f"const bool tm_bad = {' || '.join(bad)};")
        for k in poison:
            s = prog.tallies[k]
            ct = ctype(s.dtype)
            post.append(f"if (tm_bad) for (i64 i = g; i < {s.S}; i += st) "
                        f"(({ct}*)P.p[{r_out[k]}])[i] = __builtin_nanf(\"\");")
    pz = getattr(prog, "poison_ys", False)
    if pz and prog.trunc is not None:
        # a derived program (the adjoint): every float per-item result (True) or those listed (the cotangents of a
        # value_and_grad launch) is NaN when an item was truncated
        for j, a in enumerate(yav):
            if pz is not True and j not in pz:
                continue
            if a.dtype in (C.F32, C.F64):
                n = max(1, a.size)
                post.append(f"if (TM_CTL[2] != 0u) for (i64 i = g; i < n_items * {n}; i += st) "
                            f"(({ctype(a.dtype)}*)P.p[{r_ys[j]}])[i] = __builtin_nanf(\"\");")
    if post:
        # (nothing but the float64 sums to read out: only where the launch spread, which tm_launch knows)
        flags |= 8 if len(post) == len(wide) else 2
        src.append("extern \"C\" __global__ void tm_post(const TmParams P, const i64 n_items) {\n"
                   "  const i64 g = (i64)blockIdx.x * blockDim.x + threadIdx.x, st = (i64)gridDim.x * blockDim.x;\n  "
                   + "\n  ".join(post) + "\n}")
    if Q is not None:
        # tm_qnext, one wave between two generations: the next generation's item count min(tickets, Q), the
        # spawned / dropped totals and the stats they give (children_truncated: truncations past the roots'), and
        # the claim and ticket counters cleared.  `first` (after the roots' launch) keeps the roots' truncations.
        big = 2 ** 31 - 1
        src.append("extern \"C\" __global__ void tm_qnext(const TmParams P, const i64 first) {\n"
                   "  if (blockIdx.x != 0) return;\n"
                   f"  for (u32 i = threadIdx.x; i < {SHARDS}u; i += blockDim.x) "
                   f"((u64*)P.p[{r_ctl}])[{SHARD0 // 2} + i * {SHARD_WORDS // 2}u] = 0ull;\n"
                   "  if (threadIdx.x != 0) return;\n"
                   f"  u64* const c = (u64*)P.p[{r_ctl}];\n"
                   f"  const u64 cnt = c[16], n = cnt < {Q}ull ? cnt : {Q}ull;\n"
                   "  if (first) TM_CTL[48] = TM_CTL[2];\n"
                   "  const u64 sp = c[21] + n, dr = c[22] + (cnt - n);\n"
                   "  c[20] = n; c[21] = sp; c[22] = dr; c[16] = 0ull;\n"
                   f"  TM_STATS[0] = (i32)(sp < {big}ull ? sp : {big}ull);\n"
                   f"  TM_STATS[1] = (i32)(dr < {big}ull ? dr : {big}ull);\n"
                   "  TM_STATS[2] = (i32)(TM_CTL[2] - TM_CTL[48]);\n"
                   "}")

    # tm_main
    body = []
    # the item loop is named for its role (profiles tell the launches apart by name; the launcher accepts each):
    # tm_main a forward, tm_adjoint a gradient launch (forward-only or checkpointed), tm_count the tape adjoint's
    # counting pass, tm_fused an adjoint launch that also returns the forward (value_and_grad); prog.entry sets it
    entry = getattr(prog, "entry", None) or ("tm_adjoint" if getattr(prog, "poison_ys", False) is not False
                                             else "tm_main")
    lb = f"{block}, {max(1, int(min_blocks) * block // 256)}" if min_blocks else f"{block}"
    body.append(f"extern \"C\" __global__ void __launch_bounds__({lb}) {entry}(const TmParams P, "
                f"const i64 {'tm_n_arg' if Q is not None else 'n_items'}) {{")
    # (the grid size is read once, as a scalar, before any branch: the compiler may otherwise merge its address out of
    # divergent prologue branches and take the whole claim control for divergent -- 94 -> 110 VGPRs in the random walk)
    body.append("  const u32 tm_grid = tm_bcast_first(gridDim.x);")
    body.append("  u64* const tm_ctr = (u64*)P.p[%d];" % r_ctl)
    if Q is not None:          # a later generation (tm_n_arg < 0) takes its item count from tm_qnext's word
        body.append(f"  const i64 n_items = tm_n_arg >= 0 ? tm_n_arg : (i64)(tm_ctr[20] < {Q}ull ? tm_ctr[20] : {Q}ull);")
        body.append("  if (n_items <= 0) return;                // (a generation queued past the last)")
    for ri in rec_info:        # each wave's Records batch state (tm_rclaim) and the raw buffers' length
        j, w, S, cap = ri["ctr"], block // 64, ri["segments"], ri["capacity"]
        body.append(f"  __shared__ u64 tm_rbase{j}[{w}], tm_rcnt{j}[{w}];")
        body.append(f"  __shared__ u32 tm_rleft{j}[{w}], tm_rseg{j}[{w}];")
        body.append(f"  if ((threadIdx.x & 63u) == 0u) {{ tm_rbase{j}[threadIdx.x >> 6] = 0ull; "
                    f"tm_rcnt{j}[threadIdx.x >> 6] = 0ull; tm_rleft{j}[threadIdx.x >> 6] = 0u; "
                    f"tm_rseg{j}[threadIdx.x >> 6] = blockIdx.x % {S}u; }}")
        body.append(f"  const u64 tm_rawseg{j} = " + (
            f"{cap}ull + (u64)tm_grid * {w * (RB - 1)}ull;" if S == 1 else
            f"({-(-cap // RB)}ull + (u64)tm_grid * {w}ull + {S - 1}ull) / {S}ull * {RB}ull;"))
        body.append(f"  const u64 tm_rawcap{j} = tm_rawseg{j} * {S}ull;")
    if Q is not None:          # the spawn ticket counter; each wave's staging rows and their count
        body.append("  u64* const tm_qctr = tm_ctr + 16;")
        if QS:
            body.append(f"  __shared__ u32 tm_qst[{(block // 64) * QS * q_words}];")
            body.append(f"  __shared__ u32 tm_qnv[{block // 64}];")
            body.append("  volatile u32* const tm_qn = tm_qnv;")
            body.append(f"  volatile u32* const tm_qs = tm_qst + (threadIdx.x >> 6) * {QS * q_words}u;")
            body.append("  if ((threadIdx.x & 63u) == 0u) tm_qn[threadIdx.x >> 6] = 0u;")
    for k in priv:
        s = prog.tallies[k]
        if s.exact:
            nw = XW * s.S
            body.append(f"  __shared__ u64 tm_xsh{k}[{nw}];")
            body.append(f"  __shared__ u32 tm_xfl{k}[{(s.S + 31) // 32}];")
            body.append(f"  for (int i = threadIdx.x; i < {nw}; i += TM_BLOCK) tm_xsh{k}[i] = 0ull;")
            body.append(f"  for (int i = threadIdx.x; i < {(s.S + 31) // 32}; i += TM_BLOCK) tm_xfl{k}[i] = 0u;")
        elif s.fixed:
            body.append(f"  __shared__ u64 tm_wsh{k}[{s.S}];")
            body.append(f"  __shared__ i32 tm_wsc{k}[{s.S}];")
            body.append(f"  for (int i = threadIdx.x; i < {s.S}; i += TM_BLOCK) {{ tm_wsh{k}[i] = 0ull; "
                        f"tm_wsc{k}[i] = 0; }}")
        else:
            ct = "double" if k in d64 else ctype(s.dtype)
            n = s.S * ncopy.get(k, 1)
            body.append(f"  __shared__ {ct} tm_sh{k}[{n}];")
            body.append(f"  for (int i = threadIdx.x; i < {n}; i += TM_BLOCK) tm_sh{k}[i] = ({ct})0;")
    body.append("//TM_COUNT_DECLS")
    if wide:                   # (a spread launch: more workgroups than its items fill; read by the flush)
        body.append("  __shared__ u32 tm_spread_s;")
        body.append("  if (threadIdx.x == 0) tm_spread_s = (u64)tm_grid * TM_BLOCK >= (u64)n_items + TM_BLOCK ? 1u : 0u;")
    for i in staged:
        a = bav[i]
        ct = ctype(a.dtype)
        body.append(f"  __shared__ {ct} tm_tab{i}[{a.size}];")
        body.append(f"  for (int i = threadIdx.x; i < {a.size}; i += TM_BLOCK) "
                    f"tm_tab{i}[i] = ((const {ct}*)P.p[{nP + i}])[i];")
    if priv or staged:
        body.append("  __syncthreads();")
    for i, a in enumerate(bav):
        ct = ctype(a.dtype)
        if a.size > BCAST_REG:
            continue
        for e in range(max(1, a.size)):
            body.append(f"  const {ct} tm_b{i}_{e} = ((const {ct}*)P.p[{nP + i}])[{e}];")
    body += uni_lines
    wpb = block // 64
    compact_on = bool(compact) and mode == "step"
    if compact_on:
        pack, unpack, nwords = _repack_code(decls, wpb * 64)
    # one LDS array serves the operand staging of claimed chunks and, once every wave of the workgroup has drained
    # the queue (no wave stages any more), the repack pool
    n_stage = wpb * chunk * W
    n_pool = nwords * wpb * 64 if compact_on else 0
    if n_stage or n_pool:
        body.append(f"  __shared__ u32 tm_lds[{max(n_stage, n_pool)}];")
    if W:
        body.append("  u32* const tm_stage = tm_lds;")
        body.append(f"  u32* const tm_st = tm_stage + (threadIdx.x >> 6) * {chunk * W};")
    body.append("  bool tm_live = false, tm_more = true;")
    body.append("  i64 tm_item = 0;")
    body.append("  u32 tm_loc = 0;")
    body.append("  u64 tm_cb = 0;                             // the wave's chunk: base item, next unassigned, end")
    body.append("  u32 tm_cur = 0u, tm_end = 0u;")
    body.append("  u64 tm_rv = 0, tm_re = 0;                  // the wave's reservation of chunks: next, end")
    body.append("  u64 tm_t0 = 0;                             // the real-time counter at the wave's last claim")
    body.append("  u32 tm_rc = 1u;                            // chunks in the wave's last reservation")
    body.append(f"  const u32 tm_wid = blockIdx.x * {wpb}u + tm_bcast_first(threadIdx.x >> 6);")
    body.append(f"  const bool tm_one = (u64)n_items <= (u64)tm_grid * {wpb * chunk}u;      // at most a chunk per wave")
    # (with steps computed ahead, a wave takes an even share: few items per workgroup are many lanes per item)
    body.append(f"  const u32 tm_ch = (u32)(((u64)n_items + tm_grid * {wpb}u - 1u) / (tm_grid * {wpb}u));"
                if pl_ahead else f"  const u32 tm_ch = {chunk}u;")
    body.append("  // the ranges: counters, items per range (whole chunks), the wave's range, its items left, waves per range")
    body.append(f"  u64* const tm_shc = tm_ctr + {SHARD0 // 2};")
    body.append(f"  const u64 tm_shn = (((u64)n_items + {SHARDS * chunk - 1}u) / {SHARDS * chunk}u) * {chunk}u;")
    body.append(f"  u32 tm_sh = blockIdx.x % {SHARDS}u;")
    body.append("  u64 tm_left = tm_shn;")
    body.append(f"  const u64 tm_shw = (tm_grid * {wpb}u + {SHARDS - 1}u) / {SHARDS}u;")
    body.append("  i32 tm_drop = 0;")
    body.append("  u32 tm_ntr = 0;")
    if pb_h:
        body.append("  bool tm_pend = false;                      // the item's condition failed, its POST waits")
        body.append("  u32 tm_acc = 0;                            // the wave's waiting lane-iterations")
    body += decls
    body.append("//TM_LANE_DECLS")
    if compact_on:
        body.append("  u32* const tm_pool = tm_lds;                  // the repack pool, one column per word")
        body.append("  __shared__ u32 tm_pn[2];                 // pool counts, alternating between rounds")
        body.append("  __shared__ u32 tm_ndr;                   // waves of this workgroup whose queue is drained")
        body.append("  if (threadIdx.x == 0) { tm_pn[0] = 0u; tm_pn[1] = 0u; tm_ndr = 0u; }")
        body.append("  __syncthreads();")
        body.append("  bool tm_dr = false;                      // drained (counted)")
        if pl_ahead:
            body.append("  bool tm_lead = true;                     // (tail) the lane of its item's group that emits")
        body.append("  u32 tm_round = 0;")
    body.append("  while (true) {")
    body.append("    if (tm_more) {")
    free_ = "(!tm_live && !tm_pend)" if pb_h else "!tm_live"
    body.append(f"      const u64 tm_need = tm_ballot({free_});")
    if mode == "step" and refill > 1:
        body.append(f"      if (tm_need != 0ull && (__builtin_popcountll(tm_need) >= {int(refill)} || "
                    "tm_ballot(tm_live) == 0ull)) {")
    else:
        body.append("      if (tm_need != 0ull) {")
    # Claims.  One address serves ~83M returning atomics/s (12 ns each), which short items at 64 per claim reach and
    # which a launch's first claims (one per resident wave, up to 8,192) queue up for ~100 us at.  The items are
    # split into SHARDS contiguous ranges, each with a counter on its own 256-byte line; a wave claims from its home
    # range (workgroup index % SHARDS: a workgroup's XCD is its index % 8, so a range stays on one XCD and its L2)
    # and, once that is used up, from the next range that has items left, found with one load of all counters
    # (a lane each).  A wave learns that no items are left from one such load.  A launch of at most one chunk per
    # wave claims nothing: wave w takes chunk w.
    # A tape program's ranges are blocks of IL_CHUNKS chunks dealt out in turn instead (range s: blocks s, s + SHARDS, ...),
    # a chunk per claim: the rows of its tape lie in item order, and the resident waves then write and read one window
    # that moves through them, not 64.  The 68.4M-particle shower's tree adjoint, tapes of up to 16 GiB, 29.7 ms with
    # contiguous ranges, 26.3 so; the quickstart's item gradients at 4,194,304 items 1,630 us and 667 (blocks of one
    # chunk 672; slab's replay gradient at 1,048,576 519 with one, 505 with 4 or 16, 524 contiguous; transport's lost, 684
    # -> 703).
    # A wave that used up its last reservation in less than CLAIM_NS ns reserves RESERVE chunks per claim while its
    # range has more than that many chunks left per wave: a claim is a ~1 us round trip that the whole wave waits
    # for.  The pace is read from the 100 MHz real-time counter at claims only.
    resv = chunk * RESERVE
    body.append("        if (tm_cur >= tm_end) {")
    body.append("          if (tm_rv >= tm_re && tm_one) {")
    body.append("            tm_rv = (u64)tm_wid * tm_ch;")
    body.append("            tm_re = tm_rv + tm_ch < (u64)n_items ? tm_rv + tm_ch : (u64)n_items;")
    il = tape_w > 0
    body.append("          } else if (tm_rv >= tm_re) {")
    if not il:
        body.append("            const u64 tm_now = __builtin_amdgcn_s_memrealtime();")
        body.append(f"            const bool tm_big = tm_t0 != 0ull && (tm_now - tm_t0) * 10ull < tm_rc * {CLAIM_NS}ull "
                    f"&& tm_left > tm_shw * {resv}ull;")
        body.append(f"            tm_rc = tm_big ? {RESERVE}u : 1u;")
        body.append("            tm_t0 = tm_now;")
    body.append("            while (true) {")
    if il:                     # (the counter counts the range's chunks; the last block may lack some)
        body.append(f"              const u64 tm_nc = ((u64)n_items + {chunk - 1}u) / {chunk}u;")
        body.append(f"              const u64 tm_b = tm_claim(tm_shc + tm_sh * {SHARD_WORDS // 2}u, 1u);")
        body.append(f"              const u64 tm_k = (tm_b / {IL_CHUNKS}u * {SHARDS}u + tm_sh) * {IL_CHUNKS}u + tm_b % {IL_CHUNKS}u;")
        body.append("              if (tm_k < tm_nc) {")
        body.append(f"                tm_rv = tm_k * {chunk}u;")
        body.append(f"                tm_re = tm_rv + {chunk}u < (u64)n_items ? tm_rv + {chunk}u : (u64)n_items;")
        body.append("                break;")
        body.append("              }")
        body.append(f"              const u64 tm_ll = tm_range((tm_nc + {IL_CHUNKS - 1}u) / {IL_CHUNKS}u, (u32)tm_lane(), "
                    f"{SHARDS}u) * {IL_CHUNKS}u;")
    else:
        body.append("              const u64 tm_sb = tm_shn * tm_sh < (u64)n_items ? tm_shn * tm_sh : (u64)n_items;")
        body.append("              const u64 tm_sl = tm_sb + tm_shn < (u64)n_items ? tm_shn : (u64)n_items - tm_sb;")
        body.append(f"              const u64 tm_b = tm_claim(tm_shc + tm_sh * {SHARD_WORDS // 2}u, tm_rc * {chunk}u);")
        body.append("              if (tm_b < tm_sl) {")
        body.append("                tm_rv = tm_sb + tm_b;")
        body.append(f"                tm_re = tm_sb + (tm_b + tm_rc * {chunk}u < tm_sl ? tm_b + tm_rc * {chunk}u : tm_sl);")
        body.append("                tm_left = tm_sb + tm_sl - tm_re;")
        body.append("                break;")
        body.append("              }")
        body.append("              const u64 tm_lb = tm_shn * (u64)tm_lane() < (u64)n_items ? tm_shn * (u64)tm_lane() : (u64)n_items;")
        body.append("              const u64 tm_ll = tm_lb + tm_shn < (u64)n_items ? tm_shn : (u64)n_items - tm_lb;")
    body.append(f"              const u64 tm_lv = __hip_atomic_load(tm_shc + tm_lane() * {SHARD_WORDS // 2}, "
                "__ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);")
    body.append("              const u64 tm_sm = tm_ballot(tm_lv < tm_ll);")
    body.append("              if (tm_sm == 0ull) { tm_rv = (u64)n_items; tm_re = tm_rv; break; }")
    body.append("              const u64 tm_hi = tm_ballot(tm_lv < tm_ll && (u32)tm_lane() >= tm_sh);   // the next from this one on")
    body.append("              tm_sh = (u32)__builtin_ctzll(tm_hi != 0ull ? tm_hi : tm_sm);")
    body.append("              tm_rc = 1u;")
    body.append("            }")
    body.append("          }")
    body.append("          const u64 tm_b = tm_rv;")
    body.append("          if (tm_b >= (u64)n_items) {")
    body.append("            tm_more = false;")
    body.append("          } else {")
    body.append(f"            tm_cb = tm_b; tm_cur = 0u; tm_end = (u32)(tm_b + {chunk}u < tm_re ? {chunk}ull : tm_re - tm_b);")
    body.append("            tm_rv = tm_b + tm_end;")
    if W:
        body.append(f"            for (u32 q = (u32)tm_lane(); q < {chunk}u; q += 64u) {{")
        body.append("              const u64 t = tm_cb + q;")
        body.append("              if (q < tm_end) {")
        for i, off in stage_off.items():
            n = max(1, pav[i].size)
            for e in range(n):
                body.append(f"                tm_st[q * {W} + {off + e}] = ((const u32*)P.p[{i}])[t * {n} + {e}];")
        body.append("              }")
        body.append("            }")
        body.append("            __builtin_amdgcn_wave_barrier();")
    body.append("          }")
    body.append("        }")
    body.append("        if (tm_cur < tm_end) {")
    body.append("          const u32 tm_av = tm_end - tm_cur;")
    body.append("          const u32 tm_n = (u32)__builtin_popcountll(tm_need);")
    body.append(f"          if ({free_}) {{")
    body.append("            const u32 tm_r = tm_rank(tm_need);")
    body.append("            if (tm_r < tm_av) {")
    body.append("              tm_loc = tm_cur + tm_r;")
    body.append("              tm_item = (i64)(tm_cb + tm_loc);")
    body.append("              tm_live = true;")
    body += pre_lines
    if mode == "item":
        body.append("              tm_live = false;")
    body.append("            }")
    body.append("          }")
    body.append("          tm_cur += tm_n < tm_av ? tm_n : tm_av;")
    body.append("          if (tm_cur >= tm_end && (tm_one || tm_cb + tm_end >= (u64)n_items)) tm_more = false;")
    body.append("        }")
    body.append("      }")
    body.append("    }")
    # Steps until a lane is free while items are left (one step once none are): the refill's bookkeeping stays out of
    # long items' inner loop.  Wave-uniform exits only (ballots) and no `continue`, so every lane reaches the claim
    # block together: a per-lane `continue` lets the compiler's loop structurizer park idle lanes off the exec mask
    # while live lanes run the header again, and the claim and operand staging would then run with a partial wave.
    body.append("    do {")
    body.append("      if (tm_live) {")
    body += step_lines
    body.append("      }")
    if pb_h:
        # the waiting items' POST: once the wave's waiting lane-iterations reach pb_h, when no lane of the wave is
        # live, or once the queue is drained (then in the step they finish: the tail phase repacks live lanes only)
        body.append("      const u64 tm_pm = tm_ballot(tm_pend);")
        body.append("      if (tm_pm != 0ull) {")
        body.append("        tm_acc += (u32)__builtin_popcountll(tm_pm);")
        body.append(f"        if (tm_acc >= {pb_h}u || !tm_more || tm_ballot(tm_live) == 0ull) {{")
        body.append("          tm_acc = 0u;")
        body.append("          if (tm_pend) {")
        body += post_lines
        body.append("            tm_pend = false;")
        body.append("          }")
        body.append("        }")
        body.append("      }")
    if mode == "step" and refill > 1:
        body.append(f"    }} while (tm_more && __builtin_popcountll(tm_ballot({free_})) < {int(refill)} && "
                    "tm_ballot(tm_live) != 0ull);")
    else:
        body.append(f"    }} while (tm_more && tm_ballot({free_}) == 0ull);")
    if not compact_on:
        body.append("    if (tm_ballot(tm_live || tm_more) == 0ull) break;")
        body.append("  }")
    else:
        # Tail phase.  Every wave counts itself once when its queue is drained; when all are, the workgroup's waves
        # leave the claim loop and repack every `compact` iterations (a wave without live lanes goes straight to the
        # next round and waits at its barrier).  A round: live lanes write their item's loop state to the pool,
        # barrier, every wave reads the count P (the same for all), P == 0 ends the loop for the whole workgroup,
        # else wave w takes pool items 64 w .. 64 w + 63, barrier.  The two counters alternate: round r counts into
        # tm_pn[r & 1] and clears the other, whose last readers finished before this round's first barrier.  Every
        # wave runs the same number of rounds, and the loop has no other exit.
        body.append("    if (!tm_more) {")
        body.append("      if (!tm_dr) {")
        body.append("        tm_dr = true;")
        body.append("        if (tm_lane() == 0u) atomicAdd(&tm_ndr, 1u);")
        body.append("      }")
        body.append(f"      if (__builtin_amdgcn_readfirstlane(__atomic_load_n(&tm_ndr, __ATOMIC_RELAXED)) == {wpb}u) break;")
        body.append("    }")
        body.append("  }")
        body.append("  while (true) {")
        body.append("    u32* const tm_cnt = &tm_pn[tm_round & 1u];")
        body.append(f"    const u64 tm_lm = tm_ballot(tm_live{' && tm_lead' if pl_ahead else ''});")
        body.append("    u32 tm_pb = 0u;")
        body.append("    if (tm_lane() == 0u) tm_pb = atomicAdd(tm_cnt, (u32)__builtin_popcountll(tm_lm));")
        body.append("    tm_pb = __builtin_amdgcn_readfirstlane(tm_pb);")
        body.append("    if (tm_live && tm_lead) {" if pl_ahead else "    if (tm_live) {")
        body.append("      const u32 q = tm_pb + (u32)tm_rank(tm_lm);")
        body += ["      " + ln for ln in pack]
        body.append("    }")
        body.append("    tm_live = false;")
        body.append("    __syncthreads();")
        body.append("    const u32 tm_P = __builtin_amdgcn_readfirstlane(*tm_cnt);")
        body.append("    if (tm_P == 0u) break;")
        body.append("    if (threadIdx.x == 0) tm_pn[(tm_round + 1u) & 1u] = 0u;")
        if pl_ahead:
            body.append("    u32 tm_gs = 0u;")
            body.append("    while (tm_gs < 6u && (tm_P << (tm_gs + 1u)) <= TM_BLOCK) ++tm_gs;")
            body.append("    const u32 tm_g = 1u << tm_gs, tm_go = (u32)tm_lane() & (tm_g - 1u);")
            body.append("    tm_lead = tm_go == 0u;")
        body.append("    {")
        body.append("      const u32 q = threadIdx.x >> tm_gs;" if pl_ahead else "      const u32 q = threadIdx.x;")
        body.append("      if (q < tm_P) {")
        body += ["        " + ln for ln in unpack]
        body.append("        tm_live = true;")
        body.append("      }")
        body.append("    }")
        body.append("    __syncthreads();")
        body.append("    ++tm_round;")
        if pl_ahead is None:
            body.append(f"    for (u32 tm_it = 0u; tm_it < {compact}u && tm_ballot(tm_live) != 0ull; ++tm_it) {{")
            body.append("      if (tm_live) {")
            body += tail_lines
            body.append("      }")
            body.append("    }")
        else:
            # Groups of tm_g lanes hold an item each (a power of two, 1 .. 64, from the items left), every lane of a
            # group with the same state; one of them emits and writes.  With at most an item per wave left a round
            # ends with the wave's item.  The cross-lane reads (ds_bpermute, the next update's issued before this
            # one's work) stand outside any lane-dependent branch: all lanes of the wave are active there.
            head, upd, nw = tail_lines
            body.append(f"    const u32 tm_nb = tm_P <= {wpb}u ? ~0u : ({compact}u >> tm_gs) + ({compact}u >> tm_gs == 0u ? 1u : 0u);")
            body.append("    const int tm_ba = (int)(((u32)tm_lane() & ~(tm_g - 1u)) * 4u);")
            body.append("    for (u32 tm_it = 0u; tm_it < tm_nb && tm_ballot(tm_live) != 0ull; ++tm_it) {")
            body += [f"      u32 tm_h{i} = 0u;" for i in range(nw)]
            body.append("      if (tm_live) {")
            body += head
            body.append("      }")
            body += [f"      u32 tm_n{i} = (u32)__builtin_amdgcn_ds_bpermute(tm_ba, (int)tm_h{i});" for i in range(nw)]
            body.append("      for (u32 tm_j = 1u; tm_j <= tm_g && tm_ballot(tm_live) != 0ull; ++tm_j) {")
            body += [f"        const u32 tm_q{i} = tm_n{i};" for i in range(nw)]
            body += [f"        tm_n{i} = (u32)__builtin_amdgcn_ds_bpermute(tm_ba + (int)((tm_j & (tm_g - 1u)) * 4u), "
                     f"(int)tm_h{i});" for i in range(nw)]
            body += upd
            body.append("      }")
            body.append("    }")
        body.append("  }")
    if QS:                     # the wave's staged children that are left
        body.append("  {")
        body.append("    const u32 tm_sq = tm_qn[threadIdx.x >> 6];")
        body.append("    if (tm_sq != 0u) {")
        body += ["      " + ln for ln in _qflush_lines("tm_sq")]
        body.append("    }")
        body.append("  }")
    body.append("  if (tm_drop) atomicAdd(&TM_STATS[4], tm_drop);")
    for ri in rec_info:        # each wave: its records into the exact count, its last batch's unused slots keyed 0
        j, w = ri["ctr"], block // 64
        rc = f"((u64*)P.p[{r_rctr}] + {RC_WORDS // 2 * j})"
        body.append("  {")
        body.append(f"    const u64 tm_c = tm_rcnt{j}[threadIdx.x >> 6], tm_b = tm_rbase{j}[threadIdx.x >> 6];")
        body.append(f"    const u32 tm_l = tm_rleft{j}[threadIdx.x >> 6];")
        body.append("    for (u32 q = (u32)tm_lane(); q < tm_l; q += 64u) {")
        body.append("      const u64 s = tm_b + (TM_RB - tm_l) + q;")
        body.append(f"      if (s < tm_rawcap{j}) ((i32*)P.p[{r_out[ri['ki']]}])[s] = 0;")
        body.append("    }")
        body.append(f"    if ((threadIdx.x & 63u) == 0u && tm_c != 0ull) atomicAdd(&{rc}[{RC_TOTAL}], tm_c);")
        body.append(f"    if (blockIdx.x == 0u && threadIdx.x == 0u) {rc}[{RC_TOTAL + 1}] = (u64)tm_grid * {w}u;")
        body.append("  }")
    body.append("  if (tm_ntr) atomicAdd(&TM_CTL[2], tm_ntr);")
    ldecl = []
    for k in rpriv:             # each lane's register copy into the workgroup's (LDS) one
        s = prog.tallies[k]
        ct = ctype(s.dtype)
        for b in range(s.S):
            if s.dtype == C.F32:
                ldecl.append(f"  float tm_r{k}_{b} = 0.0f;")
                add = f"atomicAdd(&tm_sh{k}[{copy_of(b, ncopy[k])}], (double)tm_r{k}_{b})" if k in d64 else (
                    f"tm_ladd_f32(&tm_sh{k}[{b}], tm_r{k}_{b})")
                body.append(f"  if (tm_r{k}_{b} != 0.0f) {add};")
            else:
                ldecl.append(f"  {ct} tm_r{k}_{b} = 0;")
                body.append(f"  if (tm_r{k}_{b} != 0) atomicAdd(&tm_sh{k}[{b}], tm_r{k}_{b});")
    for (k, cbits), (names, c) in rcounts.items():
        key = (k, cbits)
        if key not in counts:          # (the workgroup's counters of this constant: the lanes' counts land there)
            counts[key] = (f"tm_cn{k}_{len(counts)}", c)
        for b, nm in enumerate(names):
            ldecl.append(f"  u32 {nm} = 0u;")
            body.append(f"  if ({nm} != 0u) atomicAdd(&{counts[key][0]}[TM_CN{k}({b})], (u64){nm});")
    body[body.index("//TM_LANE_DECLS")] = "\n".join(ldecl)
    # the constants' counters share the copies' words with the sums: every constant of a tally has the same number
    ccopy = {}
    for k in sorted({k for k, _ in counts}):
        S, n = prog.tallies[k].S, sum(kk == k for kk, _ in counts)
        ccopy[k] = copies(S, room // n)
        room -= S * n * ccopy[k] if ccopy[k] > 1 else 0
        src.append(f"#define TM_CN{k}(e) ({copy_of('(e)', ccopy[k])})")
    if priv:
        body.append("  __syncthreads();")
        if wide:
            body.append("  const bool tm_wide = __builtin_amdgcn_readfirstlane(tm_spread_s) != 0u;")
        for k in priv:
            s = prog.tallies[k]
            if s.exact:
                nw = XW * s.S
                gw = f"((u64*)P.p[{r_scr[k]}])"
                gf = f"((u32*)P.p[{r_scr[k]}] + {2 * XW * s.S})"
                body.append(f"  for (int i = threadIdx.x; i < {nw}; i += TM_BLOCK) {{ const i64 x = (i64)tm_xsh{k}[i]; "
                            f"if (x != 0 && tm_xadd(&{gw}[i / {XW} * {XW}], i % {XW}, x)) "
                            f"atomicOr(&{gf}[(i / {XW}) >> 5], 1u << ((i / {XW}) & 31)); }}")
                body.append(f"  for (int i = threadIdx.x; i < {(s.S + 31) // 32}; i += TM_BLOCK) "
                            f"if (tm_xfl{k}[i]) atomicOr(&{gf}[i], tm_xfl{k}[i]);")
            elif s.fixed:
                # a block's copy: its low word added with the carry it makes, plus the block's own carries
                glo = f"((u64*)P.p[{r_scr[k]}])"
                gc = f"((i32*)P.p[{r_scr[k]}] + {2 * s.S})"
                body.append(f"  for (int i = threadIdx.x; i < {s.S}; i += TM_BLOCK) {{ const u64 x = tm_wsh{k}[i]; "
                            f"const i32 c = tm_wsc{k}[i]; if (x != 0ull) tm_wadd(&{glo}[i], &{gc}[i], (i64)x); "
                            f"if (c != 0) atomicAdd(&{gc}[i], c); }}")
            elif s.dtype == C.F64:
                body.append(f"  for (int i = threadIdx.x; i < {s.S}; i += TM_BLOCK) {{ const double x = {sum_copies(f'tm_sh{k}', ncopy[k])}; "
                            f"if (x != 0.0) tm_gadd_f64(&((double*)P.p[{r_out[k]}])[i], x); }}")
            elif s.dtype in (C.I64, C.U64):
                ct = ctype(s.dtype)
                body.append(f"  for (int i = threadIdx.x; i < {s.S}; i += TM_BLOCK) {{ const {ct} x = tm_sh{k}[i]; "
                            f"if (x != 0) tm_gadd_u64(&((u64*)P.p[{r_out[k]}])[i], (u64)x); }}")
            elif s.dtype == C.F32:
                gw = f"(double*)P.p[{r_ctl}] + {wide[k]} + i" if k in wide else None
                go = f"&((float*)P.p[{r_out[k]}])[i]"

                def flush(total, cond, x32, x64):
                    """add bin i's total of the workgroup to the launch's."""
                    add = f"tm_gadd_f32({go}, {x32});"
                    if gw is not None:
                        add = f"{{ if (tm_wide) tm_gadd_f64({gw}, {x64}); else {add} }}"
                    body.append(f"  for (int i = threadIdx.x; i < {s.S}; i += TM_BLOCK) {{ const {total}; if ({cond}) {add} }}")
                flush(f"{'double' if k in d64 else 'float'} x = {sum_copies(f'tm_sh{k}', ncopy.get(k, 1))}", "x != 0.0f",
                      "(float)x", "x")
                for (kk, _), (nm, c) in counts.items():
                    if kk == k:
                        flush(f"u64 n = {sum_copies(nm, ccopy[k])}", "n != 0ull", f"tm_u64_f32(n) * {lit(c, np.float32)}",
                              f"(double)n * {lit(c, np.float64)}")
            else:
                ct = ctype(s.dtype)
                body.append(f"  for (int i = threadIdx.x; i < {s.S}; i += TM_BLOCK) {{ const {ct} x = tm_sh{k}[i]; "
                            f"if (x != 0) atomicAdd(&(({ct}*)P.p[{r_out[k]}])[i], x); }}")
    body.append("}")
    cdecl = []
    for (k, _), (nm, c) in counts.items():
        S = prog.tallies[k].S * ccopy[k]
        cdecl.append(f"  __shared__ u64 {nm}[{S}];")
        cdecl.append(f"  for (int i = threadIdx.x; i < {S}; i += TM_BLOCK) {nm}[i] = 0ull;")
    body[body.index("//TM_COUNT_DECLS")] = "\n".join(cdecl)
    if not lean and lds_bytes("\n".join(body)) > LDS_MAX:
        return build(prog, **opts, lean=True)
    src.append("\n".join(body))
    aux = []
    # any truncation or any Records output past its capacity: every float output NaN, every integer record field -1
    rbad = " || ".join((["TM_CTL[2] != 0u"] if prog.trunc is not None else [])
                       + [f"((const u64*)P.p[{r_rctr}])[{RC_WORDS // 2 * ri['ctr'] + RC_TOTAL}] > {ri['capacity']}ull"
                          for ri in rec_info])
    for ri in rec_info:
        src.append(_records_passes(ri, r_rctr, r_out, r_ys[ri["count"]], r_rex, r_rbs, prog, rbad))
        j = ri["ctr"]
        cap = ri["capacity"]
        aux += [(f"tm_rscan{j}", "items", 1024, cap),
                (f"tm_rtop{j}", "one", 1024, cap), (f"tm_rcanon{j}", "cap", 256, cap)]
    L = Layout(n_in=n_in, res=res, n_zero=n_zero, r_out=r_out, r_ctl=r_ctl, r_stats=r_stats, r_ys=r_ys,
               flags=flags, mode=mode, priv=priv, zero_words=zero_words, r_q=r_q,
               records=[dict(name=ri["name"], capacity=ri["capacity"], r_ctr=(r_rctr, RC_WORDS // 2 * ri["ctr"] + RC_TOTAL),
                             fields={f: rr for f, (_, rr) in ri["fields"].items()}) for ri in rec_info], aux=aux,
               scratch=sorted(r_scr.values()) + ([] if wide else [r_ctl]), n_claim=n_claim,
               emitted=emitted, spread=SPREAD if pl_ahead else 0)
    return "\n".join(src) + "\n", L
