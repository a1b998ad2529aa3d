"""Row programs: runs of row-wise graph ops planned as one anvil_row_program launch.

An op is row-wise when row t of its result depends on row t of its operands only: rmsnorm_int, qlinear (a const right
operand), add_requant, lut and lut_mul over values of dims [T, width]. In a block everything but attention is: rmsnorm
-> q, k, v, and y -> residual add -> rmsnorm -> MLP -> residual add -> the next rmsnorm -> q, k, v (or the logits).
find() splits a proven graph into maximal runs of such ops between the others; plan() lays one run out for the kernel
(LDS slots, weight stream, results written to memory when something outside the run reads them or the caller asked for
them) and emits its step.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np

from . import ir as g
from . import runtime as rt

SLOTS_MAX, OPS_MAX, TABLES_MAX = 64, 24, 4      # include/anvil_mi355x.h, with the next two
LUT_MAX = 4096               # entries of a rsqrt table
LDS_MAX = 96 << 10           # a wave's slots, the tables and the weight stream
WIDTH_MAX = 256              # of any value of a program
BLOCK = 32                   # rows of a wave's tile, columns of a value's slot, K bytes of a weight fragment

# fragment row i of a weight block is result column ORDER[i] of the block (include/anvil_mi355x.h, anvil_row_create)
ORDER = np.array([16 * ((i >> 2) & 1) + 4 * (i >> 3) + (i & 3) for i in range(32)])


def pack_weights(bt: np.ndarray) -> np.ndarray:
    """A transposed weight (N, K) int8 as its part of the weight stream: zero-padded to whole blocks, one KiB a
    fragment, [N / 32][K / 32][lane = 32 half + i][16]."""
    N, K = bt.shape
    Nb, Kb = -(-N // BLOCK), -(-K // BLOCK)
    w = np.zeros((Nb * BLOCK, Kb * BLOCK), np.int8)
    w[:N, :K] = bt
    w = w.reshape(Nb, BLOCK, Kb, BLOCK)[:, ORDER].reshape(Nb, BLOCK, Kb, 2, 16)
    return np.ascontiguousarray(w.transpose(0, 2, 3, 1, 4))


class Program:
    """The ops of one run, in graph order."""

    def __init__(self, ops):
        self.ops = ops

    def __repr__(self):
        return "+".join(op.sym_str or op.name for op in self.ops)


def _product_min(rows) -> int:
    """The bound on the smaller of a product's K and N. A program trades launches for a chain of ops that each wave runs
    in turn, so it gains where its products are small. Measured on 256 CUs: 32-wide blocks (hidden width 128) took 19 us
    against 21 op by op at 16 rows, 27 against 46 at 65,536 and 116 against 207 in two layers of 131,072; the frozen
    32-wide models 39 against 57 at 32 rows and 123 against 242 at 262,144. 64-wide blocks gain once four row blocks a CU
    hide the chain: 46 against 56 at 32,768 rows (42 against 46 in longer sequences), but 30 against 25 at 32 rows and 31
    against 26 at 2,048; between those two the line was not measured. From widths of 96 on programs lost at every
    size."""
    return 64 if rows >= 32768 else 32


def _eligible(cm, op, nb) -> bool:
    """Whether a proven graph's op can be part of a row program over nb sequences."""
    r = op.results[0] if op.results else None
    if r is None or r in cm.is_const:
        return False
    t = g.qt(r)
    if len(t.dims) != 2 or t.dims[1] % 16 or not 16 <= t.dims[1] <= WIDTH_MAX or t.dtype not in ("i8", "i16"):
        return False
    row = lambda v: (v not in cm.is_const and len(g.qt(v).dims) == 2 and g.qt(v).dims[0] == t.dims[0]   # noqa: E731
                     and g.qt(v).dims[1] % 16 == 0 and 16 <= g.qt(v).dims[1] <= WIDTH_MAX
                     and g.qt(v).dtype in ("i8", "i16"))
    if isinstance(op, (g.QLinearOp, g.QMatmulOp)):
        return (row(op.a) and op.b in cm.is_const and len(g.qt(op.b).dims) == 2
                and min(g.qt(op.a).dims[1], t.dims[1]) <= _product_min(nb * t.dims[0])
                and (op.lut is None or isinstance(op.lut.owner, g.ConstOp)))
    if isinstance(op, g.RmsNormIntOp):
        w, lut = cm._const_array(op.w), cm._const_array(op.lut)
        if w is None or lut is None or not 1 <= lut.size <= LUT_MAX or lut.size % 4 or int(lut.min()) < 0 or not row(op.x):
            return False
        if g.qt(op.x).dtype == "i8" and (op.ss_shift_int or op.ss_init_int):
            return False
        return int(lut.max()) * abs(int(op.M)) < 1 << 23
    if isinstance(op, g.AddRequantOp):
        return row(op.a) and row(op.b)
    if isinstance(op, g.LutOp):
        return row(op.x) and isinstance(op.table.owner, g.ConstOp)
    if isinstance(op, g.LutMulOp):
        return row(op.x) and row(op.y) and isinstance(op.table.owner, g.ConstOp)
    return False


def _row_operands(op) -> list:
    """The operands an op reads by rows."""
    if isinstance(op, (g.QLinearOp, g.QMatmulOp)):
        return [op.a]
    if isinstance(op, g.AddRequantOp):
        return [op.a, op.b]
    if isinstance(op, g.LutMulOp):
        return [op.x, op.y]
    return [op.x]


def find(cm, nb) -> list:
    """The graph's runs of at least two row-wise ops, a product among them. A run is planned where its first op stands, so
    its ops may read only what is planned by then: each other's results, and values from before it. Graph inputs and views
    (transposes, reshapes) inside a run cost no launch: it goes on past them until an op reads one."""
    if not cm.proven:
        return []
    progs, cur, T = [], [], None
    late = set()                        # inputs and views that stand inside the open run

    def close():
        nonlocal cur
        if len(cur) > 1 and any(isinstance(op, (g.QLinearOp, g.QMatmulOp)) for op in cur):
            progs.append(Program(cur))
        cur = []
        late.clear()

    for op in cm.ops:
        if isinstance(op, g.ConstOp):
            continue
        r = op.results[0]
        if isinstance(op, (g.InputOp, g.TransposeOp, g.ReshapeOp)):
            if cur:
                late.add(r)
            continue
        if not _eligible(cm, op, nb):
            close()
            continue
        rows = g.qt(r).dims[0]
        if (cur and rows != T) or any(v in late for v in _row_operands(op)):
            close()
        T = rows
        cur.append(op)
    close()
    return progs


class _Slots:
    """LDS slots (KiB) of one wave: first fit, freed at a value's last use."""

    def __init__(self):
        self.used = []                                      # (first, end) of live values

    def take(self, n) -> int:
        at = 0
        for lo, hi in sorted(self.used):
            if lo - at >= n:
                break
            at = max(at, hi)
        self.used.append((at, at + n))
        return at

    def free(self, at, n):
        self.used.remove((at, at + n))

    @property
    def top(self):
        return max((hi for _, hi in self.used), default=0)


def layout(cm, prog, external) -> dict | None:
    """The kernel's op list without pointers: dicts of its integer fields, plus the values each one reads from or
    writes to memory; None when the program does not fit its limits. `external` holds the values read elsewhere."""
    chunks = lambda v: -(-g.qt(v).dims[1] // BLOCK) * (2 if g.qt(v).dtype == "i16" else 1)   # noqa: E731
    wide = lambda v: int(g.qt(v).dtype == "i16")                                        # noqa: E731
    members = {op.results[0] for op in prog.ops}
    last = {}
    for i, op in enumerate(prog.ops):
        for v in _row_operands(op):
            last[v] = i
    slots, at, top, out, tables, stream, lds = _Slots(), {}, 0, [], [], [], 0

    def table(v):
        if v not in tables:
            tables.append(v)
        return tables.index(v)

    def place(v):
        nonlocal top
        at[v] = slots.take(chunks(v))
        top = max(top, slots.top)
        return at[v]

    for v in dict.fromkeys(v for op in prog.ops for v in _row_operands(op)):
        if v not in members:                                # computed outside the program: loaded first, all together
            out.append(dict(kind=rt.ROW_LOAD, n=g.qt(v).dims[1], dst=place(v), wide=wide(v), load=v))
    for i, op in enumerate(prog.ops):
        r = op.results[0]
        n = g.qt(r).dims[1]
        reads = _row_operands(op)
        d = dict(n=n, wide=wide(r), wide_a=wide(reads[0]), a=at[reads[0]], table=-1, value=r)
        trans = cm.phys.get(r) == [1, 0]
        if trans and (r in last or wide(r) or not isinstance(op, (g.QLinearOp, g.QMatmulOp))):
            return None
        if isinstance(op, (g.QLinearOp, g.QMatmulOp)):
            K = g.qt(op.a).dims[1]
            if wide(op.a):
                return None
            m24 = cm.acc_bounds.get(r, 1 << 31) < 1 << 23 and abs(int(op.M)) < 1 << 23
            d.update(kind=rt.ROW_GEMM, k=-(-K // BLOCK), mult=int(op.M), shift=int(op.s), m24=int(m24), trans=int(trans))
            if op.lut is not None:
                d["table"] = table(op.lut)
            stream.append(op)
            lds += 1024 * d["k"] * -(-n // BLOCK)
        elif isinstance(op, g.RmsNormIntOp):
            d.update(kind=rt.ROW_NORM, mult=int(op.M), shift=int(op.s), c=op.ss_shift_int, e=op.ss_init_int, norm=op)
            lds += 1024 * (1 + -(-4 * math.prod(g.qt(op.lut).dims) // 1024))
        elif isinstance(op, g.AddRequantOp):
            ma, mb = int(op.Ma), int(op.Mb)
            lim = 1 << 23 if d["wide"] or d["wide_a"] or wide(op.b) else 1 << 24
            d.update(kind=rt.ROW_ADD, mult=ma, mult2=mb, shift=int(op.s), b=at[op.b], wide_b=wide(op.b),
                     m24=int(max(abs(ma), abs(mb)) < lim))
        elif isinstance(op, g.LutOp):
            d.update(kind=rt.ROW_LUT, table=table(op.table))
        else:
            d.update(kind=rt.ROW_LUT_MUL, mult=int(op.M), shift=int(op.s), b=at[op.y], table=table(op.table),
                     m24=int(abs(int(op.M)) < 1 << 23))
        if not trans:
            # an element-wise op may write over an operand of the same size that nothing reads any more
            old = [v for v in dict.fromkeys(reads) if last[v] == i and chunks(v) == chunks(r) and wide(v) == wide(r)]
            if old and d["kind"] != rt.ROW_GEMM:
                at[r] = d["dst"] = at.pop(old[0])
            else:
                d["dst"] = place(r)
        d["store"] = r in external
        out.append(d)
        for v in dict.fromkeys([*reads, r]):
            if v in at and last.get(v, -1) <= i and (v in members or v in reads):
                slots.free(at[v], chunks(v))
                del at[v]
    if top > SLOTS_MAX or len(out) > OPS_MAX or len(tables) > TABLES_MAX \
            or lds + 256 * TABLES_MAX + 1024 * top > LDS_MAX:
        return None
    return dict(ops=out, tables=tables, stream=stream)


def _memory(view, rows, n):
    """(view, ld, kb) of a value's rows in memory, or None when they are not rows of one stride in order."""
    flat = view.reshape((rows, n))
    if flat is None or flat.strides[-1] != 1:
        return None
    unit = 16 // flat.itemsize
    if flat.kb > 64:
        ld, kb = 64, flat.kb
    else:                                                   # K blocks of one row (kb = 64) follow each other: row-major
        ld, kb = (flat.strides[0] if rows > 1 else -(-n // unit) * unit), 64
    if ld % unit or kb % 16 or flat.offset % unit or (flat.kb and flat.itemsize != 1):
        return None
    if kb == 64 and ld < n:
        return None
    return flat, ld, kb


class Launch:
    """One planned program: the op list with its buffers, and its weight stream on the device."""

    def __init__(self, cm, prog, lay, rows, seq, stream):
        self.cm, self.prog, self.lay, self.rows, self.seq, self.stream = cm, prog, lay, rows, seq, stream
        self.mem = []                                       # per op: (view, ld, kb) in memory, or None
        self.program = None

    def desc(self):
        """The C op list, the table pointers and their number."""
        arr = (rt.RowOp * len(self.lay["ops"]))()
        for o, d, mem in zip(arr, self.lay["ops"], self.mem):
            for f in ("kind", "a", "b", "dst", "n", "k", "table", "m24", "wide", "wide_a", "wide_b", "trans", "mult", "mult2",
                      "shift", "c", "e"):
                setattr(o, f, d.get(f, -1 if f == "table" else 0))
            if mem is not None:
                view, o.ld, o.kb = mem
                if "load" in d:
                    setattr(o, "in", view.ptr)
                else:
                    o.out = view.ptr
            if "norm" in d:
                w, lut = (self.cm._const_views[v] for v in (d["norm"].w, d["norm"].lut))
                setattr(o, "in", w.ptr)
                o.lut, o.lut_len = lut.ptr, lut.size
        tabs = [self.cm._const_views[v] for v in self.lay["tables"]]
        return arr, (C.c_void_p * max(1, len(tabs)))(*[t.ptr for t in tabs]), len(tabs)

    def work(self):
        """(kind, int ops, bytes) as driver._work counts them: operands and stored results once, weights once."""
        ops = nbytes = 0
        for d, mem in zip(self.lay["ops"], self.mem):
            if d["kind"] == rt.ROW_GEMM:
                K = g.qt(self._op(d["value"]).a).dims[1]
                ops += 2 * self.rows * d["n"] * K
                nbytes += d["n"] * K
            if mem is not None:
                nbytes += self.rows * d["n"] * (2 if d["wide"] else 1)
            if "norm" in d:
                nbytes += d["n"] + 4 * self.cm._const_views[d["norm"].lut].size
        return "gemm", ops, nbytes

    def _op(self, value):
        return value.owner


def call(dev, launch):
    if launch.program is None:                              # once its buffers are allocated
        arr, ptrs, ntab = launch.desc()
        launch.program = dev.row_program(arr, launch.rows, launch.seq, launch.stream, ptrs, ntab)
    launch.program.launch()


def plan(cm, P, prog, views, nb, keep, step) -> bool:
    """Plan a program's step and its results' views; False when it has to run op by op."""
    T = g.qt(prog.ops[0].results[0]).dims[0]
    rows = nb * T
    if any(op in P.fused_adds or op in P.fused_norms for op in prog.ops):   # part of it runs in an earlier epilogue
        return False
    members = {op.results[0] for op in prog.ops}
    inside = set(prog.ops)
    external = {v for v in members if keep == "all" or v in cm.output_values
                or any(u not in inside for u in cm.users.get(v, []))}
    lay = layout(cm, prog, external)
    if lay is None:
        return False
    mem, results, nbufs = [], {}, len(P.bufs)
    for d in lay["ops"]:                                    # operands and stored results
        m = None
        if "load" in d:
            m = _memory(views[d["load"]], rows, d["n"])
        elif d["store"]:
            r = d["value"]
            view = results[r] = cm._alloc_result(P, r.owner, (nb, *g.qt(r).dims), r.owner.sym_str or "row")
            m = (view, view.strides[-1], view.strides[0]) if d.get("trans") else _memory(view, rows, d["n"])
        if m is None and ("load" in d or d["store"]):       # no rows of one stride: nothing is kept of the program
            del P.bufs[nbufs:]
            return False
        mem.append(m)
    views.update(results)
    launch = Launch(cm, prog, lay, rows, T, cm._row_stream(lay))
    launch.mem = mem
    step("+".join(op.sym_str or op.name.split(".")[-1] for op in prog.ops), call, cm.dev, launch)
    for op in prog.ops:
        if isinstance(op, g.AddRequantOp):
            P.fused_adds.add(op)
    return True
