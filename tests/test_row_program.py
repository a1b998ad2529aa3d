"""Row programs (anvil_row_create): the planner's runs of row-wise ops on a CPU stand-in that decodes the weight stream
lane by lane, and the kernels against the oracle at tile edges, widths and sequence lengths where they can go wrong."""
import gzip
import json
import math

import numpy as np
import pytest

import anvil_mi355x
import fake_device
import helpers
from anvil_mi355x import models, rowprog
from anvil_mi355x import runtime as rt
from anvil_mi355x.ir import GraphBuilder
from oracle import interp
from oracle import semantics as sem


class RowFakeProgram:
    def __init__(self, dev, args):
        self.dev, self.args = dev, args

    def launch(self):
        self.dev.run_row_program(*self.args)


class RowFake(fake_device.FakeDevice):
    """The stand-in with anvil_row_program, op by op on the oracle, from the C structs."""

    def row_program(self, *args):
        self.check_program(*args)
        return RowFakeProgram(self, args)

    @staticmethod
    def check_program(ops, rows, seq, stream, tables, ntables):
        """What anvil_row_create refuses."""
        assert 1 <= len(ops) <= rowprog.OPS_MAX and 0 <= ntables <= rowprog.TABLES_MAX
        assert rows >= 1 and seq >= 1 and rows % seq == 0 and rows < (1 << 31) - 32
        top = norm = frags = 0
        for i, o in enumerate(ops):
            gemm, load = o.kind == rt.ROW_GEMM, o.kind == rt.ROW_LOAD
            trans, only8 = gemm and o.trans, o.kind in (rt.ROW_LUT, rt.ROW_LUT_MUL)
            chunks = -(-o.n // 32)
            assert 16 <= o.n <= 4096 and o.n % 16 == 0 and 0 <= o.shift <= 31
            values = [] if trans else [(o.dst, chunks, o.wide)]
            values += [] if load else [(o.a, o.k if gemm else chunks, o.wide_a)]
            values += [(o.b, chunks, o.wide_b)] if o.kind in (rt.ROW_ADD, rt.ROW_LUT_MUL) else []
            for at, n, wide in values:
                assert 0 <= at and at + n * (1 + wide) <= rowprog.SLOTS_MAX
                top = max(top, at + n * (1 + wide))
            assert not load or all(p.kind == rt.ROW_LOAD for p in ops[:i])
            assert not (only8 and (o.wide or o.wide_a or o.wide_b)) and not (o.kind == rt.ROW_NORM and o.wide)
            assert not (gemm and o.wide_a) and not (trans and o.wide)
            if gemm:
                assert 1 <= o.k <= rowprog.SLOTS_MAX and o.table < ntables and not (o.table >= 0 and o.wide)
                frags += chunks * o.k
            assert not only8 or 0 <= o.table < ntables
            if o.m24 and o.kind == rt.ROW_ADD:
                assert max(abs(o.mult), abs(o.mult2)) < 1 << (23 if o.wide or o.wide_a or o.wide_b else 24)
            elif o.m24:
                assert abs(o.mult) < 1 << 23
            src = getattr(o, "in")
            if load:
                assert src and src % 16 == 0
            if o.kind == rt.ROW_NORM:
                assert src and src % 16 == 0 and o.lut and 1 <= o.lut_len <= rowprog.LUT_MAX and o.lut_len % 4 == 0
                assert 0 <= o.c <= 30 and o.e >= 0
                norm += 1024 * (-(-4 * o.lut_len // 1024) + -(-o.n // 1024))
            if trans:
                assert o.out and o.out % 4 == 0 and o.ld % 4 == 0 and o.kb % 4 == 0 and o.ld >= seq and o.kb >= 0
            elif o.out or load:
                assert (o.out or 0) % 16 == 0 and o.ld * (1 + o.wide) % 16 == 0 and o.kb % 16 == 0 and o.ld <= 1 << 24
                blocked = not o.wide and o.kb != 64
                assert (o.ld == 64 and o.kb >= rows * 64) if blocked else o.ld >= o.n
        assert all(tables[i] and tables[i] % 4 == 0 for i in range(ntables))
        assert 1024 * frags == (stream.nbytes if stream is not None else 0)
        assert 256 * rowprog.TABLES_MAX + norm + 1024 * (frags + top) <= rowprog.LDS_MAX

    def run_row_program(self, ops, rows, seq, stream, tables, ntables):
        self.calls.append(("row_program", rows, seq, len(ops)))
        nb = 32
        left = self._raw(stream, np.int8, stream.nbytes) if stream is not None else np.zeros(0, np.int8)
        tabs = [self.view(tables[i], "i8", (256,), (1,)).astype(np.int64) for i in range(ntables)]
        slots = {}

        def put(o, v):
            dt = "i16" if o.wide else "i8"
            n = -(-o.n // nb) * (1 + o.wide)
            assert o.dst >= 0 and o.dst + n <= rowprog.SLOTS_MAX
            for k in [k for k, (m, _) in slots.items() if k < o.dst + n and o.dst < k + m]:
                del slots[k]                              # overwritten
            slots[o.dst] = (n, v)
            if o.out and not o.trans:
                if o.wide or o.kb == 64:
                    self.store(o.out, dt, (rows, o.n), (o.ld, 1), v)
                else:
                    self.store(o.out, dt, (rows, -(-o.n // 64), 64), (64, o.kb, 1), v.reshape(rows, -1, 64))

        for o in ops:
            a = slots[o.a][1] if o.kind != rt.ROW_LOAD else None
            if o.kind == rt.ROW_LOAD:
                src = getattr(o, "in")
                if o.wide or o.kb == 64:
                    put(o, self.view(src, "i16" if o.wide else "i8", (rows, o.n), (o.ld, 1)).astype(np.int64))
                else:
                    v = self.view(src, "i8", (rows, o.n // 64, 64), (64, o.kb, 1)).astype(np.int64)
                    put(o, v.reshape(rows, o.n))
            elif o.kind == rt.ROW_NORM:
                w = self.view(getattr(o, "in"), "i8", (o.n,), (1,)).astype(np.int64)
                lut = self.view(o.lut, "i32", (o.lut_len,), (1,)).astype(np.int64)
                put(o, sem.rmsnorm_wide(a, w, lut, o.mult, o.shift, o.c, o.e, "i16" if o.wide_a else "i8"))
            elif o.kind == rt.ROW_GEMM:
                K, N = o.k * nb, -(-o.n // nb) * nb
                W = np.zeros((N, K), np.int64)
                for j in range(N // nb):
                    for k in range(o.k):
                        frag, left = left[:1024].reshape(64, 16), left[1024:]
                        for lane in range(64):
                            i = lane % 32
                            col = 16 * ((i >> 2) & 1) + 4 * (i >> 3) + (i & 3)
                            W[32 * j + col, 32 * k + 16 * (lane // 32):32 * k + 16 * (lane // 32) + 16] = frag[lane]
                x = np.zeros((rows, K), np.int64)
                x[:, :a.shape[1]] = a
                y = sem.qmatmul(x, W.T, o.mult, o.shift, tabs[o.table] if o.table >= 0 else None,
                                "i16" if o.wide else "i8")[:, :o.n]
                if o.trans:
                    self.store(o.out, "i8", (rows // seq, o.n, seq), (o.kb, o.ld, 1),
                               y.reshape(-1, seq, o.n).transpose(0, 2, 1))
                else:
                    put(o, y)
            elif o.kind == rt.ROW_ADD:
                put(o, sem.add_requant(a, slots[o.b][1], o.mult, o.mult2, o.shift, "i16" if o.wide else "i8"))
            elif o.kind == rt.ROW_LUT:
                put(o, sem.lut_i8(a, tabs[o.table]))
            else:
                put(o, sem.swiglu_lut(a, slots[o.b][1], tabs[o.table], o.mult, o.shift))
        assert left.size == 0


def frozen(model):
    with gzip.open(helpers.ROOT / "tests" / "golden" / f"model_graph_{model}.json.gz", "rt") as f:
        body = json.load(f)
    return anvil_mi355x.parse_ir(body["ir"]), {k: np.asarray(v, dtype=np.int64).reshape(body["shapes"][k])
                                               for k, v in body["consts"].items()}


def check(module, consts, model, x, keep, quantized):
    cm = anvil_mi355x.compile(model)
    res = cm.run(x, "mi355x", batch=True, keep=keep, quantized=quantized)
    xq = x if quantized else cm.quantize_input(x)
    want = interp.run(module, {cm.inputs[0]: xq}, consts, batch=True, fast=True)
    for k in res.ints:
        assert np.array_equal(res.ints[k], want.values[k]), (k, np.argwhere(res.ints[k] != want.values[k])[:4])
    return cm


def block(C, H, T, layers=1, vocab=0, gelu="fused", causal=True):
    spec = models.BlockSpec(C, H, T, layers=layers, vocab=vocab, gelu=gelu, causal=causal, calib_batches=1)
    return models.build(spec, 9)


def block_inputs(built, n, seed=4):
    return models.to_float_input(built.spec, built.params, models.eval_inputs(built.spec, n, 9, seed))


BLOCKS = [(32, 2, 16, 1, 0, "fused"), (32, 1, 5, 2, 0, "lut"), (16, 1, 33, 1, 0, "fused"), (32, 2, 10, 2, 64, "fused"),
          (32, 2, 7, 1, 512, "lut")]


@pytest.mark.parametrize("C,H,T,layers,vocab,gelu", BLOCKS)
@pytest.mark.parametrize("keep", ["outputs", "all"])
def test_planner_runs_row_programs(monkeypatch, C, H, T, layers, vocab, gelu, keep):
    dev = RowFake()
    monkeypatch.setattr(rt, "device", lambda index=0: dev)
    b = block(C, H, T, layers, vocab, gelu)
    check(b.module, b.consts, b, block_inputs(b, 3), keep, False)
    kinds = [c[0] for c in dev.calls if c[0] != "quantize"]
    assert kinds == (["row_program", "attention" + ("_keep" if keep == "all" else "")] * layers + ["row_program"]
                     + ["gemm"] * (vocab == 512))


def test_wider_products_run_op_by_op(monkeypatch):
    dev = RowFake()
    monkeypatch.setattr(rt, "device", lambda index=0: dev)
    b = block(64, 4, 8)
    cm = check(b.module, b.consts, b, block_inputs(b, 2), "outputs", False)
    assert "row_program" not in [c[0] for c in dev.calls]
    assert not rowprog.find(cm, 4095) and len(rowprog.find(cm, 4096)) == 2      # 32,768 rows
    b = block(96, 3, 8)
    assert not rowprog.find(check(b.module, b.consts, b, block_inputs(b, 2), "outputs", False), 4096)


@pytest.mark.parametrize("model", ["v1", "v2"])
@pytest.mark.parametrize("keep", ["outputs", "all"])
def test_planner_runs_the_frozen_models_as_row_programs(monkeypatch, model, keep):
    dev = RowFake()
    monkeypatch.setattr(rt, "device", lambda index=0: dev)
    module, consts = frozen(model)
    lim = 128 if model == "v1" else 1 << 15
    check(module, consts, (module, consts), np.random.default_rng(3).integers(-lim, lim, (3, 16, 32)), keep, True)
    assert [c[0] for c in dev.calls].count("row_program") == 3 and len(dev.calls) == 5


@pytest.mark.parametrize("C,H", [(32, 2), (32, 1), (64, 1)])
@pytest.mark.parametrize("keep", ["outputs", "all"])
def test_one_row_of_k_blocked_values(monkeypatch, C, H, keep):
    """One sequence of one row: a K-blocked value's blocks follow each other, which the kernel takes as a row."""
    dev = RowFake()
    monkeypatch.setattr(rt, "device", lambda index=0: dev)
    monkeypatch.setattr(rowprog, "_product_min", lambda rows: 64)
    b = block(C, H, 1)
    cm = check(b.module, b.consts, b, block_inputs(b, 1), keep, False)
    assert [c[0] for c in dev.calls].count("row_program") == 2
    if keep == "all":
        assert any(v.kb for v in cm.plan(1, keep).views.values())


def test_a_result_without_rows_of_one_stride_runs_op_by_op(monkeypatch):
    """A program whose stored result the kernel cannot address is refused whole, and leaves no buffer behind."""
    dev, memory, refused = RowFake(), rowprog._memory, []
    monkeypatch.setattr(rt, "device", lambda index=0: dev)
    b = block(32, 2, 16)
    op_by_op = anvil_mi355x.compile(b)
    op_by_op.row_programs = False
    names = [buf.name for buf in op_by_op.plan(3).bufs]

    def no_results(view, rows, n):
        if view.buf.name == "out":
            return refused.append(view)
        return memory(view, rows, n)
    monkeypatch.setattr(rowprog, "_memory", no_results)
    cm = check(b.module, b.consts, b, block_inputs(b, 3), "outputs", False)
    assert refused and [c[0] for c in dev.calls].count("row_program") == 1
    names.remove("h1")                                   # inside the first program
    assert [buf.name for buf in cm.plan(3).bufs] == names


def late_graph(late):
    """h = x w, then r = h + z, where z is an input after h, or a view made after h of an earlier input."""
    rng = np.random.default_rng(21)
    bld = GraphBuilder("late")
    x = bld.input("x", [16, 32])
    z = bld.input("z", {"reshape": [16, 2, 16], "transpose": [32, 16]}[late]) if late != "input" else None
    weight = lambda s: bld.const(s, [32, 32], value=rng.integers(-128, 128, (32, 32)))     # noqa: E731
    h = bld.qlinear("h", x, weight("w"), 3, 13)
    h2 = bld.qlinear("h2", h, weight("w2"), 3, 13)
    if late == "input":
        zr = bld.input("z", [16, 32])
    else:
        zr = bld.reshape("zr", z, [16, 32]) if late == "reshape" else bld.transpose("zr", z, [1, 0])
    r = bld.add_requant("r", h2, zr, 100, 90, 8)
    bld.output(bld.qlinear("y", r, weight("w3"), 3, 13))
    return bld.module()


@pytest.mark.parametrize("late", ["input", "reshape", "transpose"])
@pytest.mark.parametrize("keep", ["outputs", "all"])
def test_a_run_ends_before_an_operand_that_stands_inside_it(monkeypatch, late, keep):
    dev = RowFake()
    monkeypatch.setattr(rt, "device", lambda index=0: dev)
    m = late_graph(late)
    cm = anvil_mi355x.compile(m)
    rng = np.random.default_rng(5)
    x = {s: rng.integers(-128, 128, (3, *cm.meta[s][1])) for s in cm.inputs}
    res = cm.run([x[s] for s in cm.inputs], "mi355x", batch=True, keep=keep, quantized=True)
    want = interp.run(m, x, {}, batch=True, fast=True)
    for k in res.ints:
        assert np.array_equal(res.ints[k], want.values[k]), k
    # rows of the transposed input are no rows of one stride: those ops run one by one
    assert [c[0] for c in dev.calls].count("row_program") == (1 if late == "transpose" else 2)


@pytest.mark.gpu
@pytest.mark.parametrize("C,H,T,layers,vocab,gelu", BLOCKS)
@pytest.mark.parametrize("nb,keep", [(1, "outputs"), (3, "all"), (37, "outputs")])
def test_row_programs_match_the_oracle(C, H, T, layers, vocab, gelu, nb, keep):
    """Whole blocks: widths below and at a K block (zero-padded weights), rows that end inside a tile, sequences of odd
    length (V^T byte stores)."""
    b = block(C, H, T, layers, vocab, gelu)
    cm = check(b.module, b.consts, b, block_inputs(b, nb), keep, False)
    assert any(fn is rowprog.call for _, fn, _ in cm.plan(nb, keep).steps)


@pytest.mark.gpu
@pytest.mark.parametrize("C,H", [(32, 2), (16, 1)])
@pytest.mark.parametrize("keep", ["outputs", "all"])
def test_one_row_matches_the_oracle(C, H, keep):
    b = block(C, H, 1)
    cm = check(b.module, b.consts, b, block_inputs(b, 1), keep, False)
    assert any(fn is rowprog.call for _, fn, _ in cm.plan(1, keep).steps)


@pytest.mark.gpu
@pytest.mark.parametrize("T,nb,keep", [(33, 993, "outputs"), (16, 2048, "all")])
def test_64_wide_rows_match_the_oracle(T, nb, keep):
    b = block(64, 2, T)
    cm = check(b.module, b.consts, b, block_inputs(b, nb), keep, False)
    assert any(fn is rowprog.call for _, fn, _ in cm.plan(nb, keep).steps)


@pytest.mark.gpu
@pytest.mark.parametrize("model", ["v1", "v2"])
@pytest.mark.parametrize("nb", [1, 5, 700])
@pytest.mark.parametrize("keep", ["outputs", "all"])
def test_frozen_models_match_the_oracle(model, nb, keep):
    module, consts = frozen(model)
    lim = 128 if model == "v1" else 1 << 15
    x = np.random.default_rng(nb).integers(-lim, lim, (nb, 16, 32))
    x[0] = -lim
    cm = check(module, consts, (module, consts), x, keep, True)
    assert math.prod(cm.meta[cm.inputs[0]][1]) == 512
