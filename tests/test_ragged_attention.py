"""Fused attention over sequences whose length is no multiple of 32 (ANVIL_ATTN_RAGGED): the planner's routing and
padded V^T, score and probability rows (on the CPU stand-in), and the kernels against the oracle at tile edges."""
import numpy as np
import pytest

import anvil_mi355x
import fake_device
import test_row_program
from anvil_mi355x import models
from anvil_mi355x import runtime as rt
from anvil_mi355x.ir import GraphBuilder
from oracle import interp
from oracle import semantics as sem


@pytest.mark.parametrize("T,C,H", [(5, 64, 2), (16, 64, 1), (31, 64, 4), (33, 128, 2), (48, 64, 2), (100, 64, 1)])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("keep", ["outputs", "all"])
def test_planner_fuses_any_length(monkeypatch, T, C, H, causal, keep):
    dev = fake_device.FakeDevice()
    monkeypatch.setattr(rt, "device", lambda index=0: dev)
    spec = models.BlockSpec(C, H, T, causal=causal, calib_batches=1)
    built = models.build(spec, 9)
    cm = anvil_mi355x.compile(built)
    x = models.eval_inputs(spec, 3, 9)
    res = cm.run(x, "mi355x", batch=True, keep=keep)
    want = interp.run(built.module, {"x": cm.quantize_input(x)}, built.consts, batch=True)
    for k in res.ints:
        assert np.array_equal(res.ints[k], want.values[k]), k
    kinds = [c[0] for c in dev.calls]
    assert "softmax" not in kinds and "copy" not in kinds
    (att,) = [c for c in dev.calls if c[0] in ("attention", "attention_keep")]
    assert bool(att[6] & rt.ATTN_RAGGED) == (T % 32 != 0)
    assert all(s % 16 == 0 for s in att[5])                      # V^T, score and probability rows start 16-byte aligned


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,T,D", [(2, 2, 1, 16), (2, 3, 5, 64), (1, 2, 16, 64), (3, 2, 31, 32), (2, 2, 33, 16),
                                     (2, 1, 48, 128), (1, 3, 127, 64), (2, 2, 129, 32), (1, 2, 250, 64), (1, 1, 529, 128),
                                     (1, 2, 993, 64), (1, 1, 1023, 16)])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("keep", [False, True])
def test_ragged_attention_matches_the_three_ops(B, H, T, D, causal, keep):
    """anvil_attention_i8 and _keep with ANVIL_ATTN_RAGGED, O written into a buffer with a guard after each sequence's
    last row, V^T rows of T rounded up to 16 whose padding holds 0x7F: one row, one key past a tile, one short of it."""
    from test_gpu_ops import _attention_case, up
    dev = rt.device(0)
    C, ldv, lds = H * D, -(-T // 16) * 16, -(-T // 32) * 32
    for seed, sign, kind, one in ((0, 1, "exp", 127), (1, -1, "exp", 127), (2, 1, "random", 127), (3, 1, "steep", 100),
                                  (4, 1, "self", 127), (5, 1, "shift25", 127)):
        q, k, v, (ms, ss, mo, so), lut, want = _attention_case(B, H, T, D, causal, seed, sign, kind, one)
        vt = np.full((B, C, ldv), 0x7F, np.int64)
        vt[..., :T] = np.swapaxes(v, 1, 2)
        out = dev.upload(np.full((B, T + 1, C), 0x5A, np.int8))
        strides = [T * C, D, C, T * C, D, C, C * ldv, D * ldv, ldv, (T + 1) * C, D, C]
        flags = rt.OP_UNCHECKED | rt.ATTN_RAGGED
        args = (up(dev, q, "i8"), up(dev, k, "i8"), up(dev, vt, "i8"), out)
        tail = (ms, ss, up(dev, lut, "i32"), one, causal, mo, so, flags)
        if keep:
            sb, pb = dev.alloc(B * H * T * lds), dev.alloc(B * H * T * lds)
            st = [H * T * lds, T * lds, lds]
            dev.attention_i8_keep(*args, sb, pb, B, H, T, D, strides + st + st, *tail)
        else:
            dev.attention_i8(*args, B, H, T, D, strides, *tail)
        dev.sync()
        got = out.download((B, T + 1, C), np.int8).astype(np.int64)
        assert np.array_equal(got[:, :T], want), (seed, kind, np.argwhere(got[:, :T] != want)[:5])
        assert np.all(got[:, T] == 0x5A), (seed, kind, "a row past the sequence was written")
        if keep:
            split = lambda a: a.reshape(B, T, H, D).transpose(0, 2, 1, 3)       # noqa: E731
            scores = sem.qmatmul(split(q), np.swapaxes(split(k), -1, -2), ms, ss, fast=True)
            p = sem.softmax_lut(scores, lut, one, causal)
            for b, ref in ((sb, scores), (pb, p)):
                a = b.download((B, H, T, lds), np.int8).astype(np.int64)[..., :T]
                assert np.array_equal(a, ref), (seed, kind, np.argwhere(a != ref)[:5])


@pytest.mark.gpu
@pytest.mark.parametrize("T,C,H,keep", [(250, 384, 6, "outputs"), (45, 128, 4, "all"), (16, 128, 2, "all")])
def test_ragged_block_matches_the_oracle(T, C, H, keep):
    spec = models.BlockSpec(C, H, T, calib_batches=1)
    built = models.build(spec, 9)
    cm = anvil_mi355x.compile(built)
    x = models.eval_inputs(spec, 3, 9)
    res = cm.run(x, "mi355x", batch=True, keep=keep)
    want = interp.run(built.module, {"x": cm.quantize_input(x)}, built.consts, batch=True, fast=True)
    for k in res.ints:
        assert np.array_equal(res.ints[k], want.values[k]), k


def const_operand_graph(T, const, dim=32):
    """One head whose q, k or v is a const, over computed values otherwise."""
    rng = np.random.default_rng([31, T])
    bld = GraphBuilder("const_" + const)
    x = bld.input("x", [T, dim])
    vals = {}
    for s in "qkv":
        if s == const:
            vals[s] = bld.const(s, [T, dim], value=rng.integers(-128, 128, (T, dim)))
        else:
            w = bld.const("w" + s, [dim, dim], value=rng.integers(-128, 128, (dim, dim)))
            vals[s] = bld.qlinear(s, x, w, 3, 13)
    scores = bld.qmatmul("s", vals["q"], bld.transpose("kt", vals["k"], [1, 0]), 3, 13)
    exp = np.round(16384.0 * np.exp((np.arange(256) - 255.0) / 20))
    p = bld.softmax_lut("p", scores, bld.const("e", [256], dtype="i32", value=exp), 127, True)
    o = bld.qmatmul("o", p, vals["v"], 1, 7)
    w = bld.const("wy", [dim, dim], value=rng.integers(-128, 128, (dim, dim)))
    bld.output(bld.add_requant("r", bld.qlinear("y", o, w, 3, 13), x, 100, 90, 8))
    return bld.module()


@pytest.mark.parametrize("T", [5, 16, 32, 33])
@pytest.mark.parametrize("const", ["q", "k", "v"])
@pytest.mark.parametrize("keep", ["outputs", "all"])
@pytest.mark.parametrize("row_programs", [False, True])
def test_a_const_operand_leaves_the_three_ops(monkeypatch, T, const, keep, row_programs):
    """q, k and v of a fused chain have the batch dim; a const has none."""
    dev = test_row_program.RowFake() if row_programs else fake_device.FakeDevice()
    monkeypatch.setattr(rt, "device", lambda index=0: dev)
    m = const_operand_graph(T, const)
    cm = anvil_mi355x.compile(m)
    x = np.random.default_rng(3).integers(-128, 128, (3, T, 32))
    res = cm.run(x, "mi355x", batch=True, keep=keep, quantized=True)
    want = interp.run(m, {"x": x}, {}, batch=True, fast=True)
    for k in res.ints:
        assert np.array_equal(res.ints[k], want.values[k]), k
    assert "softmax" in [c[0] for c in dev.calls]
