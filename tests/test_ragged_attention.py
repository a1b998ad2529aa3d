"""Fused attention over sequences whose length is no multiple of 32 (ANVIL_ATTN_RAGGED): the planner's routing and
padded V^T, score and probability rows (on the CPU stand-in), and the kernels against the oracle at tile edges."""
import numpy as np
import pytest

import anvil_mi355x
import fake_device
from anvil_mi355x import models
from anvil_mi355x import runtime as rt
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
