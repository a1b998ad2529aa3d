"""A run that fails part way leaves nothing behind: no violation that the next run would report, and no kernel that still
reads the host input (on a CPU stand-in with the one-wait read-back, and on the GPU)."""
import numpy as np
import pytest

import anvil_mi355x
import fake_device
from anvil_mi355x import models
from anvil_mi355x import runtime as rt
from oracle import interp


class HeapHost:
    """A page-locked buffer whose address the stand-in's kernels can read."""

    def __init__(self, dev, nbytes):
        self.buf, self.nbytes = fake_device.FakeBuffer(dev, nbytes), int(nbytes)
        self.dev, self.ptr = dev, self.buf.ptr

    def array(self, dtype, count):
        return self.dev._raw(self.ptr, dtype, count)


class FetchFake(fake_device.FakeDevice):
    """The stand-in with anvil_fetch: copies, one wait (counted), and with check what sync() reports."""
    waits = 0

    def host_alloc(self, nbytes):
        return HeapHost(self, nbytes)

    def fetch(self, items):
        def go(check=False):
            self.waits += 1
            for b, h, n in items:
                h.array(np.uint8, n)[:] = b.download((n,), np.uint8)
            if check:
                self.sync()
        return go


def fake(monkeypatch):
    dev = FetchFake()
    monkeypatch.setattr(rt, "device", lambda index=0: dev)
    return dev


def model(C=64, H=2, T=24, vocab=0):
    spec = models.BlockSpec(C, H, T, layers=1, vocab=vocab, calib_batches=1)
    return spec, models.build(spec, 5)


def float_inputs(spec, b, n=2):
    return models.to_float_input(spec, b.params, models.eval_inputs(spec, n, 5, 3))


class Stop(BaseException):
    pass


@pytest.mark.parametrize("error", [MemoryError, Stop])
@pytest.mark.parametrize("bad", [False, True])
def test_a_failed_launch_leaves_no_violation(monkeypatch, error, bad):
    """bad: the failed run's input held a NaN, which is what an ordinary error of that run then says."""
    dev = fake(monkeypatch)
    spec, b = model()
    cm = anvil_mi355x.compile(b)
    f = float_inputs(spec, b)
    f[1, 3, 5] = np.nan if bad else f[1, 3, 5]
    launch = cm.launch

    def failing(*args):
        launch(*args)
        dev.flags = dev.flags or OverflowError("an aborted forward's violation")
        raise error("launch")
    cm.launch = failing
    with pytest.raises(ValueError if bad and error is MemoryError else error,
                       match="'x' has NaN or infinite values" if bad and error is MemoryError else "launch"):
        cm.run(f, "mi355x", batch=True)
    assert dev.waits == 1
    cm.launch = launch
    f = float_inputs(spec, b)
    got = cm.run(f, "mi355x", batch=True)
    want = interp.run(b.module, {"x": cm.quantize_input(f)}, b.consts, batch=True)
    assert all(np.array_equal(got.ints[k], want.values[k]) for k in got.ints)


def test_a_broken_device_keeps_the_first_error(monkeypatch):
    dev = fake(monkeypatch)
    spec, b = model()
    cm = anvil_mi355x.compile(b)

    def broken(items):
        raise RuntimeError("the device is gone")
    cm.plan(2)
    cm.launch = lambda *a: (setattr(dev, "fetch", broken), (_ for _ in ()).throw(MemoryError("launch")))
    with pytest.raises(MemoryError, match="launch"):
        cm.run(float_inputs(spec, b), "mi355x", batch=True)


@pytest.mark.gpu
@pytest.mark.parametrize("error", [MemoryError, Stop])
def test_a_failed_launch_leaves_no_violation_on_the_gpu(error):
    spec, b = model()
    cm = anvil_mi355x.compile(b)
    f = float_inputs(spec, b)
    want = cm.run(f, "mi355x", batch=True)
    launch = cm.launch

    def failing(*args):
        raise error("launch")
    for _ in range(2):
        cm.launch = failing
        bad = f.copy()
        bad[0, 1, 2] = np.inf
        with pytest.raises(ValueError if error is MemoryError else error):
            cm.run(bad, "mi355x", batch=True)
        cm.launch = launch
        got = cm.run(f, "mi355x", batch=True)
        assert all(np.array_equal(got.ints[k], want.ints[k]) for k in want.ints)
