"""anvil_fetch (several device buffers into page-locked memory with one wait) and the host inputs that run() lets a kernel
read in place."""
import numpy as np
import pytest

import anvil_mi355x
from anvil_mi355x import driver, models
from anvil_mi355x import runtime as rt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [[], [1], [15, 16, 17], [4096 * 16 + 5], [100 * i + 1 for i in range(19)], [(4 << 20) + 3, 33, 4 << 20]])
def test_buffers_arrive(sizes):
    dev = rt.device(0)
    rng = np.random.default_rng(len(sizes))
    data = [rng.integers(0, 256, n).astype(np.uint8) for n in sizes]
    bufs = [dev.upload(d) for d in data]
    hosts = [dev.host_alloc(n + 16) for n in sizes]
    for h, n in zip(hosts, sizes):
        h.array(np.uint8, n + 16)[:] = 0x5A
    fetch = dev.fetch(list(zip(bufs, hosts, sizes)))
    for check in (False, True, False):
        fetch(check)
        for h, d in zip(hosts, data):
            got = h.array(np.uint8, len(d) + 16)
            assert np.array_equal(got[:len(d)], d) and np.all(got[len(d):] == 0x5A)


def test_violations_are_reported_when_asked():
    dev = rt.device(0)
    x, out = dev.upload(np.array([1.0, np.nan], np.float32)), dev.alloc(16)
    fetch = dev.fetch([])
    dev.quantize(x, False, 1.0, 2, out, "i8")
    fetch()                                              # leaves them
    with pytest.raises(ValueError, match="NaN or infinite"):
        fetch(True)
    fetch(True)                                          # and reporting clears them


@pytest.mark.parametrize("limit", [0, 1 << 20])
@pytest.mark.parametrize("vocab", [0, 64])
def test_runs_in_place_and_through_a_copy(monkeypatch, limit, vocab):
    """The same results both ways, for inputs that change from run to run, and after a refused one."""
    monkeypatch.setattr(driver, "ZERO_COPY_MAX", limit)
    spec = models.BlockSpec(64, 2, 24, layers=1, vocab=vocab, calib_batches=1)
    b = models.build(spec, 5)
    cm = anvil_mi355x.compile(b)
    for seed in range(5):
        x = models.eval_inputs(spec, 3, 5, seed)
        f = models.to_float_input(spec, b.params, x)
        want = cm.run(cm.quantize_input(f), "mi355x", batch=True, quantized=True)
        got = cm.run(f, "mi355x", batch=True)
        assert all(np.array_equal(got.ints[k], want.ints[k]) for k in want.ints)
        assert np.array_equal(got.output, want.output)
        if vocab:
            ids = cm.run(x, "mi355x", batch=True, tokens=True)
            assert all(np.array_equal(ids.ints[k], want.ints[k]) for k in want.ints)
        bad = f.copy()
        bad[1, 3, 7] = np.inf
        with pytest.raises(ValueError, match="'x' has NaN or infinite values"):
            cm.run(bad, "mi355x", batch=True)
