"""Recorded and captured launch lists (anvil_record_begin / _end, anvil_graph_begin / _end) on the GPU: replays over new
inputs, lists taken while another list replays (nested recording, capture of a replay), and the kernel timer."""
import threading

import numpy as np
import pytest

from anvil_mi355x import runtime as rt
from oracle import semantics as sem

pytestmark = pytest.mark.gpu

N = 1000                                              # a vector part and a tail: two kernels an op


@pytest.fixture(scope="module")
def dev():
    return rt.device(0)


def chain(dev, x, t1, t2, mid, out):
    dev.lut_i8(x, t1, N, mid)
    dev.lut_i8(mid, t2, N, out)


@pytest.mark.parametrize("kind", ["record", "capture", "record of a replay", "capture of a replay", "nested"])
def test_list_replays_over_new_inputs(dev, kind):
    rng = np.random.default_rng(7)
    tabs = [rng.integers(-128, 128, 256).astype(np.int8) for _ in range(2)]
    t1, t2 = (dev.upload(t) for t in tabs)
    x, mid, out = (dev.alloc(N) for _ in range(3))
    x.upload(rng.integers(-128, 128, N).astype(np.int8))
    seq = dev.sequence(chain, dev, x, t1, t2, mid, out)
    if kind == "capture":
        seq = dev.capture(chain, dev, x, t1, t2, mid, out)
    elif kind == "record of a replay":
        seq = dev.sequence(seq.launch)
    elif kind == "capture of a replay":
        seq = dev.capture(seq.launch)
    elif kind == "nested":
        inner = []
        seq = dev.sequence(lambda: inner.append(dev.sequence(chain, dev, x, t1, t2, mid, out)))
        inner[0].free()
    for j in range(3):
        v = rng.integers(-128, 128, N).astype(np.int8)
        x.upload(v)
        dev.zero(out, N)
        if j == 2:                                    # a replay under the timer carries its events
            dev.timed(0, 1, seq.launch)
        else:
            seq.launch()
        dev.sync()
        want = sem.lut_i8(sem.lut_i8(v.astype(np.int64), tabs[0].astype(np.int64)), tabs[1].astype(np.int64))
        assert np.array_equal(out.download((N,), np.int8).astype(np.int64), want), (kind, j)
    assert dev.elapsed_ms(0, 1) > 0
    seq.free()


def test_record_end_without_a_begin_is_refused(dev):
    with pytest.raises(ValueError, match="nothing is being recorded"):
        dev.lib.call("anvil_record_end", dev.ctx, rt.C.byref(rt.C.c_void_p()))


def on_another_thread(fn):
    """fn() on a thread of its own; its result, or its exception raised here."""
    got = {}

    def go():
        try:
            got["value"] = fn()
        except BaseException as e:
            got["error"] = e
    t = threading.Thread(target=go)
    t.start()
    t.join()
    if "error" in got:
        raise got["error"]
    return got["value"]


@pytest.mark.parametrize("launcher", ["the thread that began", "the other thread", "both"])
def test_a_capture_ended_on_another_thread(dev, launcher):
    """It replays, and leaves no recording open on the thread that began it."""
    rng = np.random.default_rng(8)
    tabs = [rng.integers(-128, 128, 256).astype(np.int8) for _ in range(2)]
    t1, t2 = (dev.upload(t) for t in tabs)
    x, mid, out = (dev.alloc(N) for _ in range(3))
    x.upload(np.zeros(N, np.int8))
    chain(dev, x, t1, t2, mid, out)
    dev.sync()

    def end():
        handle = rt.C.c_void_p()
        dev.lib.call("anvil_graph_end", dev.ctx, rt.C.byref(handle))
        return rt.HipGraph(dev, handle.value)
    first, second = (lambda: dev.lut_i8(x, t1, N, mid)), (lambda: dev.lut_i8(mid, t2, N, out))
    dev.lib.call("anvil_graph_begin", dev.ctx)
    (on_another_thread(first) if launcher == "the other thread" else first())
    (second() if launcher == "the thread that began" else on_another_thread(second))
    seq = on_another_thread(end)
    with pytest.raises(ValueError, match="nothing is being recorded"):
        dev.lib.call("anvil_record_end", dev.ctx, rt.C.byref(rt.C.c_void_p()))
    for j in range(3):
        v = rng.integers(-128, 128, N).astype(np.int8)
        x.upload(v)
        dev.zero(out, N)
        (seq.launch() if j else on_another_thread(seq.launch))
        dev.sync()
        want = sem.lut_i8(sem.lut_i8(v.astype(np.int64), tabs[0].astype(np.int64)), tabs[1].astype(np.int64))
        assert np.array_equal(out.download((N,), np.int8).astype(np.int64), want), j
    seq.free()


def test_a_recording_ends_on_its_own_thread(dev):
    x, out = dev.upload(np.arange(16, dtype=np.int8)), dev.alloc(16)
    t = dev.upload(np.arange(256).astype(np.uint8).view(np.int8))
    dev.lib.call("anvil_record_begin", dev.ctx)
    handle = rt.C.c_void_p()
    with pytest.raises(ValueError, match="nothing is being recorded"):
        on_another_thread(lambda: dev.lib.call("anvil_record_end", dev.ctx, rt.C.byref(rt.C.c_void_p())))
    dev.lut_i8(x, t, 16, out)
    dev.lib.call("anvil_record_end", dev.ctx, rt.C.byref(handle))
    dev.sync()
    rt.HipGraph(dev, handle.value).free()


def test_a_destroyed_context_drops_its_recordings():
    """Contexts made after it, whose stream may have the same address, have none open."""
    for _ in range(8):
        d = rt.Device(0)
        with pytest.raises(ValueError, match="nothing is being recorded"):
            d.lib.call("anvil_record_end", d.ctx, rt.C.byref(rt.C.c_void_p()))
        d.lib.call("anvil_record_begin", d.ctx)
        d.close()
