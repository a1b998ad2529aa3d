"""Products of operands at any alignment (gemm_any.hip; unproven ones: the checked kernel) against the oracle: K below a
16-byte chunk, at its edges, at and past the 128-byte stages in flight, rows that start at any byte, both tile shapes,
batches and both causal modes."""
import numpy as np
import pytest

from anvil_mi355x import runtime as rt
from oracle import semantics as sem

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return rt.device(0)


def up(dev, a, pad=0):
    """The bytes of a after `pad` others: (buffer, address of the first)."""
    buf = dev.upload(np.concatenate([np.full(pad, 99, np.int8), np.ascontiguousarray(a).astype(np.int8).reshape(-1)]))
    return buf, buf.ptr + pad


@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (3, 70, 7), (16, 17, 15), (63, 65, 17), (64, 64, 127), (65, 129, 129), (130, 100, 255),
                                   (100, 200, 385), (16, 1001, 1000), (257, 33, 513), (1500, 1501, 143), (1541, 1500, 3001)])
@pytest.mark.parametrize("form", ["plain", "lut", "i16", "checked"])
@pytest.mark.parametrize("mul24", [True, False])
def test_products(dev, M, N, K, form, mul24):
    rng = np.random.default_rng([54, M, N, K])
    a, w = rng.integers(-128, 128, (M, K)), rng.integers(-128, 128, (K, N))
    lut = rng.integers(-128, 128, 256) if form == "lut" else None
    dt = "i16" if form == "i16" else "i8"
    flags = 0 if form == "checked" else rt.GEMM_UNCHECKED
    flags |= rt.GEMM_MUL24 if mul24 and flags and K * 2 ** 14 < 1 << 23 else 0
    mult, shift = 31, 12 if form == "i16" else 18                  # |acc| mult below 2^31 at every K here
    want = sem.qmatmul(a, w, mult, shift, lut, dt, fast=True)
    (abuf, A), (bbuf, B) = up(dev, a, 3), up(dev, w.T, 5)
    guard = 64
    C = dev.upload(np.full(M * N * rt.ITEMSIZE[dt] + guard, 0x5A, np.uint8))
    L = None if lut is None else dev.upload(lut.astype(np.int8))
    dev.gemm_i8(A, B, C, 1, 1, M, N, K, [0, 0, K, 0, 0, K, 0, 0, N], mult, shift, L, dt, flags)
    dev.sync()
    got = C.download((M, N), rt.NP_DTYPE[dt]).astype(np.int64)
    assert np.array_equal(got, want), np.argwhere(got != want)[:5]
    assert np.all(C.download((guard,), np.uint8, M * N * rt.ITEMSIZE[dt]) == 0x5A)


@pytest.mark.parametrize("T,D", [(33, 20), (130, 64), (250, 17), (600, 72)])
@pytest.mark.parametrize("checked", [False, True])
def test_batched_causal_products(dev, T, D, checked):
    """Scores q k^T with the tiles above the diagonal skipped, and P V (P lower triangular) with the K loop cut there."""
    rng = np.random.default_rng([55, T, D])
    b0, b1 = 2, 3
    flags = 0 if checked else rt.GEMM_UNCHECKED
    q, k = rng.integers(-128, 128, (2, b0, b1, T, D))
    (qb, Q), (kb, Kp) = up(dev, q), up(dev, k, 1)
    S = dev.alloc(b0 * b1 * T * T)
    st = [b1 * T * D, T * D, D, b1 * T * D, T * D, D, b1 * T * T, T * T, T]
    dev.gemm_i8(Q, Kp, S, b0, b1, T, T, D, st, 31, 18, None, "i8", flags | rt.GEMM_CAUSAL_SKIP)
    want = sem.qmatmul(q, k.swapaxes(-1, -2), 31, 18, fast=True)
    dev.sync()
    low = np.tril(np.ones((T, T), bool))
    assert np.array_equal(S.download((b0, b1, T, T), np.int8)[..., low], want[..., low])
    p, v = np.tril(rng.integers(0, 128, (b0, b1, T, T))), rng.integers(-128, 128, (b0, b1, T, D))
    (pb, P), (vb, V) = up(dev, p), up(dev, v.swapaxes(-1, -2), 7)
    O = dev.alloc(b0 * b1 * T * D)
    st = [b1 * T * T, T * T, T, b1 * T * D, T * D, T, b1 * T * D, T * D, D]
    dev.gemm_i8(P, V, O, b0, b1, T, D, T, st, 31, 18, None, "i8", flags | rt.GEMM_CAUSAL_K)
    dev.sync()
    assert np.array_equal(O.download((b0, b1, T, D), np.int8), sem.qmatmul(p, v, 31, 18, fast=True))
