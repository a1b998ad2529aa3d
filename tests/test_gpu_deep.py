"""The deep-pipelined GEMM (gemm_deep.hip), which products of at most two 64 x 64 tiles a CU take: against the oracle at
tile edges, K below, at and past its two and four stages of 128 bytes, unaligned result rows, batches, groups, the LUT
and the fused residual add."""
import numpy as np
import pytest

from anvil_mi355x import runtime as rt
from oracle import semantics as sem

pytestmark = pytest.mark.gpu

MULT, SHIFT = 40, 19


@pytest.fixture(scope="module")
def dev():
    return rt.device(0)


def up(dev, a, dt="i8"):
    return dev.upload(np.ascontiguousarray(a).astype(rt.NP_DTYPE[dt]))


def kblocked(a):
    """(rows, K) as K blocks of 64: (K / 64, rows, 64)."""
    return a.reshape(len(a), -1, 64).transpose(1, 0, 2)


@pytest.mark.parametrize("M,N,K", [(1, 16, 16), (16, 3072, 768), (63, 65, 48), (64, 64, 128), (65, 200, 256), (130, 80, 272),
                                   (1000, 777, 512), (257, 48, 1008), (300, 130, 3072), (64, 1024, 144)])
@pytest.mark.parametrize("form", ["plain", "kblocked", "lut", "i16"])
@pytest.mark.parametrize("mul24", [True, False])
def test_products(dev, M, N, K, form, mul24):
    rng = np.random.default_rng([51, M, N, K])
    a, w = rng.integers(-128, 128, (M, K)), rng.integers(-128, 128, (K, N))
    lut = rng.integers(-128, 128, 256) if form == "lut" else None
    dt = "i16" if form == "i16" else "i8"
    flags = rt.GEMM_UNCHECKED | (rt.GEMM_MUL24 if mul24 and K * 2 ** 14 < 1 << 23 else 0)
    shift = 12 if form == "i16" else SHIFT
    mult = MULT if K * 2 ** 14 * MULT < (1 << 31) - (1 << 20) else 1     # the proof keeps acc M + rnd inside int32
    shift = shift if mult == MULT else 16
    want = sem.qmatmul(a, w, mult, shift, lut, dt, fast=True)
    A, B, st = up(dev, a), up(dev, w.T), [0, 0, K, 0, 0, K, 0, 0, N]
    if form == "kblocked" and K % 64 == 0:
        A, B, st = up(dev, kblocked(a)), up(dev, kblocked(w.T)), [0, 0, M * 64, 0, 0, N * 64, 0, 0, N]
        flags |= rt.GEMM_A_KBLOCK | rt.GEMM_B_KBLOCK
    guard = 64
    C = dev.upload(np.full(M * N * rt.ITEMSIZE[dt] + guard, 0x5A, np.uint8))
    dev.gemm_i8(A, B, C, 1, 1, M, N, K, st, mult, shift, None if lut is None else up(dev, lut), dt, flags)
    dev.sync()
    got = C.download((M, N), rt.NP_DTYPE[dt]).astype(np.int64)
    assert np.array_equal(got, want), np.argwhere(got != want)[:5]
    assert np.all(C.download((guard,), np.uint8, M * N * rt.ITEMSIZE[dt]) == 0x5A)


@pytest.mark.parametrize("M,N,K,ldr", [(16, 64, 64, 64), (65, 80, 256, 96), (200, 72, 272, 72), (1024, 768, 3072, 768),
                                       (63, 130, 128, 130)])
@pytest.mark.parametrize("store_y", [True, False])
@pytest.mark.parametrize("ma,mb,s2", [(300, -200, 9), (16777216, -16777216, 25)])
def test_residual_add(dev, M, N, K, ldr, store_y, ma, mb, s2):
    """Residual rows 16-byte aligned or not, a wider residual stride than the row, multipliers on both sides of 2^24."""
    rng = np.random.default_rng([52, M, N, K])
    if ma > 1 << 23:
        ma, mb = ma // 2 * 2, mb // 4
    a, w, r = rng.integers(-128, 128, (M, K)), rng.integers(-128, 128, (K, N)), rng.integers(-60, 60, (M, ldr))
    y = sem.qmatmul(a, w, 3, 16, fast=True)
    want = sem.add_requant(r[:, :N], np.clip(y, -128, 127), ma, mb, s2) if ma < 1 << 24 else \
        np.clip((r[:, :N] * ma + y * mb + (1 << (s2 - 1))) >> s2, -128, 127)
    C = dev.alloc(M * N) if store_y else None
    D = dev.upload(np.full(M * N + 64, 0x5A, np.uint8))
    dev.gemm_i8_add(up(dev, a), up(dev, w.T), C, 1, 1, M, N, K, [0, 0, K, 0, 0, K, 0, 0, N], 3, 16, None, up(dev, r), ma, mb,
                    s2, D, [0, 0, ldr, 0, 0, N], rt.GEMM_UNCHECKED)
    dev.sync()
    got = D.download((M, N), np.int8).astype(np.int64)
    assert np.array_equal(got, want), np.argwhere(got != want)[:5]
    assert np.all(D.download((64,), np.uint8, M * N) == 0x5A)
    if store_y:
        assert np.array_equal(C.download((M, N), np.int8).astype(np.int64), y)


def test_batched_and_grouped_products(dev):
    """Three products of one group: plain, batched with a shared left operand (V^T of each sequence), and one whose
    result rows are unaligned."""
    rng = np.random.default_rng(53)
    T, C, B = 50, 96, 3
    x, w = rng.integers(-128, 128, (B, T, C)), rng.integers(-128, 128, (3, C, C))
    w[2][:, 70:] = 0
    X = up(dev, x)
    W = [up(dev, m.T) for m in w]
    out = [dev.alloc(B * T * C) for _ in range(3)]
    fl = rt.GEMM_UNCHECKED | rt.GEMM_MUL24
    dev.gemm_i8_group([(X, W[0], out[0], 1, 1, B * T, C, C, [0, 0, C, 0, 0, C, 0, 0, C], MULT, SHIFT, None, "i8", fl),
                       (W[1], X, out[1], 1, B, C, T, C, [0, 0, C, 0, T * C, C, 0, C * T, T], MULT, SHIFT, None, "i8", fl),
                       (X, W[2], out[2], 1, 1, B * T, 70, C, [0, 0, C, 0, 0, C, 0, 0, 70], MULT, SHIFT, None, "i8", fl)])
    dev.sync()
    y = [sem.qmatmul(x, m, MULT, SHIFT, fast=True) for m in w]
    assert np.array_equal(out[0].download((B, T, C), np.int8), y[0])
    assert np.array_equal(out[1].download((B, C, T), np.int8), y[1].transpose(0, 2, 1))
    assert np.array_equal(out[2].download((B, T, 70), np.int8), y[2][..., :70])


# Past two 64 x 64 tiles a CU (512 on 256 CUs) the one-tile-per-workgroup kernels take the same calls: 128 x 128 tiles
# with ragged rows and columns, K below, at and past their stages of 64 bytes, whole rotations of three stages (192) or not

@pytest.mark.parametrize("M,N,K", [(2080, 1030, 16), (2049, 1090, 48), (4100, 600, 144), (2177, 1040, 192), (2100, 1100, 1008),
                                   (8193, 300, 384), (2177, 1152, 256)])
@pytest.mark.parametrize("form", ["plain", "kblocked", "lut", "i16"])
@pytest.mark.parametrize("mul24", [True, False])
def test_products_past_the_line(dev, M, N, K, form, mul24):
    assert -(-M // 64) * -(-N // 64) > 512
    test_products(dev, M, N, K, form, mul24)


@pytest.mark.parametrize("M,N,K,ldr", [(2080, 1040, 64, 1040), (2049, 1090, 272, 1090), (4100, 592, 192, 608)])
@pytest.mark.parametrize("store_y", [True, False])
@pytest.mark.parametrize("ma,mb,s2", [(300, -200, 9), (16777216, -16777216, 25)])
def test_residual_add_past_the_line(dev, M, N, K, ldr, store_y, ma, mb, s2):
    test_residual_add(dev, M, N, K, ldr, store_y, ma, mb, s2)


@pytest.mark.parametrize("B,H,T,d", [(40, 4, 100, 64), (70, 2, 130, 48)])
def test_batched_products_past_the_line(dev, B, H, T, d):
    """scores = q k^T of every head, read in place: batch strides (T C, d), row stride C."""
    rng = np.random.default_rng([57, B, T])
    C = H * d
    q, k = rng.integers(-128, 128, (2, B, T, C))
    S = dev.alloc(B * H * T * T)
    dev.gemm_i8(up(dev, q), up(dev, k), S, B, H, T, T, d, [T * C, d, C, T * C, d, C, H * T * T, T * T, T], MULT, SHIFT, None,
                "i8", rt.GEMM_UNCHECKED | rt.GEMM_MUL24)
    dev.sync()
    heads = lambda a: a.reshape(B, T, H, d).transpose(0, 2, 1, 3)                 # noqa: E731
    want = sem.qmatmul(heads(q), heads(k).swapaxes(-1, -2), MULT, SHIFT, fast=True)
    assert np.array_equal(S.download((B, H, T, T), np.int8), want)
