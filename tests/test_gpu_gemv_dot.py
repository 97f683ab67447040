"""The int8-dot decode GEMV (qgemv_dot.hip) at the edges of its shapes: one row, rows fewer and
more than the CUs, units that do not fill the lanes of a row, rows of q3_K / q6_K that start
two bytes off a dword, weights that start 4 bytes off a 16-byte boundary, K above the range of
one pass over x, tall matrices (rows of 16, 32 and 64 lanes, odd and even counts of steps, several
rows a slot, several parts a row), and block scales that are not finite.

Bar: 2e-6 relative Frobenius against fp64.  Block sums are exact in int32 and rounded to
fp32 once; a lane then adds at most K / (16 * 32) + 6 fp32 terms per row (34 at K = 14336,
each rounding at most 2^-24 of the running sum), 2e-6 in the worst case.
"""
import numpy as np
import pytest

import oracle
import tier_amd
from tier_amd import hip

pytestmark = pytest.mark.gpu
T = tier_amd
# shapes that no other kernel takes (but q5_K up to K = 5120, which its MFMA kernel does)
SMALL = [T.Q4_0, T.Q4_1, T.Q5_0, T.Q5_1, T.IQ4_NL, T.Q8_0]
SUPER = [T.Q2_K, T.Q3_K, T.IQ4_XS, T.Q4_K, T.Q5_K, T.Q6_K]
SHAPES = [(1, 256), (3, 512), (255, 1280), (257, 2304), (600, 5376), (40, 14336), (17, 18432)]
ODD_K = [(5, 64), (33, 320), (300, 1088)]


def _run(blocks, t, x, N, K, offset=0):
    rb = T.q_row_bytes(t, K)
    W = hip.DeviceBuffer(N * rb + offset)
    W.upload(np.ascontiguousarray(blocks).view(np.uint8).ravel(), offset)
    X, Y = hip.to_device(x), hip.DeviceBuffer(N * 4)
    Y.fill_bytes(0x3f)
    T.gemv_q(W.ptr + offset, t, rb, X.ptr, Y.ptr, N, K)
    hip.synchronize()
    return Y.download(np.float32, N)


def _blocks(t, N, K, seed):
    rng = np.random.default_rng(seed)
    return oracle.random_blocks(rng, t, N * (K // oracle.block(t)[0]), moderate=True).reshape(N, -1), \
        rng.standard_normal(K).astype(np.float32)


@pytest.mark.parametrize("t,N,K", [(t, N, K) for t in SMALL + SUPER for N, K in SHAPES] +
                         [(t, N, K) for t in SMALL for N, K in ODD_K],
                         ids=lambda v: str(v))
def test_dot_gemv_shapes(gpu, t, N, K):
    blocks, x = _blocks(t, N, K, 7 * N + K + t)
    want = oracle.gemv_f64(blocks, t, x, N, K)
    for offset in (0, 4) if t not in (T.Q4_K, T.Q5_K) else (0,):  # those rows are 16-byte aligned by contract
        y = _run(blocks, t, x, N, K, offset)
        assert np.all(np.isfinite(y))
        assert oracle.rel_fro(y, want) <= 2e-6, offset


@pytest.mark.parametrize("t", [T.Q4_0, T.Q5_1, T.IQ4_XS, T.Q2_K, T.Q3_K, T.Q6_K])
def test_dot_gemv_nonfinite_scale(gpu, t):
    """An infinite or NaN block scale: the row takes gemv_q's own classes, the others are untouched."""
    N, K = 40, 1280
    blocks, x = _blocks(t, N, K, 3 + t)
    bb = oracle.block(t)[1]
    at = {T.Q4_0: 0, T.Q5_1: 0, T.IQ4_XS: 0, T.Q2_K: 80, T.Q3_K: 108, T.Q6_K: 208}[t]
    b = blocks.reshape(N, -1, bb)
    for row, bits in ((3, 0x7c00), (11, 0xfc00), (30, 0x7e00)):
        b[row, 2, at:at + 2] = np.array([bits], np.uint16).view(np.uint8)
    y = _run(blocks, t, x, N, K)
    want = oracle.gemv_lanes(blocks, t, x, N, K)
    for f in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(f(y), f(want))
    ok = np.isfinite(want)
    assert ok.sum() == N - 3
    assert oracle.rel_fro(y[ok], oracle.gemv_f64(blocks, t, x, N, K)[ok]) <= 2e-6


# units of 64 elements (iq4), of 128 (q2_K, q3_K) on 256 CUs: lanes a row, steps a row, rows a slot
TALL = [(14336, 5120),  # 16, 5, 1; 16, 3, 1
        (9001, 2304),   # 64, 1, 3; 32, 1, 2; ragged rows a workgroup, q3_K rows at both phases
        (4097, 5376),   # 32, 3, 1; 64, 1, 2
        (2500, 8192),   # 64, 2, 1; 64, 1, 1
        (20001, 1024),  # 16, 1, 2
        (5120, 14336)]  # 64, 1, 5 in four parts; 64, 1, 3 in two


@pytest.mark.parametrize("N,K", TALL)
@pytest.mark.parametrize("t", [T.IQ4_XS, T.IQ4_NL, T.Q2_K, T.Q3_K])
def test_dot_gemv_tall(gpu, t, N, K):
    """Every row: the largest error against the outputs' root mean square (34 roundings of sums up
    to some four times that: 1e-5)."""
    blocks, x = _blocks(t, N, K, N + K + t)
    want = oracle.gemv_f64(blocks, t, x, N, K)
    y = _run(blocks, t, x, N, K)
    assert oracle.rel_fro(y, want) <= 2e-6
    assert np.abs(y - want).max() <= 1e-5 * np.sqrt(np.mean(want ** 2))


def _zero_at(t, b, j):
    """Element j < 16 of each 32-element block (of each 256-element one, for the K types) set to weight 0."""
    b = b.copy()
    if t == T.Q4_0:
        b[..., 2 + j] = b[..., 2 + j] & 0xf0 | 8
    elif t == T.Q4_1:  # m = -8 d
        d = b[..., 0:2].copy().view(np.float16)
        b[..., 2:4] = (d * np.float16(-8)).view(np.uint8)
        b[..., 4 + j] = b[..., 4 + j] & 0xf0 | 8
    elif t == T.Q5_0:
        b[..., 2 + j // 8] |= 1 << (j % 8)
        b[..., 6 + j] &= 0xf0
    elif t == T.Q5_1:  # m = -16 d
        d = b[..., 0:2].copy().view(np.float16)
        b[..., 2:4] = (d * np.float16(-16)).view(np.uint8)
        b[..., 4 + j // 8] |= 1 << (j % 8)
        b[..., 8 + j] &= 0xf0
    elif t == T.Q8_0:
        b[..., 2 + j] = 0
    elif t == T.Q2_K:  # d sc 1 - dmin m, with dmin = d and m = sc
        b[..., :16] = (b[..., :16] & 15) * 17
        b[..., 82:84] = b[..., 80:82]
        b[..., 16 + j] = b[..., 16 + j] & 0xfc | 1
    elif t == T.Q3_K:
        b[..., j] |= 1
        b[..., 32 + j] &= 0xfc
    elif t == T.Q6_K:
        b[..., j] &= 0xf0
        b[..., 128 + j] = b[..., 128 + j] & 0xfc | 2
    return b


@pytest.mark.parametrize("mag", [64.0, 2.0 ** 40])
@pytest.mark.parametrize("t", [T.Q4_0, T.Q4_1, T.Q5_0, T.Q5_1, T.Q8_0, T.Q2_K, T.Q3_K, T.Q6_K])
def test_dot_gemv_outlier_in_x(gpu, t, mag):
    """An outlier of x where every row's weight is zero, beside ordinary values: its block's other
    elements keep the bits that fp32 sums would give them.  Outliers in every block and in every third;
    rows in several parts, and several rows a slot (9001; q6_K's dot kernel stops short of that)."""
    be, bb = oracle.block(t)
    for N, K, step in ((40, 1280, 1), (257, 14336, 3), (1000 if t == T.Q6_K else 9001, 2304, 1)):
        blocks, x = _blocks(t, N, K, 5 * N + t)
        b = _zero_at(t, blocks.reshape(N, -1, bb), 5).reshape(N, -1)
        at = np.arange(5, K, be)[::step]
        assert np.all(oracle.dequant(b, t, K, oracle.OUT_F32).reshape(N, K)[:, at] == 0)
        x[at] = mag * np.where(np.arange(at.size) % 2, 1, -1)
        rest = x.copy()
        rest[at] = 0
        y = _run(b, t, x, N, K)
        assert oracle.rel_fro(y, oracle.gemv_f64(b, t, rest, N, K)) <= 2e-6, (N, K)


@pytest.mark.parametrize("t", SMALL + SUPER)
def test_dot_gemv_tiny_x(gpu, t):
    """x of 2^-114: beyond the exponent that scales the digits to full width."""
    N, K = 40, 5376
    blocks, x = _blocks(t, N, K, 31 + t)
    x *= np.float32(2.0 ** -114)
    y = _run(blocks, t, x, N, K).astype(np.float64) * 2.0 ** 114
    assert oracle.rel_fro(y, oracle.gemv_f64(blocks, t, x, N, K) * 2.0 ** 114) <= 2e-6
