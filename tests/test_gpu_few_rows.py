"""The few-row quantized GEMM (qgemm_skinny.hip) at the edges of its shapes: row counts around
its 16-row tiles and its largest, widths that leave a partial tile, one unit of K and several,
units cut short (K not a multiple of 256), rows that start in the middle of a dword, x and Y off
a 16-byte boundary, beta, experts of different sizes and types in one call.

Bars.  F32: 2^-20 against fp64 (x in 22 bits, the weights exact, at most K / 4 products in one
fp32 sum).  x3-ref: 2^-20 against the fp64 product with the fp16 weight; and bit for bit on unit
vectors, whose product is a column of the fp16 weight itself.  Errors are relative to the root of
the summed squares of all products x_k w_k: the Frobenius norm that random signs give, and what the
rounding errors scale with also where a call has so few outputs that theirs cancel (one, here).
"""
import numpy as np
import pytest

import oracle
import tier_amd
from helpers import activations, quantized_weight
from tier_amd import hip

pytestmark = pytest.mark.gpu
BAR = 2.0 ** -20
T = tier_amd
TYPES = [T.Q4_K, T.Q5_K, T.Q6_K, T.Q8_0, T.Q5_0]
SHAPES = [(1, 1, 256), (2, 300, 512), (15, 128, 1280), (16, 129, 768), (17, 1000, 2048), (32, 257, 2304),
          (37, 130, 3328), (48, 640, 5120), (49, 64, 1024), (4, 65, 768), (5, 200, 512), (8, 300, 1280), (9, 70, 512)]
TAILS = [(2, 70, 32), (7, 129, 416), (16, 200, 1408), (33, 40, 5088)]  # q8_0 / q5_0


def _weight(t, N, K, seed, out):
    blocks = quantized_weight(t, N, K, seed)
    w = oracle.dequant(blocks, t, K, out)
    w = w if out == oracle.OUT_F32 else oracle.h2f_array(w)
    return blocks, w.reshape(N, K).astype(np.float64)


def _err(got, want, x, w):
    scale = np.sqrt(((x.astype(np.float64) ** 2) @ (w ** 2).T).sum())
    return np.linalg.norm(got.astype(np.float64) - want) / scale


def _run(blocks, t, x, N, K, mode, y0=None, ldy=None, off=0):
    """The product with x and Y `off` bytes into their buffers; y0 (M, ldy) given: beta = 1."""
    M, ldy = x.shape[0], ldy or N
    W, X, Y = hip.to_device(blocks), hip.DeviceBuffer(x.nbytes + off), hip.DeviceBuffer(M * ldy * 4 + off)
    X.upload(x, off)
    Y.upload(np.full(M * ldy, 7.5, np.float32) if y0 is None else y0, off)
    T.qgemm(W.ptr, t, T.q_row_bytes(t, K), X.ptr + off, Y.ptr + off, M, N, K, ldy=ldy, mode=mode,
            beta=0.0 if y0 is None else 1.0)
    hip.synchronize()
    return Y.download(np.float32, M * ldy, off).reshape(M, ldy)


@pytest.mark.parametrize("mode", [T.MODE_F32, T.MODE_X3REF], ids=["f32", "x3ref"])
@pytest.mark.parametrize("t,M,N,K", [(t, *s) for t in TYPES for s in SHAPES] +
                         [(t, *s) for t in (T.Q8_0, T.Q5_0) for s in TAILS], ids=lambda v: str(v))
def test_few_rows(gpu, t, M, N, K, mode):
    blocks, w = _weight(t, N, K, M + N + K + t, oracle.OUT_F32 if mode == T.MODE_F32 else oracle.OUT_F16)
    x = activations(M, K, seed=M + t)
    want = x.astype(np.float64) @ w.T
    assert _err(_run(blocks, t, x, N, K, mode), want, x, w) <= BAR
    y0 = np.random.default_rng(M).standard_normal((M, N + 3)).astype(np.float32)
    got = _run(blocks, t, x, N, K, mode, y0=y0, ldy=N + 3, off=4)
    assert _err(got[:, :N], want + y0[:, :N], x, w) <= BAR + 2.0 ** -24 * np.linalg.norm(y0) / np.linalg.norm(want)
    assert np.array_equal(got[:, N:], y0[:, N:])


@pytest.mark.parametrize("t", TYPES)
def test_few_rows_x3ref_weight_bits(gpu, t):
    """Unit vectors: every product is one fp16 weight, exactly the dequant's bits."""
    M, N, K = 16, 400, 768
    blocks, w = _weight(t, N, K, 5 + t, oracle.OUT_F16)
    cols = np.random.default_rng(t).choice(K, (12, M), replace=False)
    for c in cols:
        x = np.zeros((M, K), np.float32)
        x[np.arange(M), c] = 1.0
        assert np.array_equal(_run(blocks, t, x, N, K, T.MODE_X3REF).astype(np.float64), w[:, c].T)


def test_few_rows_nonfinite_scale(gpu):
    """A block scale that is not finite makes its weight row's outputs NaN and no others."""
    M, N, K = 5, 40, 512
    for t, at in ((T.Q4_K, 0), (T.Q6_K, 208), (T.Q8_0, 0)):
        blocks, w = _weight(t, N, K, 9 + t, oracle.OUT_F32)
        b = blocks.reshape(N, -1, oracle.block(t)[1]).copy()
        for row, bits in ((3, 0x7c00), (11, 0x7e00)):
            b[row, 1, at:at + 2] = np.array([bits], np.uint16).view(np.uint8)
        x = activations(M, K, seed=t)
        y = _run(b.reshape(N, -1), t, x, N, K, T.MODE_F32)
        bad = np.isin(np.arange(N), (3, 11))
        assert np.all(np.isnan(y[:, bad]))
        assert oracle.rel_fro(y[:, ~bad], (x.astype(np.float64) @ w.T)[:, ~bad]) <= BAR


@pytest.mark.parametrize("N,K", [(1408, 512), (130, 1408)])
def test_few_rows_grouped(gpu, N, K):
    """70 experts of 0 to 31 rows and of three alternating types: one launch a type and number of
    row tiles, some of them with more tiles than the CUs."""
    E = 70
    types = [T.Q8_0, T.Q5_0, T.Q8_0] if K % 256 else [T.Q4_K, T.Q5_0, T.Q6_K]
    rng = np.random.default_rng(N)
    sizes = rng.choice([0, 1, 2, 3, 16], E)
    sizes[5] = 16 if K % 256 else 31
    offs = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    P = int(offs[-1])
    x = activations(P, K, seed=N)
    qts = [types[e % 3] for e in range(E)]
    made = {t: _weight(t, N, K, 3 + t, oracle.OUT_F16) for t in set(types)}
    bufs = {t: hip.to_device(made[t][0]) for t in made}
    X, Y = hip.to_device(x), hip.DeviceBuffer(P * N * 4)
    T.qgemm_grouped([bufs[t].ptr for t in qts], qts, [T.q_row_bytes(t, K) for t in qts], X.ptr, offs, Y.ptr, N, K)
    hip.synchronize()
    got = Y.download(np.float32, P * N).reshape(P, N)
    want = np.concatenate([x[offs[e]:offs[e + 1]].astype(np.float64) @ made[qts[e]][1].T for e in range(E)])
    assert oracle.rel_fro(got, want) <= BAR


@pytest.mark.parametrize("mode", [T.MODE_F32, T.MODE_X3REF], ids=["f32", "x3ref"])
@pytest.mark.parametrize("t,M,N,K", [(T.Q4_K, 16, 1024, 4096), (T.Q8_0, 3, 300, 1408)])
def test_few_rows_in_a_workspace_of_the_general_path(gpu, monkeypatch, t, M, N, K, mode):
    """A workspace of the general path's own size: too small for the split sums of the few-row kernel,
    which then leaves the call to the general path."""
    monkeypatch.setenv("TIERMM_QGEMM_TILE", "-")
    general = T.qgemm_ws_bytes(t, M, N, K, mode)
    monkeypatch.delenv("TIERMM_QGEMM_TILE")
    assert general < T.qgemm_ws_bytes(t, M, N, K, mode)
    blocks, w = _weight(t, N, K, 3, oracle.OUT_F32 if mode == T.MODE_F32 else oracle.OUT_F16)
    x = activations(M, K, seed=4)
    W, X, Y = hip.to_device(blocks), hip.to_device(x), hip.DeviceBuffer(M * N * 4)
    for size in (general, T.qgemm_ws_bytes(t, M, N, K, mode)):
        ws = hip.DeviceBuffer(size)
        T.qgemm(W.ptr, t, T.q_row_bytes(t, K), X.ptr, Y.ptr, M, N, K, mode=mode, ws=ws.ptr, ws_bytes=size)
        hip.synchronize()
        assert _err(Y.download(np.float32, M * N).reshape(M, N), x.astype(np.float64) @ w.T, x, w) <= BAR


@pytest.mark.parametrize("t,M,N,K", [(T.Q4_K, 16, 1024, 4096), (T.Q5_0, 3, 300, 1408), (T.Q6_K, 32, 600, 2048)])
def test_few_rows_parts_bits_in_workspaces_of_a_larger_batch(gpu, t, M, N, K):
    """x3-ref, workspaces sized once for 512 rows: tiermm_qgemm and tiermm_qgemm_x3parts take the same
    kernel for fewer rows, as in workspaces of their own sizes, and give the same bits."""
    blocks, w = _weight(t, N, K, 5, oracle.OUT_F16)
    x = activations(M, K, seed=6)
    rb = T.q_row_bytes(t, K)
    W, X, Y, P = hip.to_device(blocks), hip.to_device(x), hip.DeviceBuffer(M * N * 4), hip.DeviceBuffer(3 * M * K * 2)
    T.split3(X.ptr, P.ptr, M * K, M * K, T.HML)
    got = []
    for rows in (M, 512):
        a, b = T.qgemm_ws_bytes(t, rows, N, K), T.qgemm_x3parts_ws_bytes(t, rows, N, K)
        ws = hip.DeviceBuffer(max(a, b))
        T.qgemm(W.ptr, t, rb, X.ptr, Y.ptr, M, N, K, ws=ws.ptr, ws_bytes=a)
        hip.synchronize()
        got.append(Y.download(np.uint32, M * N))
        T.qgemm_x3parts(W.ptr, t, rb, P.ptr, M * K, Y.ptr, M, N, K, ws=ws.ptr, ws_bytes=b, layout=T.PARTS_ROWS)
        hip.synchronize()
        got.append(Y.download(np.uint32, M * N))
    assert _err(got[0].view(np.float32).reshape(M, N), x.astype(np.float64) @ w.T, x, w) <= BAR
    assert all(np.array_equal(g, got[0]) for g in got[1:])


@pytest.mark.parametrize("types,sizes,N,K", [
    ([T.Q4_K], [16], 2816, 2048), ([T.Q4_K] * 64, [0] * 37 + [1] + [0] * 26, 2816, 2048),
    ([T.Q5_0] * 3, [0, 5, 0], 600, 1408), ([T.Q4_K, T.Q6_K, T.Q4_K], [3, 20, 0], 1024, 4096)],
    ids=["one", "one_of_64", "one_short_k", "one_of_each_type"])
def test_few_rows_one_routed_expert(gpu, types, sizes, N, K):
    """One expert of a type has rows: its product stays inside a workspace of exactly the queried size
    (it may not split K, whose partial sums that size does not hold), and its bits are those that it
    has beside a second expert of its type."""
    offs = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    P = int(offs[-1])
    x = activations(P, K, seed=N)
    made = {t: _weight(t, N, K, 11 + t, oracle.OUT_F16) for t in set(types)}
    bufs = {t: hip.to_device(made[t][0]) for t in made}

    def run(types, offs, x):
        need, guard = T.qgemm_grouped_ws_bytes(types, offs.tolist(), N, K), 8 << 20
        X, Y, ws = hip.to_device(x), hip.DeviceBuffer(x.shape[0] * N * 4), hip.DeviceBuffer(need + guard)
        ws.fill_bytes(0x5a)
        T.qgemm_grouped([bufs[t].ptr for t in types], types, [T.q_row_bytes(t, K) for t in types], X.ptr, offs, Y.ptr,
                        N, K, ws=ws.ptr, ws_bytes=need)
        hip.synchronize()
        assert np.all(ws.download(np.uint8, guard, need) == 0x5a)
        return Y.download(np.float32, x.shape[0] * N).reshape(-1, N)

    got = run(types, offs, x)
    for e, t in enumerate(types):
        r = slice(offs[e], offs[e + 1])
        if sizes[e]:
            w = made[t][1]
            assert _err(got[r], x[r].astype(np.float64) @ w.T, x[r], w) <= BAR, e
    beside = run(types + types, np.concatenate([offs, offs[1:] + P]).astype(np.int32), np.concatenate([x, x]))
    assert np.array_equal(beside[:P].view(np.uint32), got.view(np.uint32))
    assert np.array_equal(beside[P:].view(np.uint32), got.view(np.uint32))


def _shifted(kind, M, K, seed):
    """Rows of x whose mean outweighs their spread, and rows of few distinct values."""
    n = activations(M, K, seed)
    c = np.exp(activations(M, 1, seed + 1))
    x = {"constant": np.broadcast_to(np.linspace(0.1, 3.0, M)[:, None], (M, K)), "two": np.where(n > 0, 0.1, 0.3),
         "near_one": 1 + 0.01 * n, "scaled": c * (1 + 0.3 * n), "three": 3 + n, "abs": np.abs(n)}[kind]
    return np.ascontiguousarray(x, np.float32)


@pytest.mark.parametrize("kind", ["constant", "two", "near_one", "scaled", "three", "abs"])
@pytest.mark.parametrize("M", [1, 8, 9, 37, 48])
@pytest.mark.parametrize("t", [T.Q4_K, T.Q5_K])
def test_few_rows_f32_shifted_x(gpu, monkeypatch, t, M, kind):
    """F32 where x does not average out: codes and minima of q4_K / q5_K are each several times the
    weight, so their products with x may not be rounded apart.  Every row within 2^-20, and no further
    off than the tiled kernel, which multiplies the weights themselves (TIERMM_QGEMM_TILE asks for it)."""
    N, K = 300, 5120
    blocks, w = _weight(t, N, K, 21 + t, oracle.OUT_F32)
    x = _shifted(kind, M, K, M + t)
    want = x.astype(np.float64) @ w.T
    rows = lambda y: np.linalg.norm(y - want, axis=1) / np.linalg.norm(want, axis=1)  # noqa: E731
    got = _run(blocks, t, x, N, K, T.MODE_F32)
    monkeypatch.setenv("TIERMM_QGEMM_TILE", "-")
    tiled = _run(blocks, t, x, N, K, T.MODE_F32)
    assert rows(got).max() <= BAR
    assert oracle.rel_fro(got, want) <= oracle.rel_fro(tiled, want)


@pytest.mark.parametrize("t", [T.Q4_K, T.Q5_K])
def test_few_rows_nonfinite_kq_scales(gpu, t):
    """q4_K / q5_K, d or dmin infinite or NaN: that weight row's outputs are NaN, the others finite."""
    M, N, K = 20, 40, 512
    blocks, w = _weight(t, N, K, 29 + t, oracle.OUT_F32)
    b = blocks.reshape(N, -1, oracle.block(t)[1]).copy()
    rows = (3, 8, 11, 17, 30, 39)
    for i, row in enumerate(rows):  # d (bytes 0, 1) and dmin (2, 3) of either super-block
        b[row, i // 3, 2 * (i % 2):2 * (i % 2) + 2] = np.array([(0x7c00, 0xfc00, 0x7e00)[i % 3]], np.uint16).view(np.uint8)
    x = activations(M, K, seed=t)
    y = _run(b.reshape(N, -1), t, x, N, K, T.MODE_F32)
    bad = np.isin(np.arange(N), rows)
    assert np.all(np.isnan(y[:, bad]))
    assert oracle.rel_fro(y[:, ~bad], (x.astype(np.float64) @ w.T)[:, ~bad]) <= BAR


# experts of one type, rows of each, columns, K
ROUTED = {
    "packed, two launches": (T.Q4_K, [1 + i % 4 for i in range(70)], 192, 512),
    "packed, many items": (T.Q4_K, [1 + i % 3 for i in range(64)], 1408, 512),
    "packed, one unit": (T.Q6_K, [2] * 64, 1408, 256),
    "packed, short unit": (T.Q5_0, [1 + i % 4 for i in range(68)], 640, 1408),
    "packed and two tiles": (T.Q4_K, [1, 17, 4, 32, 2, 0, 25, 3, 31, 0, 18, 1], 300, 768),
    "one tile, many items": (T.Q5_K, [5 + i % 12 for i in range(66)], 900, 512),
    "one tile, short unit": (T.Q8_0, [1 + i % 16 for i in range(64)], 640, 1408),
    "two tiles, many items": (T.Q4_K, [17 + i % 16 for i in range(40)], 1280, 512),
    "two tiles, short unit": (T.Q5_0, [17 + i % 16 for i in range(40)], 1000, 1056),
}


@pytest.mark.parametrize("case", ROUTED)
def test_few_rows_routed(gpu, case):
    """Experts of one type each with its own weight (every 16 rows on in one matrix), each against
    fp64: groups past the 64 of a launch, parts packed in a tile beside and without a second launch,
    and more (expert, columns) items than the grid has workgroups (two a CU, one above 16 rows), so that
    the ring of units runs on from one item into the next, with whole and short last units."""
    t, sizes, N, K = ROUTED[case]
    E, rb = len(sizes), T.q_row_bytes(t, K)
    blocks, w = _weight(t, N + 16 * E, K, 41 + t, oracle.OUT_F16)
    offs = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    P = int(offs[-1])
    x = activations(P, K, seed=E)
    W, X, Y = hip.to_device(blocks), hip.to_device(x), hip.DeviceBuffer(P * N * 4)
    Y.fill_bytes(0xff)
    T.qgemm_grouped([W.ptr + 16 * e * rb for e in range(E)], [t] * E, [rb] * E, X.ptr, offs, Y.ptr, N, K)
    hip.synchronize()
    got = Y.download(np.float32, P * N).reshape(P, N)
    for e in range(E):
        r = slice(offs[e], offs[e + 1])
        if sizes[e]:
            we = w[16 * e:16 * e + N]
            assert _err(got[r], x[r].astype(np.float64) @ we.T, x[r], we) <= BAR, e
