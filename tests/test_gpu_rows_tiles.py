"""x3_rows at the edges of its 64 x 64 tiles and on both sides of the 160-tile line to the
128 x 128 ones, against fp64 on the same rows (2^-20: x in three parts, fp32 sums)."""
import numpy as np
import pytest

import tier_amd as T
from helpers import activations
from tier_amd import hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(1, 1, 32), (63, 65, 64), (64, 64, 96), (65, 129, 4096), (129, 200, 6176),
                                   (3, 20480, 32), (3, 20481, 32), (7, 130, 7)])
def test_rows_at_tile_edges(gpu, M, N, K):
    x = activations(M, K, seed=M)
    w = (np.random.default_rng(N).standard_normal((N, K)) * 0.02).astype(np.float16)
    W, X, Y = hip.to_device(w), hip.to_device(x), hip.DeviceBuffer(M * (N + 3) * 4)
    Y.upload(np.full(M * (N + 3), 7.5, np.float32))
    assert T.chat_fp3(W.ptr, X.ptr, Y.ptr, M, K, N, N + 3)
    hip.synchronize()
    got = Y.download(np.float32, M * (N + 3)).reshape(M, N + 3)
    scale = np.sqrt(((x.astype(np.float64) ** 2) @ (w.astype(np.float64) ** 2).T).sum())
    assert np.linalg.norm(got[:, :N] - x.astype(np.float64) @ w.astype(np.float64).T) <= 2.0 ** -20 * scale
    assert np.all(got[:, N:] == 7.5)
