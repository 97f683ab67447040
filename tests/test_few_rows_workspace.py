"""Workspace sizes of products with few rows, on the host: a routed batch's size holds for every
routing of as many rows to as many experts, and a small M's is no less than what the general path,
to which the few-row kernel leaves a call that has no room for its own, needs (TIERMM_QGEMM_TILE
asks for that path)."""
import random

import pytest

import tier_amd as T

TYPES = [T.Q4_K, T.Q5_K, T.Q6_K, T.Q8_0, T.Q5_0]


@pytest.mark.parametrize("t", [T.Q4_K, T.Q6_K, T.Q5_0])
@pytest.mark.parametrize("P,E", [(1, 8), (8, 64), (64, 64), (200, 16), (700, 64)])
def test_routed_size_does_not_depend_on_the_routing(t, P, E):
    rng = random.Random(P)
    sizes = set()
    for _ in range(6):
        cut = sorted(rng.randint(0, P) for _ in range(E - 1))
        sizes.add(T.qgemm_grouped_ws_bytes([t] * E, [0, *cut, P], 1408, 2048))
    sizes.add(T.qgemm_grouped_ws_bytes([t] * E, [0] + [min(P, i + 1) for i in range(E - 1)] + [P], 1408, 2048))
    assert len(sizes) == 1


@pytest.mark.parametrize("mode", [T.MODE_F32, T.MODE_X3REF], ids=["f32", "x3ref"])
@pytest.mark.parametrize("t", TYPES)
def test_size_covers_the_general_path(t, mode, monkeypatch):
    for M in (1, 2, 16, 17, 33, 48):
        for N, K in ((64, 256), (1024, 4096), (14336, 5120)):
            both = T.qgemm_ws_bytes(t, M, N, K, mode)
            monkeypatch.setenv("TIERMM_QGEMM_TILE", "-")  # no plan: the general path's own
            assert both >= T.qgemm_ws_bytes(t, M, N, K, mode)
            monkeypatch.delenv("TIERMM_QGEMM_TILE")
