"""Workspace sizes of products with few rows, on the host: a routed batch's size holds for every
routing of as many rows to as many experts, and a small M's is no less than what the general path,
to which the few-row kernel leaves a call that has no room for its own, needs (TIERMM_QGEMM_TILE
asks for that path), and an x3-ref size for many rows holds what the few-row kernel needs of fewer,
so that a workspace sized once leaves every call the kernel that it has in one of its own size."""
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


@pytest.mark.parametrize("mode", [T.MODE_F32, T.MODE_X3REF, "parts"], ids=["f32", "x3ref", "x3parts"])
@pytest.mark.parametrize("t", TYPES)
def test_size_covers_fewer_rows(t, mode, monkeypatch):
    def size(M, N, K):
        return T.qgemm_x3parts_ws_bytes(t, M, N, K) if mode == "parts" else T.qgemm_ws_bytes(t, M, N, K, mode)

    for N, K in ((64, 256), (1024, 4096), (14336, 5120)):
        for m in (1, 4, 5, 16, 17, 32, 33, 48):
            own = size(m, N, K)
            monkeypatch.setenv("TIERMM_QGEMM_TILE", "-")
            general = size(m, N, K)
            monkeypatch.delenv("TIERMM_QGEMM_TILE")
            if own > general:  # the few-row kernel's need, or that of fewer rows still
                for M in (m, 32, 48) if mode == T.MODE_F32 else (m, 32, 48, 49, 64, 300, 4096):
                    assert M < m or size(M, N, K) >= own, (N, K, m, M)
