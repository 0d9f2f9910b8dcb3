"""The bytes that bench.py prices the edge-parallel leap's draws with, against hand
counts: counts, the forward CSR (each undirected edge once) and the 32-bit balances."""
import numpy as np
import pytest

import bench


@pytest.mark.parametrize("weighted", [False, True])
def test_bytes_of_the_draws(weighted):
    S, N, E = 5, 1000, 8000
    t = {"N": N, "col": np.zeros(E, dtype=np.uint32)}
    if weighted:
        t["w"] = np.ones(E, dtype=np.float32)
    forward = 4 * (N + 1) + 4 * (E // 2) + (4 * (E // 2) if weighted else 0)
    assert bench.algorithmic_bytes(S, [t], "leap_draws") == 4 * S * N + forward + 4 * S * N
    assert bench.algorithmic_bytes(S, [t, t], "leap_draws") == 2 * bench.algorithmic_bytes(S, [t], "leap_draws")
