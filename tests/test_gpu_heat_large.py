"""Conduction on shells around the size from which the search direction's dot
products are summed once instead of by every workgroup that needs them."""
import numpy as np
import pytest

from falcon_amd import HeatSolver, Shell, configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("np_", [34, 36])     # 9.46 M and 10.6 M partial reads: below and above 10 M
def test_batched_systems_equal_single_solves(np_):
    """Every system's sums have the same order whatever the batch, and the
    recomputed residual is the solve's tolerance (1e-10, twice that for its own
    rounding)."""
    s = Shell({"ni": 16, "nj": 16, "nk": 16, "ng": 2, "r_rsun": configs.R_RANGE, "ops": [("split", (4, 8, np_))]})
    hs = HeatSolver(s, 1.0, 0.7, 1)
    dt = 30.0 * hs.dt_explicit
    T = 1e-3 * np.random.default_rng(2).standard_normal(hs.shape)
    runs = []
    for graph in (True, False):
        hs.set_dt(dt)
        hs.set_graph(graph)
        hs.set_T(T)
        it, rel, _ = hs.solve(1e-10, 200)
        runs.append((int(it[0]), float(rel[0]), hs.get_T(0)))
    print("[heat large]", np_, runs[0][:2], flush=True)
    x = runs[0][2]
    b = hs.apply(np.ones_like(T)) * T          # rows of A sum to V/dt (insulated boundaries)
    assert np.linalg.norm(b - hs.apply(x[None])) / np.linalg.norm(b) < 2e-10
    assert runs[0][1] <= 1e-10
    assert runs[0][:2] == runs[1][:2] and np.array_equal(x, runs[1][2])
    h2 = HeatSolver(s, 1.0, 0.7, 2)
    h2.set_dt(np.array([100.0 * h2.dt_explicit, dt]))
    h2.set_T(np.concatenate([0.5 * T, T]))
    it, rel, _ = h2.solve(1e-10, 200)
    assert (int(it[1]), float(rel[1])) == runs[0][:2] and np.array_equal(h2.get_T(1), x)
