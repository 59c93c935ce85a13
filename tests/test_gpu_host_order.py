"""Vectors crossing the host boundary: the caller's Fortran order (i fastest)
against the device layouts, turned on the GPU."""
import numpy as np
import pytest

from falcon_amd import HeatSolver, Shell, configs

pytestmark = pytest.mark.gpu


def _shell(edges):
    return Shell({"ni": edges[0], "nj": edges[1], "nk": edges[2], "ng": 2, "r_rsun": configs.R_RANGE,
                  "ops": [("split", (1, 2, 6))]})


# rows (I, J) around a multiple of 64, K around a multiple of 4, a block whose
# variables (68 x 36 x 52 cells, 1.02 MB) are so large that each half of the
# staging buffer holds one of them
@pytest.mark.parametrize("edges", [(4, 4, 4), (5, 7, 6), (12, 12, 13), (13, 11, 9), (64, 32, 48)])
def test_state_and_psi_read_back(edges):
    s = _shell(edges)
    s.background_polytrope(20.0)
    s.set_gc_all()
    s.set_divb(1)
    rng = np.random.default_rng(1)
    for b in (0, s.nblocks - 1):
        u = rng.standard_normal((8,) + s.pad[::-1])
        p = rng.standard_normal(s.pad[::-1])
        u[3, 0, 0, 0], u[7, -1, -1, -1], p[-1, 0, -1] = np.nan, np.inf, -0.0
        print("[read back]", edges, b, flush=True)
        s.set_state(b, u)
        s.set_psi(b, p)
        assert np.array_equal(s.get_state(b).view(np.int64), u.view(np.int64))
        assert np.array_equal(s.get_psi(b).view(np.int64), p.view(np.int64))


@pytest.mark.parametrize("m", [2, 4, 8, 16])
@pytest.mark.parametrize("nsys", [1, 3])
def test_heat_vectors_in_callers_order(m, nsys):
    """T in and out in the caller's order: the solution's residual, formed with
    the operator in that order, is the solve's tolerance (1e-10, twice that
    for the recomputed residual's own rounding)."""
    s = _shell((m, m, m))
    hs = HeatSolver(s, 1.0, 0.7, nsys)
    hs.set_dt(50.0 * hs.dt_explicit)
    T = 1e-3 * np.random.default_rng(2).standard_normal(hs.shape)
    print("[heat order]", m, nsys, flush=True)
    hs.set_T(T)
    hs.solve(1e-10, 300)
    x = np.stack([hs.get_T(k) for k in range(nsys)])
    b = hs.apply(np.ones_like(T)) * T          # rows of A sum to V/dt (insulated boundaries)
    for k in range(nsys):
        assert np.linalg.norm((b - hs.apply(x))[k]) / np.linalg.norm(b[k]) < 2e-10
