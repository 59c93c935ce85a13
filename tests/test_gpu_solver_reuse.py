"""One solver used again: what a solve or an operator call left behind does not
reach the next solve."""
import numpy as np
import pytest

from falcon_amd import Cnn, HeatSolver, Pfss, Shell, configs

pytestmark = pytest.mark.gpu

LAY = configs.cubic((16, 32, 96), 16)


def _heat(mode):
    s = Shell(LAY)
    hs = HeatSolver(s, 1.0, 0.7, 2)
    if mode != "plain":
        Cnn(s, seed=3)
        hs.attach_corrector()
        hs.set_learned_blockstep(mode == "blockstep")
    hs.set_dt(np.array([30.0, 100.0]) * hs.dt_explicit)
    return hs


@pytest.mark.parametrize("mode", ["plain", "blockstep", "systemstep"])
@pytest.mark.parametrize("left_by", ["solve", "apply"])
def test_heat_solve_after_non_finite_input(mode, left_by):
    """A system that once held a NaN or an infinity solves finite data as a
    fresh solver does, bit for bit."""
    learned = mode != "plain"
    T = 1e-3 * np.random.default_rng(5).standard_normal((2,) + _heat(mode).shape[1:])
    bad = T.copy()
    bad[0, 0, 3, 2, 1], bad[1, 1, 0, 0, 0] = np.nan, np.inf
    hs = _heat(mode)
    if left_by == "solve":
        hs.set_T(bad)
        _, rel, _ = hs.solve(1e-10, 50, use_corrector=learned)
        assert not np.isfinite(rel).any()
    else:
        hs.apply(bad)
    print("[solver reuse]", mode, left_by, flush=True)
    hs.set_T(T)
    it, rel, _ = hs.solve(1e-10, 200, use_corrector=learned)
    fresh = _heat(mode)
    fresh.set_T(T)
    it0, rel0, _ = fresh.solve(1e-10, 200, use_corrector=learned)
    assert (rel0 <= 1e-10).all()
    assert np.array_equal(it, it0) and np.array_equal(rel, rel0)
    for k in range(2):
        assert np.array_equal(hs.get_T(k), fresh.get_T(k))


def test_pfss_solve_after_a_non_finite_magnetogram():
    pf, fresh = Pfss(Shell(LAY)), Pfss(Shell(LAY))
    br = np.random.default_rng(6).standard_normal(pf.mshape)
    bad = br.copy()
    bad[0, 2, 3] = np.nan
    pf.set_magnetogram(bad)
    assert not np.isfinite(pf.solve(1e-10, 50)[1])
    for p in (pf, fresh):
        p.set_magnetogram(br)
        assert p.solve(1e-10, 500)[1] <= 1e-10
    assert np.array_equal(pf.phi(), fresh.phi()) and np.array_equal(pf.field(), fresh.field())


def test_a_solve_leaves_its_core_to_other_threads():
    """The host waits for each iteration's convergence test asleep: 200
    iterations of about 0.4 ms take less than half of their time on the core
    (graph launches of about 10 us and one look in 55 us are a few percent)."""
    import time
    hs = HeatSolver(Shell(configs.SHELL_64x128x384_B16), 1.0, 0.7, 1)
    hs.set_dt(100.0 * hs.dt_explicit)
    hs.seed_T(3, 1e-3)
    hs.solve(0.0, 5)
    cpu = time.thread_time()
    sec = hs.solve(0.0, 200)[2]
    cpu = time.thread_time() - cpu
    print("[solver reuse] core", cpu / sec, flush=True)
    assert cpu < 0.5 * sec


@pytest.mark.parametrize("edge", [4, 16])
def test_operator_of_a_solver_without_a_time_step(edge):
    """Before the first set_dt 1/dt is 0: the diagonals that the set-up makes are
    those of the pure diffusion operator, in every new solver."""
    import pyoracle
    lay = {"ni": edge, "nj": edge, "nk": edge, "ng": 2, "r_rsun": configs.R_RANGE, "ops": [("split", (2, 4, 12))]}
    H = pyoracle.HeatOracle(pyoracle.Oracle(lay), 1.0, 0.7)
    s = Shell(lay)
    x = np.random.default_rng(edge).standard_normal((1, s.nblocks, edge, edge, edge))
    want = H.apply(float("inf"), x[0])
    for _ in range(5):
        assert np.array_equal(HeatSolver(s, 1.0, 0.7, 1).apply(x)[0], want)
