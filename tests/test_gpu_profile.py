"""falcon_profile_step: every kind of launch timed on its own, on real steps."""
import numpy as np
import pytest

from falcon_amd import Shell, configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,pull", [("fp64", True), ("glm", True), ("fp32", True), ("fp32", False)])
@pytest.mark.parametrize("fixed_dt", [0.0, 10.0])
def test_profiled_steps_are_steps_with_every_kind_timed(prec, pull, fixed_dt):
    def shell():
        s = Shell(configs.small_mixed())
        s.background_polytrope(20.0)
        s.set_gc_all()
        s.set_precision("fp32" if prec == "fp32" else "fp64")
        s.set_ghost_pull(pull)
        if prec == "glm":
            s.set_divb(1)
        s.init_synthetic(seed=3, s_amp=1e-4, b_ratio=1e-3)
        if fixed_dt:
            s.set_fixed_dt(fixed_dt)
        return s

    a, b = shell(), shell()
    print("[profile]", prec, pull, fixed_dt, flush=True)
    ms = a.profile_step(3, 0.5)
    b.advance(3, 0.5)
    assert all(ms[k] > 0.0 for k in ("dt", "boundary", "stage", "exchange_stage", "exchange_state", "diffusion")), ms
    assert ms["step"] >= ms["dt"] + 4 * (ms["boundary"] + ms["stage"]) + ms["diffusion"]
    for ib in range(a.nblocks):
        assert np.array_equal(a.get_state(ib), b.get_state(ib)), ib
        if prec == "glm":
            assert np.array_equal(a.get_psi(ib), b.get_psi(ib)), ib
    # and the steps after them
    a.advance(2, 0.5)
    b.advance(2, 0.5)
    assert all(np.array_equal(a.get_state(ib), b.get_state(ib)) for ib in range(a.nblocks))
