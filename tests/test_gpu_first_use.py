"""Buffers that a call makes are cleared before a stream uses them."""
import numpy as np
import pytest

from falcon_amd import Shell, configs

pytestmark = pytest.mark.gpu

LAY = configs.SHELL_64x128x384_B16      # 800 MB per FP64 buffer


def test_a_new_state_and_psi_read_as_zero():
    s = Shell(LAY)
    s.set_gc_all()
    last = s.get_state(s.nblocks - 1)
    assert not last.any() and not s.get_state(0).any()
    s.set_divb(1)
    assert not s.get_psi(s.nblocks - 1).any() and not s.get_psi(0).any()


@pytest.mark.parametrize("prec", ["fp64", "glm", "fp32"])
def test_the_first_step_does_not_depend_on_when_its_buffers_were_made(prec):
    def step(early):
        s = Shell(LAY)
        s.background_polytrope(20.0)
        s.set_gc_all()
        s.set_precision("fp32" if prec == "fp32" else "fp64")
        if prec == "glm":
            s.set_divb(1)
        s.init_synthetic(seed=5, s_amp=1e-4, b_ratio=1e-3)
        if early:
            s.sendrecv_gc(1)             # makes the stage buffers and waits
        print("[first use]", prec, early, flush=True)
        dt = s.advance_rk4(0.5)
        return dt, np.stack([s.get_state(b) for b in range(0, s.nblocks, 37)])

    a, b = step(True), step(False)
    assert a[0] == b[0] and np.array_equal(a[1], b[1])
