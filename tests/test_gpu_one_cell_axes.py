"""FP32 path on blocks with one cell along theta or phi: the ghost fill reads
donors at interior cells only."""
import numpy as np
import pytest

from falcon_amd import Shell, configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("edges", [(4, 4, 1), (4, 1, 4), (4, 1, 1), (4, 4, 4)])
def test_ghost_values_do_not_reach_an_fp32_step(edges):
    """Steps from a state whose ghosts hold NaN equal those from filled ghosts."""
    def run(poison):
        s = Shell({"ni": edges[0], "nj": edges[1], "nk": edges[2], "ng": 2, "r_rsun": configs.R_RANGE,
                   "ops": [("split", (2, 3, 9))]})
        s.background_polytrope(20.0)
        s.set_gc_all()
        s.init_synthetic(seed=4, s_amp=1e-4, b_ratio=1e-3)
        if poison:
            for b in range(s.nblocks):
                u = s.get_state(b)
                v = np.full_like(u, np.nan)
                v[:, 2:-2, 2:-2, 2:-2] = u[:, 2:-2, 2:-2, 2:-2]
                s.set_state(b, v)
        s.set_precision("fp32")
        s.set_fixed_dt(1.0)
        print("[one-cell axes]", edges, poison, flush=True)
        s.advance(2, 0.5)
        return np.stack([s.get_state(b) for b in range(s.nblocks)])

    ref, got = run(False), run(True)
    assert np.isfinite(ref).all()
    assert np.array_equal(ref, got)
