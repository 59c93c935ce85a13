"""FP64 stage: quotients by the density over the range of dividends, bit for bit
the oracle's."""
import numpy as np
import pytest

import pyoracle
from conftest import random_inputs
from falcon_amd import Shell, configs

pytestmark = pytest.mark.gpu


# entropy whose pressure gradient is, over the density, a normal quotient of a
# dividend between 1e-307 and 1e-300 (its remainder is no normal number), of
# ordinary ones, and of dividends up to 1e287
@pytest.mark.parametrize("lo,hi", [(-302.0, -295.0), (0.0, 10.0), (200.0, 290.0)])
@pytest.mark.parametrize("tile,wgs", [(16, 0), (8, 0), (16, 5)])
def test_pressure_gradient_over_density_bit_exact(lo, hi, tile, wgs):
    print("[division range]", lo, hi, tile, wgs, flush=True)
    lay = configs.small_mixed()
    s, o = Shell(lay), pyoracle.Oracle(lay)
    s.set_gc_all()
    s.set_tiles(0, tile, tile, wgs, wgs)
    rng = np.random.default_rng(8)
    bgs, sts = random_inputs(o.nblocks, lambda ib: o.centres(ib)[0], o.pad, 9)
    for ib in range(o.nblocks):
        st = np.zeros_like(sts[ib])
        st[7] = np.sign(rng.standard_normal(st[7].shape)) * 10.0 ** rng.uniform(lo, hi, st[7].shape)
        st[7][rng.random(st[7].shape) < 0.125] *= 0.0
        s.set_background(ib, bgs[ib]); o.set_background(ib, bgs[ib])
        s.set_state(ib, st); o.set_state(ib, st)
    s.sendrecv_gc(0); o.exchange(0)
    want = np.stack([o.rhs(ib) for ib in range(o.nblocks)])
    assert np.isfinite(want).all() and (np.abs(want[:, 1:4]) > 0).any()
    assert np.array_equal(s.rhs(), want)
