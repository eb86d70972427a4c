"""Velocity rescale of few and of very many atoms (more than its 1,024 blocks hold
256 each) against numpy in 64 bits.

Tolerance: sums of n terms in FP64, 1e-12 of the largest velocity."""
import numpy as np
import pytest

import gpu_util as G
from mdff_amd import capi, configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("natm", [1, 3, 255, 257, 262144, 262145, 700001])
def test_rescale(natm):
    G.note(f"rescale {natm}")
    base = configs.fcc_lj(ncell=2)
    d = base.desc
    d.natm = natm
    rng = np.random.default_rng(natm)
    v = rng.normal(0.3, 1.0, (natm, 3))
    e = capi.gpu_engine(d, np.ones(natm, np.int32))
    e.set_velocities(v)
    e.rescale_velocities(0.7)
    want = 0.7 * v
    want -= want.mean(axis=0)
    assert np.abs(e.get_velocities() - want).max() < 1e-12 * np.abs(v).max()
    if natm > 1:
        e.set_velocities(v)
        temp, r1, noise = 1.3, 0.4, float(3 * natm - 4)
        conint = e.csvr_rescale(temp, 0.0, r1, noise, 2.0)
        ekin, ndeg = 0.5 * (v * v).sum() * d.mass[0], 3 * natm - 3
        sigma = 0.5 * ndeg * temp
        knew = ekin + sigma * (noise + r1 * r1) / ndeg - ekin      # no correlation time: factor 0
        want = v * np.sqrt(knew / ekin)
        want -= want.mean(axis=0)
        assert np.abs(e.get_velocities() - want).max() < 1e-12 * np.abs(v).max()
        assert abs(conint - (2.0 - (knew - ekin))) < 1e-11 * max(ekin, knew)
    e.close()
