"""The transforms (mesh.hip) where their accuracy or their sizes are at a limit:
systems with dipoles that ask for FP64 sums in the mixed form, and k meshes
whose planes do not fit LDS at once.

Tolerances: between sums of FP64 accuracy 1e-12 of the reciprocal energy or
largest force (alias error 4e-15 a direction, measured at three times that,
rounding below 1e-13 on either side); the mixed form's cut-off of 1e-9 shows
in the energy at 1e-10 and above."""
import copy

import numpy as np
import pytest

import gpu_util as G
from mdff_amd import capi, configs

pytestmark = pytest.mark.gpu


def _engine(s, prec, **over):
    d = copy.deepcopy(s.desc)
    d.precision = prec
    for k, v in over.items():
        setattr(d, k, v)
    e = capi.gpu_engine(d, s.itype)
    e.set_positions(s.pos)
    return e


@pytest.mark.parametrize("charges", [True, False], ids=["charges", "dipoles_only"])
@pytest.mark.parametrize("mesh", ["0", "1"], ids=["direct", "mesh"])
def test_mixed_dipoles_in_fp64(charges, mesh, monkeypatch):
    """MDFF_DIP_RECIP_FP64=1, and dipoles without charges: the reciprocal sums
    of the mixed form are the FP64 form's.  Static dipoles, so that both forms
    sum over the same ones."""
    s = configs.mgo_pim(cells=(3, 4, 5))
    s.desc.ldip_polar[:] = [0] * 16
    for k, v in enumerate((0.3, -0.2, 0.25)):
        s.desc.dip[1 + 16 * k] = v
    if not charges:
        s.desc.qch[0] = s.desc.qch[1] = 0.0
    G.note(f"mixed dipoles fp64 {charges} {mesh}")
    monkeypatch.setenv("MDFF_RECIP_MESH", mesh)
    u64 = _engine(s, capi.PREC_FP64).engforce()[1]["u_rec"]
    if charges:
        monkeypatch.setenv("MDFF_DIP_RECIP_FP64", "1")
    u = _engine(s, capi.PREC_MIXED).engforce()[1]["u_rec"]
    assert abs(u - u64) < 1e-12 * abs(u64)
