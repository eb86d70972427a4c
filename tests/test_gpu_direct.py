"""The direct reciprocal sums (recip.hip) at the ends of their launch shapes,
against the oracle: few ions in a large k mesh, whose gather has more than 64
splits.

Tolerances: the parity bar of the FP64 form, 1e-10 of the largest force,
gradient and of the energies."""
import numpy as np
import pytest

import gpu_util as G
from mdff_amd import capi, configs

pytestmark = pytest.mark.gpu


def _nacl(k, alpha, dip, ncell=2):
    s = configs.nacl(ncell=ncell, alpha=alpha)
    d = s.desc
    d.kES[:] = list(k)
    if dip:
        d.dip[0 + 16 * 0], d.dip[0 + 16 * 1], d.dip[0 + 16 * 2] = 0.11, -0.05, 0.07
        d.dip[1 + 16 * 0], d.dip[1 + 16 * 1], d.dip[1 + 16 * 2] = -0.04, 0.09, 0.13
    return s


@pytest.mark.parametrize("dip", [False, True], ids=["charges", "dipoles"])
@pytest.mark.parametrize("k", [(40, 40, 40), (33, 14, 9), (90, 30, 5)])
def test_few_ions_in_a_large_mesh(k, dip, monkeypatch):
    monkeypatch.setenv("MDFF_RECIP_MESH", "0")
    s = _nacl(k, 1.5, dip)
    G.note(f"direct {k} {dip}")
    g, o = G.pair(s, doefg=1, doefield=1)
    (fg, tg), (fo, to) = g.engforce(), o.engforce()
    assert G.rel_force_err(fg, fo) < 1e-10
    assert not G.compare_terms(tg, to, 1e-10)
    assert G.rel(g.get_efg(), o.get_efg()) < 1e-10
    g.close()
