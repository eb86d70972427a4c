"""The direct reciprocal sums (recip.hip) at the ends of their launch shapes,
against the oracle: few ions in a large k mesh, whose gather has more than 64
splits; and on the vector-ALU kernels (MDFF_RECIP_VALU=1), which long kES(3) reach
by themselves.

Tolerances: the parity bars, FP64 1e-10 of the largest force, gradient and of
the energies, mixed 1e-5 of the force."""
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


@pytest.mark.parametrize("prec", [capi.PREC_FP64, capi.PREC_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("dip", [False, True], ids=["charges", "dipoles"])
@pytest.mark.parametrize("k", [(8, 7, 9), (3, 11, 16), (12, 2, 1), (2, 3, 50)])
def test_vector_kernels(k, dip, prec, monkeypatch):
    """k_sk, the reduction without the matrix-core operand, and k_gather with
    three and nine moments."""
    monkeypatch.setenv("MDFF_RECIP_VALU", "1")
    s = _nacl(k, 0.9, dip, ncell=3)
    G.note(f"valu {k} {dip} {prec}")
    g, o = G.pair(s, precision=prec, doefg=1, doefield=1)
    (fg, tg), (fo, to) = g.engforce(), o.engforce()
    if prec == capi.PREC_MIXED:
        assert G.rms_force_err(fg, fo) < 1e-5
    else:
        assert G.rel_force_err(fg, fo) < 1e-10
        assert not G.compare_terms(tg, to, 1e-10)
    assert G.rel(g.get_efg(), o.get_efg()) < (1e-10 if prec == capi.PREC_FP64 else 1e-5)
    monkeypatch.setenv("MDFF_RECIP_VALU", "0")
    m, _ = G.pair(s, precision=prec, doefg=1, doefield=1)
    fm = m.engforce()[0]
    assert G.rel_force_err(fg, fm) < 1e-12                   # the same FP64 sums in another order
    g.close()
    m.close()


def test_vector_kernels_with_induced_dipoles(monkeypatch):
    monkeypatch.setenv("MDFF_RECIP_VALU", "1")
    s = configs.mgo_pim(cells=(2, 3, 2), kmax=5)
    G.note("valu induced")
    g, o = G.pair(s)
    (fg, tg), (fo, to) = g.engforce(), o.engforce()
    assert G.rel_force_err(fg, fo) < 1e-10 and tg["n_scf"] == to["n_scf"]
    g.close()
