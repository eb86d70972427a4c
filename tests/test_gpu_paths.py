"""Where a rule picks between kernels: both sides of each line against the
oracle.

Tolerances: the parity bars of the two forms, 1e-10 (FP64) and 1e-5 (mixed)
of the largest force."""
import numpy as np
import pytest

from gpu_util import note, pair, rel, rel_force_err
from mdff_amd import capi, configs

pytestmark = pytest.mark.gpu

TOL = {capi.PREC_FP64: 1e-10, capi.PREC_MIXED: 1e-5}
PRECS = pytest.mark.parametrize("prec", [capi.PREC_FP64, capi.PREC_MIXED], ids=["fp64", "mixed"])


def _lj(ncell, p=6.0, q=12.0, rc=2.5):
    s = configs.fcc_lj(ncell=ncell, L=1.5414361 * ncell, rc=rc)
    s.pos = s.pos + np.random.default_rng(5).normal(0.0, 0.04, s.pos.shape)
    capi.set_pair(s.desc, "plj", 1, 1, p)
    capi.set_pair(s.desc, "qlj", 1, 1, q)
    return s


@PRECS
@pytest.mark.parametrize("p,q", [(6, 12), (7, 12), (6, 9), (0, 12), (10, 24), (5.5, 11.0), (30, 254), (30, 256)])
def test_lj_exponents(p, q, prec):
    """Even exponents below 256 by squaring, the others by pow.  A power of
    a rounded number carries k times its rounding, in both."""
    s = _lj(4, float(p), float(q))
    note(f"lj {p} {q}")
    g, o = pair(s, precision=prec)
    (fg, tg), (fo, to) = g.engforce(), o.engforce()
    assert rel_force_err(fg, fo) < TOL[prec] * (1 if q < 30 else 10)
    assert abs(tg["u_lj"] - to["u_lj"]) <= TOL[prec] * abs(to["u_lj"]) * (1 if q < 30 else 10)


@PRECS
@pytest.mark.parametrize("ncell", [10, 11])
def test_lj_lanes(ncell, prec):
    """4,000 and 5,324 atoms: 32 and 16 lanes an atom."""
    s = _lj(ncell)
    note(f"lj n={s.natm}")
    g, o = pair(s, precision=prec)
    assert rel_force_err(g.engforce()[0], o.engforce()[0]) < TOL[prec]


@PRECS
@pytest.mark.parametrize("cells", [(16, 16, 15), (16, 16, 16)], ids=["64_lanes", "16_lanes"])
def test_dipole_field_lanes(cells, prec):
    """30,720 and 32,768 ions: 64 and 16 lanes an ion in the dipoles' field."""
    s = configs.mgo_pim(cells=cells, rcut=4.2, kmax=2, tol=1e-9, alpha=0.8, skin=0.3)
    note(f"mgo n={s.natm}")
    g, o = pair(s, precision=prec)
    assert rel_force_err(g.engforce()[0], o.engforce()[0]) < TOL[prec]


def _long_mesh(k, dip):
    s = configs.nacl(ncell=2, alpha=0.9)
    s.desc.kES[:] = list(k)
    if dip:
        d = s.desc
        d.dip[0 + 16 * 0], d.dip[0 + 16 * 1], d.dip[0 + 16 * 2] = 0.11, -0.05, 0.07
        d.dip[1 + 16 * 0], d.dip[1 + 16 * 1], d.dip[1 + 16 * 2] = -0.04, 0.09, 0.13
    return s


@pytest.mark.parametrize("mesh", ["0", "1"], ids=["direct", "mesh"])
@pytest.mark.parametrize("k,dip", [((2, 3, 60), False), ((2, 3, 52), True), ((3, 2, 101), True), ((410, 2, 2), False),
                                   ((3, 420, 2), True)])
def test_mixed_long_k_mesh(k, dip, mesh, monkeypatch):
    """k meshes that the mixed form takes and whose tiles need more than 64
    KiB of LDS in the direct kernels."""
    monkeypatch.setenv("MDFF_RECIP_MESH", mesh)
    s = _long_mesh(k, dip)
    note(f"long mesh {k} {dip}")
    g, o = pair(s, precision=capi.PREC_MIXED)
    assert rel_force_err(g.engforce()[0], o.engforce()[0]) < TOL[capi.PREC_MIXED]


@pytest.mark.parametrize("dip", [False, True], ids=["charges", "dipoles"])
@pytest.mark.parametrize("kz", [1, 8, 9, 12, 16, 17, 24, 25, 32, 33, 40, 50, 56])
def test_second_moments(kz, dip, monkeypatch):
    """Every size of the matrix-core gather: forces and field gradient."""
    if dip and kz > 50:
        pytest.skip("dipole forces take kES(3) up to 50")
    monkeypatch.setenv("MDFF_RECIP_MESH", "0")
    s = _long_mesh((2, 3, kz), dip)
    note(f"second moments {kz} {dip}")
    g, o = pair(s, doefg=1)
    assert rel_force_err(g.engforce()[0], o.engforce()[0]) < TOL[capi.PREC_FP64]
    assert rel(g.get_efg(), o.get_efg()) < TOL[capi.PREC_FP64]


@pytest.mark.parametrize("mesh", ["0", "1"], ids=["direct", "mesh"])
@pytest.mark.parametrize("prec,k,dip", [(capi.PREC_FP64, (2, 3, 60), False), (capi.PREC_FP64, (2, 3, 51), True),
                                        (capi.PREC_FP64, (410, 2, 2), False), (capi.PREC_MIXED, (2, 3, 102), False)])
def test_too_long_k_mesh_refused(prec, k, dip, mesh, monkeypatch):
    monkeypatch.setenv("MDFF_RECIP_MESH", mesh)
    s = _long_mesh(k, dip)
    note(f"refused mesh {k} {dip}")
    g, _ = pair(s, precision=prec)
    with pytest.raises(RuntimeError, match="too large"):
        g.engforce()
