"""Where a rule picks between kernels: both sides of each line against the
oracle.

Tolerances: the parity bars of the two forms, 1e-10 (FP64) and 1e-5 (mixed)
of the largest force."""
import numpy as np
import pytest

from gpu_util import note, pair, rel, rel_force_err
from mdff_amd import capi, configs
from mdff_amd import fit as F

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
@pytest.mark.parametrize("ncell,rc", [(7, 2.5), (10, 2.5), (11, 2.5), (11, 5.4)])
def test_lj_lanes(ncell, rc, prec):
    """1,372, 4,000 and 5,324 atoms, the last with short and long rows: 64, 32,
    16 and 32 lanes an atom."""
    s = _lj(ncell, rc=rc)
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


def _fit_problem(kz, params, nsnap=3):
    snaps = configs.fit_snapshots(nsnap, nmin=64, nmax=260, seed=17)
    for n, s in enumerate(snaps):
        s.desc.kES[:] = [3 + n, 4, kz[n % len(kz)]]
    return snaps, F.FitProblem(snaps, params, scf_tol=1e-12, max_iter=400)


@pytest.mark.parametrize("kz", [(1, 4, 5), (7, 8, 9), (10, 11, 12), (13, 14, 15), (16, 17, 24), (24, 25, 3)],
                         ids=lambda k: "-".join(map(str, k)))
def test_fit_iterations(kz):
    """Dipole iterations over every size of the matrix-core kernels, and the
    vector-ALU ones where a kES(3) is above 24: forces and stress of the single
    configurations (converged to 1e-12; bar of the fit's forward parity)."""
    params = [("A", 1, 2), ("ALPHA", 2, 0)]
    snaps, p = _fit_problem(kz, params)
    note(f"fit kz {kz}")
    f, t = F.plain_targets(snaps, scf_tol=1e-12, max_iter=400)
    p.set_targets(f, t, 1.0)
    r = p.eval(F.theta_of(params, configs.FIT_THETA_STAR), capi.PREC_FP64, grad=False, outputs=True)
    assert rel(r.forces, f) < 1e-9
    assert rel(r.stress, t) < 1e-9
    p.close()


def test_fit_most_parameters():
    """32 parameters, the last of each kind and pair in force: its gradient
    is that of the short list, and the others' is zero."""
    short = [("A", 1, 2), ("RHO", 1, 2), ("A", 2, 2), ("RHO", 2, 2), ("C", 2, 2), ("ALPHA", 2, 0), ("TTB", 2, 1),
             ("TTC", 2, 1)]
    g = []
    for params in (short, short * 4):
        snaps, p = _fit_problem((7, 9, 8), params)
        n = sum(s.natm for s in snaps)
        rng = np.random.default_rng(2)
        p.set_targets(rng.normal(size=(n, 3)), rng.normal(size=(len(snaps), 9)), 0.1)
        note(f"fit {len(params)} parameters")
        g.append(np.asarray(p.eval(F.theta_of(params, configs.FIT_THETA_STAR) * 1.02, capi.PREC_FP64, grad=True).grad))
        p.close()
    assert rel(g[1][24:], g[0]) < 1e-12
    assert not np.any(g[1][:24])


@pytest.mark.parametrize("ncell", [3, 13, 14])
def test_arrays_through_mapped_memory(ncell):
    """108 and 8,788 atoms: arrays go through mapped memory; 10,976: copies.
    Two positions in a row before the device has read the first."""
    s = _lj(ncell)
    note(f"arrays n={s.natm}")
    g, o = pair(s)
    for k in range(3):
        g.set_positions(s.pos + 0.1 * k)
        v = s.pos * (k + 1.0)
        g.set_velocities(v)
    assert np.array_equal(g.get_positions(), s.pos + 0.2)
    assert np.array_equal(g.get_velocities(), v)
    o.set_positions(s.pos + 0.2)
    f = g.engforce()[0]
    assert rel_force_err(f, o.engforce()[0]) < TOL[capi.PREC_FP64]
    assert not np.any(g.get_dipoles()[0])


@pytest.mark.parametrize("rc", [3.3, 5.0, 7.0, 9.0])
@pytest.mark.parametrize("shape", ["perfect", "displaced", "unwrapped", "sheared", "mirrored"])
def test_pair_sets_over_cell_widths(rc, shape):
    """Cells of a third, half and all of the cutoff and axes swept whole, in one
    box of 12.6 x 21.1 x 37.9 A; ions on cell boundaries, far outside the box, a
    box that is not orthogonal and one with a negative axis."""
    s = configs.mgo_pim(cells=(3, 5, 9), rcut=rc, kmax=2, skin=0.4, sigma=0.0 if shape == "perfect" else 0.1)
    A = np.array(s.desc.cell[:]).reshape(3, 3, order="F")
    if shape == "unwrapped":
        s.pos = s.pos + (np.random.default_rng(4).integers(-3, 4, s.pos.shape) @ A.T)
    elif shape == "sheared":
        m = np.array([[1.0, 0.18, -0.07], [0.0, 1.0, 0.11], [0.0, 0.0, 1.0]])
        s.desc.cell[:] = list((m @ A).reshape(-1, order="F"))
        s.pos = s.pos @ m.T
    elif shape == "mirrored":
        m = np.diag([1.0, -1.0, 1.0])
        s.desc.cell[:] = list((A @ m).reshape(-1, order="F"))
        s.pos = s.pos @ m
    note(f"pair sets rc {rc} {shape}")
    g, o = pair(s)
    g.vnlist_build()
    o.vnlist_build()
    for which in (0, 1):
        (pg, lg), (po, lo) = g.get_pairs(which), o.get_pairs(which)
        assert np.array_equal(pg, po) and np.array_equal(lg, lo)
        assert lg.size > 0
