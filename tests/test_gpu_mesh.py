"""The reciprocal sums as non-uniform transforms (mesh.hip) against the oracle
and against the direct kernels, on grids of one tile and more, uneven and
skewed cells, atoms on cell boundaries, charges and dipoles.

Tolerances: FP64, the parity bar of the FP64 form against the oracle (1e-10);
against the direct kernels 1e-12 of the largest force (the grid is chosen for
an alias error of 4e-15 a direction, measured at three times that; rounding
of both sides is below 1e-13).  Mixed: 1e-5, the form's bar; its grid is
chosen for 1e-9, so mesh against direct reciprocal sums on the same FP32 pairs
stays below 2e-6 (the direct mixed sums' own error)."""
import copy

import numpy as np
import pytest

import gpu_util as G
from mdff_amd import capi, configs

pytestmark = pytest.mark.gpu


def _skew(s, t):
    """The system in a skewed cell (same fractional coordinates)."""
    cell = np.array(s.desc.cell[:]).reshape(3, 3)
    frac = s.pos @ np.linalg.inv(cell)
    new = cell.copy()
    new[1, 0] += t * cell[1, 1]
    new[2, 1] -= t * cell[2, 2]
    s.desc.cell[:] = list(new.reshape(9))
    s.pos = frac @ new
    return s


def _nacl(ncell, k, alpha=0.3):
    s = configs.nacl(ncell=ncell, alpha=alpha)
    s.desc.kES[:] = list(k)
    return s


def _uneven():
    s = configs.mgo_pim(cells=(2, 5, 3))
    s.desc.kES[:] = [5, 12, 8]
    return s


def _charges_only(s):
    s.desc.ldip_polar[:] = [0] * 16
    return s


CASES = {
    "one_tile": lambda: _nacl(2, [2, 2, 2]),
    "small_mesh_sharp": lambda: _nacl(2, [4, 3, 5], alpha=0.5),
    "two_tiles": lambda: _nacl(3, [7, 8, 9]),
    "slow_decay": lambda: _nacl(2, [5, 5, 5], alpha=1.2),
    "skewed": lambda: _skew(_nacl(4, [9, 10, 8]), 0.17),
    "uneven": lambda: _charges_only(_uneven()),
    "dipoles": _uneven,
    "dipoles_skewed": lambda: _skew(configs.mgo_pim(cells=(3, 3, 4)), 0.1),
    "two_charges": configs.two_charges,
    "two_dipoles": configs.two_dipoles,
}


def _engine(s, prec, mode, monkeypatch, **over):
    monkeypatch.setenv("MDFF_RECIP_MESH", mode)
    d = copy.deepcopy(s.desc)
    d.precision = prec
    for k, v in over.items():
        setattr(d, k, v)
    e = capi.gpu_engine(d, s.itype)
    e.set_positions(s.pos)
    return e


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("prec", [capi.PREC_FP64, capi.PREC_MIXED], ids=["fp64", "mixed"])
def test_mesh_matches_direct_and_oracle(name, prec, monkeypatch):
    G.note(f"mesh {name} prec {prec}")
    s = CASES[name]()
    m = _engine(s, prec, "1", monkeypatch, doefield=1)
    fm, tm = m.engforce()
    d = _engine(s, prec, "0", monkeypatch, doefield=1)
    fd, td = d.engforce()
    _, o = G.pair(s, doefield=1)
    fo, to = o.engforce()
    scale = max(np.abs(fo).max(), 1e-300)
    if prec == capi.PREC_FP64:
        assert np.abs(fm - fd).max() / scale < 1e-12
        assert G.rel_force_err(fm, fo) < 1e-10
        assert not G.compare_terms(tm, to, 1e-10)
        assert tm["n_scf"] == to["n_scf"]
        for a, b in zip(m.get_dipoles(), o.get_dipoles()):
            assert np.abs(a - b).max() <= 1e-10 * max(np.abs(b).max(), 1e-300)
    else:
        assert G.rms_force_err(fm, fo) < 1e-5
        assert G.rms_force_err(fm, fd) < 2e-6 + G.rms_force_err(fd, fo)
    m.close()
    d.close()


@pytest.mark.parametrize("prec", [capi.PREC_FP64, capi.PREC_MIXED], ids=["fp64", "mixed"])
def test_mesh_boundary_atoms_and_repeat(prec, monkeypatch):
    """Atoms exactly on grid points, cell faces and several cells away; a
    second evaluation and a second context give the same bits."""
    s = _nacl(3, [7, 7, 7])
    L = s.desc.cell[0]
    s.pos[0] = [0.0, 0.0, 0.0]
    s.pos[1] = [L / 2, L / 2 + 3 * L, 0.0]
    s.pos[2] = [L - 1e-15, -2 * L + 2.8, L / 4]
    s.pos[3] = [-1e-18, L / 2, 5 * L + L / 2]
    G.note(f"mesh boundary prec {prec}")
    out = []
    for _ in range(2):
        e = _engine(s, prec, "1", monkeypatch)
        f1, t1 = e.engforce()
        f2, t2 = e.engforce()
        assert np.array_equal(f1, f2) and t1["u_coul"] == t2["u_coul"]
        out.append(f1)
        e.close()
    assert np.array_equal(out[0], out[1])
    _, o = G.pair(s)
    fo, _ = o.engforce()
    assert G.rms_force_err(out[0], fo) < (1e-10 if prec == capi.PREC_FP64 else 1e-5)


def test_mesh_trajectory_follows_oracle(monkeypatch):
    """20 velocity-Verlet steps with list rebuilds: bins re-made every step."""
    monkeypatch.setenv("MDFF_RECIP_MESH", "1")
    s = _nacl(3, [7, 7, 7])
    s.desc.skindiff = 0.05
    G.note("mesh trajectory")
    g, o = G.pair(s)
    for e in (g, o):
        e.engforce()
    a, b = g.md_vv(20, s.dt), o.md_vv(20, s.dt)
    assert np.abs(a[1] - b[1]).max() / np.abs(b[1]).max() < 1e-10
    assert np.abs(g.get_positions() - o.get_positions()).max() < 1e-9
    g.close()
