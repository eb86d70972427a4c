"""The transforms (mesh.hip) where their accuracy or their sizes are at a limit:
systems with dipoles that ask for FP64 sums in the mixed form, and k meshes
whose planes do not fit LDS at once.

Tolerances: between sums of FP64 accuracy 1e-12 of the reciprocal energy or
largest force (alias error 4e-15 a direction, measured at three times that,
rounding below 1e-13 on either side); the mixed form's cut-off of 1e-9 shows
in the energy at 1e-10 and above."""
import copy
import ctypes as C

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


def _table_launches(e):
    """Launches of the phase tables (direct sums: one) or of the kernel values
    (transforms: three) of an evaluation."""
    lib = capi.gpu_lib()
    ms, count = (C.c_double * 16)(), (C.c_int32 * 16)()
    lib.mdff_profile_name.restype = C.c_char_p
    lib.mdff_profile(e.h, 1)
    e.engforce()
    lib.mdff_profile_read(e.h, ms, count, 16)
    lib.mdff_profile(e.h, 0)
    return count[[lib.mdff_profile_name(k) for k in range(16)].index(b"k_tables")]


@pytest.mark.parametrize("ncell,k,fp64,mixed", [
    (3, (50, 50, 50), 0, 1),                 # 216 ions: 275/447 us in FP64, 275/247 in the mixed form
    (4, (40, 40, 40), 0, 1),                 # 512: 232/306, 232/205
    (6, (28, 28, 28), 1, 1),                 # 1,728: 224/183, 224/144
    (2, (80, 80, 50), 0, 0),                 # 64: 434/1198, 434/640
    (2, (100, 100, 57), None, 1),            # (mixed only) no matrix-core gather of the direct sums: 1457 at kES 60, 64 ions
])
def test_route_of_few_ions_in_a_large_mesh(ncell, k, fp64, mixed, monkeypatch):
    """The rule weighs the transforms' own work; either way the forces are those of
    both kernels (to the forms' parity bars: splittings this sharp round at 1e-15
    of alpha^2 q^2, a thousand times the forces)."""
    s = configs.nacl(ncell=ncell, alpha=max(0.3, 0.15 * max(k) / ncell))
    s.desc.kES[:] = list(k)
    s.desc.cutshortrange = s.desc.cutlongrange = 5.0
    G.note(f"route {ncell} {k}")
    for prec, mesh in ((capi.PREC_FP64, fp64), (capi.PREC_MIXED, mixed)):
        if mesh is None:
            continue
        monkeypatch.delenv("MDFF_RECIP_MESH", raising=False)
        e = _engine(s, prec)
        f = e.engforce()[0]
        assert (_table_launches(e) > 1) == bool(mesh)
        e.close()
        for mode in ("0", "1"):
            monkeypatch.setenv("MDFF_RECIP_MESH", mode)
            e = _engine(s, prec)
            err = G.rel_force_err(e.engforce()[0], f)
            assert err < (1e-10 if prec == capi.PREC_FP64 else 1e-5)
            e.close()


def _stretched(f, k, dip=False):
    """NaCl with the cell's axes stretched (no two ions nearer than before),
    so that the k mesh's far entries still carry weight."""
    s = configs.nacl(ncell=2, alpha=0.9)
    d = s.desc
    cell = np.array(d.cell[:]).reshape(3, 3)
    s.pos = s.pos @ np.linalg.inv(cell) @ (cell * np.array(f)[:, None])
    d.cell[:] = list((cell * np.array(f)[:, None]).reshape(9))
    d.kES[:] = list(k)
    if dip:
        d.dip[0 + 16 * 0], d.dip[0 + 16 * 1], d.dip[0 + 16 * 2] = 0.11, -0.05, 0.07
        d.dip[1 + 16 * 0], d.dip[1 + 16 * 1], d.dip[1 + 16 * 2] = -0.04, 0.09, 0.13
    return s


@pytest.mark.parametrize("f,k,dip", [
    ((8, 1, 1), (90, 8, 9), False),          # x: all staged at once
    ((24, 1, 1), (260, 8, 9), False),        # x: two slices of the grid and of the modes
    ((27, 1, 1), (290, 8, 9), True),
    ((1, 27, 1), (9, 290, 8), False),        # y: slices of the grid and of the modes
    ((1, 24, 1), (9, 260, 8), True),
    ((2, 14, 5), (20, 160, 50), True),       # y, with four tiles of nz
    ((1, 16, 16), (9, 170, 56), False),
], ids=["x_whole", "x", "x_dip", "y", "y_dip", "yz_dip", "yz"])
def test_sliced_planes_match_direct_sums(f, k, dip, monkeypatch):
    """Meshes too long for LDS: energy, forces, stress and the field of the
    transforms against the direct sums and the oracle, and in the mixed form
    against the oracle."""
    s = _stretched(f, k, dip)
    G.note(f"sliced {f} {k} {dip}")
    out = []
    for mesh in ("0", "1"):
        monkeypatch.setenv("MDFF_RECIP_MESH", mesh)
        e = _engine(s, capi.PREC_FP64, doefield=1)
        out.append((*e.engforce(), e.get_dipoles()[1]))
        again = e.engforce()
        assert np.array_equal(out[-1][0], again[0]) and out[-1][1]["u_rec"] == again[1]["u_rec"]
        e.close()
    (fd, td, ed), (fm, tm, em) = out
    assert np.abs(fm - fd).max() < 1e-12 * np.abs(fd).max()
    assert np.abs(em - ed).max() < 1e-12 * np.abs(ed).max()
    assert abs(tm["u_rec"] - td["u_rec"]) < 1e-12 * abs(td["u_rec"])
    assert np.abs(tm["tau_coul"] - td["tau_coul"]).max() < 1e-12 * np.abs(td["tau_coul"]).max()
    _, o = G.pair(s)
    fo, to = o.engforce()
    assert G.rel_force_err(fm, fo) < 1e-10
    assert not G.compare_terms(tm, to, 1e-10)
    e = _engine(s, capi.PREC_MIXED)
    assert G.rms_force_err(e.engforce()[0], fo) < 1e-5
    e.close()


def test_sliced_planes_take_a_mixed_mesh_beyond_the_fp64_form(monkeypatch):
    """Two slices of the modes in x and three in y."""
    monkeypatch.setenv("MDFF_RECIP_MESH", "1")
    s = _stretched((30, 24, 1), (330, 260, 8))
    G.note("sliced mixed")
    e = _engine(s, capi.PREC_MIXED)
    _, o = G.pair(s)
    fo, to = o.engforce()
    fm, tm = e.engforce()
    assert G.rms_force_err(fm, fo) < 1e-5
    assert abs(tm["u_rec"] - to["u_rec"]) < 1e-8 * abs(to["u_rec"])
    e.close()
