"""The batched fit as it runs on the GPU (the iterations' reciprocal field on the
matrix cores) built for the host (tests/emu/hip_cpu_wave.h) and checked on the
CPU against the same with the vector-ALU iterations in their place: every compiled size of
the gather and the structure factor, remainders of chunks, splits and tiles,
snapshots without polarisable ions.  Device arrays and LDS end at a guard page,
so an access past their end ends the process; each problem runs in one of its
own.  The GPU tests (tests/test_fit.py, tests/test_gpu_paths.py) repeat the
checks on the device."""
from __future__ import annotations

import copy
import ctypes as C
import json
import shutil
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

HERE = Path(__file__).resolve().parent
if __name__ == "__main__":
    sys.path[:0] = [str(HERE.parent), str(HERE)]

from mdff_amd import capi, configs
from mdff_amd import fit as F

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")

PARAMS = [("A", 1, 2), ("RHO", 1, 2), ("A", 2, 2), ("RHO", 2, 2), ("C", 2, 2), ("ALPHA", 2, 0), ("TTB", 2, 1),
          ("TTC", 2, 1)]
STEP = 0.03 * np.array([1, -1, 0.5, 0.7, -0.8, 1, -0.6, 0.9])

# (cells, kES) of the snapshots of a problem
PROBLEMS = {
    # 4, 6, 8 and 10 K steps of the gather; one to five row tiles of the structure factor
    "short": [((2, 2, 2), (4, 4, 3)), ((2, 2, 3), (3, 4, 5)), ((2, 2, 2), (2, 5, 7)), ((2, 2, 2), (5, 1, 9))],
    # 12, 13, 15 and 17
    "middle": [((2, 2, 2), (3, 2, 11)), ((2, 2, 2), (1, 3, 12)), ((2, 2, 2), (2, 2, 14)), ((2, 2, 2), (2, 2, 16))],
    # 25, alone in its launch, beside a short one; rows (nx, ny) of one and of three
    "long": [((2, 2, 2), (2, 2, 24)), ((2, 2, 2), (1, 0, 17)), ((2, 2, 2), (3, 1, 4))],
    # several chunks of ions and splits of the gather, and the field's 256 threads' remainder
    "chunks": [((3, 3, 3), (5, 5, 5)), ((2, 3, 3), (6, 7, 2))],
    # beyond the matrix-core gather: every snapshot on the vector-ALU kernels
    "beyond": [((2, 2, 2), (2, 2, 25)), ((2, 2, 2), (3, 3, 3))],
    # a snapshot without a polarisable ion among others
    "bare": [((2, 2, 2), (3, 3, 3)), ("mg", (2, 2, 5)), ((2, 2, 2), (2, 3, 4))],
}


def _snapshots(name):
    out = []
    for k, (cells, kes) in enumerate(PROBLEMS[name]):
        bare = cells == "mg"
        s = configs.mgo_pim(cells=(2, 2, 2) if bare else cells, seed=31 + k, sigma=0.08)
        d = s.desc
        w = 0.5 * min(d.cell[0], d.cell[4], d.cell[8])
        d.cutshortrange = d.cutlongrange = 0.99 * w
        d.alphaES = 2.6 / w
        d.kES[:] = list(kes)
        d.conv_tol_ind = 1e-5
        d.max_scf_pol_iter = 40
        if bare:
            m = s.itype == 1
            s = configs.System("mg", copy.deepcopy(d), s.itype[m], s.pos[m], s.vel[m])
            s.desc.natm = int(m.sum())
        out.append(s)
    return out


def _evaluate(lib, name):
    snaps = _snapshots(name)
    theta = F.theta_of(PARAMS, configs.FIT_THETA_STAR) * (1.0 + STEP)
    rng = np.random.default_rng(3)
    n = sum(s.natm for s in snaps)
    P = F.FitProblem(snaps, PARAMS, scf_tol=1e-5, max_iter=40, lib=lib)
    P.set_targets(rng.normal(0, 1, (n, 3)), rng.normal(0, 1, (len(snaps), 9)), 0.05)
    P.set_launch(64, 1)
    out = {}
    for prec in ("FP64", "MIXED"):
        r = P.eval(theta, getattr(capi, "PREC_" + prec), grad=True, outputs=True)
        out[prec] = {"loss": [r.loss], "grad": r.grad.tolist(), "forces": np.ravel(r.forces).tolist(),
                     "stress": np.ravel(r.stress).tolist(), "nscf": np.ravel(r.nscf).tolist()}
    P.close()
    return out


def _run(which, name):
    r = subprocess.run([sys.executable, __file__, which, name], capture_output=True, text=True, timeout=900,
                       cwd=HERE.parent)
    assert r.returncode == 0, (which, name, r.returncode, r.stderr[-2000:])
    return json.loads(r.stdout.splitlines()[-1])


@pytest.fixture(scope="module")
def built():
    sys.path.insert(0, str(HERE / "emu"))
    import build_fit_wave
    return build_fit_wave.build()


@pytest.mark.parametrize("name", list(PROBLEMS))
def test_matrix_core_iterations_match_vector_ones(built, name):
    """FP64: the same iteration counts, and forces, stress, loss and gradient to
    1e-10 (the same iterations, summed in FP64 in different orders).  Mixed:
    the vector iterations sum phases in FP32, 1e-5 and for the gradient 1e-3, the
    form's bars."""
    a, b = _run("valu", name), _run("wave", name)
    for key, tol in (("loss", 1e-10), ("forces", 1e-10), ("stress", 1e-10), ("grad", 1e-9)):
        x, y = np.array(a["FP64"][key]), np.array(b["FP64"][key])
        assert np.isfinite(y).all() and np.abs(x - y).max() <= tol * np.abs(x).max(), key
    assert a["FP64"]["nscf"] == b["FP64"]["nscf"]
    for key, tol in (("loss", 1e-4), ("forces", 1e-5), ("stress", 1e-5), ("grad", 1e-3)):
        x, y = np.array(b["FP64"][key]), np.array(b["MIXED"][key])
        assert np.abs(x - y).max() <= tol * np.abs(x).max(), key


if __name__ == "__main__":
    lib = C.CDLL(str(HERE / "emu" / "_build" / f"libfit_{sys.argv[1]}.so"))
    print(json.dumps(_evaluate(lib, sys.argv[2])))
