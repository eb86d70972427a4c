#!/usr/bin/env python3
"""Throughput of the engforce path on one MI355X.

Workload (N=1): amorphous SiO2, 24,000 ions (Si +2.4, O -1.2), 2.2 g/cm3,
seeded random packing with 1.4 A minimum separation, Buckingham + Ewald
(rc 10 A, alpha 0.28 1/A, kmax 24), Verlet skin 1 A, velocity-Verlet NVE,
dt 1 fs.  One step = positions update, engforce, velocity update, skin
check (src/integration.f90:132-194 followed by src/tools.f90:444-537).

Both forms run: FP64, and mixed (FP32 pair / field arithmetic with FP64
accumulation, FP64 minimum image, phases, integration).  value = ns/day of
the mixed form; its force error against the FP64 form and the NVE drift of
both are reported with it.  Positions, velocities and all state live in HBM
for the whole timed region.

The cpu_baseline leg times the oracle (the project's FP64 C restatement of
the reference, OpenMP) on a bounded sample of the same workload.
"""
from __future__ import annotations

import argparse
import copy
import ctypes as C
import json
import os
import sys
import time
from pathlib import Path

import numpy as np

ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT))

from mdff_amd import capi, configs  # noqa: E402

PEAK = {"fp32": 157.3, "fp64": 78.6, "fp16": 2500.0}   # MI355X dense TFLOP/s (matrix; FP32 also packed vector)
HBM_PEAK = 8000.0                          # GB/s
# canonical algorithmic flops per unit (counting FMA = 2, sqrt/exp/sin/cos/div = 1)
FLOPS_PER_UNIT = {
    "k_sk": 2.0,           # per (atom, grid point of its 12^3 window): one multiply-add of the spread
    "k_gather": 2.7,       # the value and three derivatives, the two inner axes shared: 2 + 8 / 12
    "k_pair_force": 106.0, # per in-cutoff Buckingham + Ewald q-q pair
}
# the kernel behind each profiler class of the mixed form, and the unit it
# is bound by: the reciprocal sums are FP64 transforms (spread on the FP64
# matrix cores), the pair kernel runs on the FP32 VALU
KERNEL_OF = {"k_sk": "k_mesh_spread<12,false>", "k_gather": "k_mesh_gather<12,3>",
             "k_pair_force": "k_pair_force<float,false,16,2>"}
BOUND_OF = {"k_sk": ("mfma", "fp64"), "k_gather": ("valu", "fp64"), "k_pair_force": ("valu", "fp32")}
# HBM bytes per launch on this workload: rocprofv3 FETCH_SIZE x 1.987 +
# WRITE_SIZE x 0.996 (KiB per dispatch x 1024; the factors calibrate the
# counters on a 256 MiB device-to-device copy), measured with
# mdff_amd.profile_workload (profiles/engforce_sio2_24k_hbm_traffic.md)
TRAFFIC = {"k_pair_force": 63.39e6, "k_sk": 32.49e6, "k_gather": 8.48e6}


NKINDS = 8  # kernel classes of the library's event profiler (mdff_profile_name)


def build_system(natm: int, relax_iters: int):
    """The workload's random packing, relaxed by steepest descent on the GPU
    FP64 path (150 iterations) so that NVE starts from a sane state; the
    velocities are the seeded 300 K Maxwell-Boltzmann set."""
    s = configs.sio2(natm=natm)
    if relax_iters > 0:
        eng = capi.gpu_engine(copy.deepcopy(s.desc), s.itype)
        s.pos, fmax = configs.relax_sd(eng, s.pos, iters=relax_iters)
        eng.close()
        s.extra["relax_fmax"] = fmax
    return s


def count_pairs(pos: np.ndarray, L: float, rc: float) -> int:
    from scipy.spatial import cKDTree
    t = cKDTree(np.mod(pos, L), boxsize=L)
    return int(len(t.query_pairs(rc, output_type="ndarray")))


def run_form(s, precision: int, steps: int, warmup: int, prof_steps: int):
    """Warmup, then `steps` timed VV steps with the event profiler off (the
    throughput), then `prof_steps` more with it on (the per-kernel breakdown:
    event records add stream time, so they stay out of the timed run)."""
    d = copy.deepcopy(s.desc)
    d.precision = precision
    eng = capi.gpu_engine(d, s.itype)
    eng.set_positions(s.pos)
    eng.set_velocities(s.vel)
    f0, t0 = eng.engforce()
    if warmup:
        eng.md_vv(warmup, s.dt)
    t_start = time.perf_counter()
    ek, up = eng.md_vv(steps, s.dt)      # returns after the stream is synchronized
    t_end = time.perf_counter()
    lib = eng.lib
    lib.mdff_profile.argtypes = [C.c_void_p, C.c_int32]
    lib.mdff_profile_read.argtypes = [C.c_void_p, C.POINTER(C.c_double), C.POINTER(C.c_int32), C.c_int32]
    lib.mdff_profile(eng.h, 1)
    eng.md_vv(prof_steps, s.dt)
    ms = (C.c_double * NKINDS)()
    cnt = (C.c_int32 * NKINDS)()
    lib.mdff_profile_read(eng.h, ms, cnt, NKINDS)
    lib.mdff_profile(eng.h, 0)
    lib.mdff_profile_name.restype = C.c_char_p
    names = [lib.mdff_profile_name(k).decode() for k in range(NKINDS)]
    prof = {names[k]: {"ms_total": ms[k], "launches": cnt[k],
                       "ms_avg": (ms[k] / cnt[k]) if cnt[k] else 0.0} for k in range(NKINDS)}
    eng.close()
    return {"f0": f0, "t0": t0, "sec": t_end - t_start, "ek": ek, "up": up, "prof": prof,
            "prof_steps": prof_steps}


def force_errors(f, fref) -> dict:
    """max_i |dF_i| / RMS_i |F_i^ref|, the median per-atom relative error, and
    max |dF| / max |F^ref| over components."""
    dF = np.linalg.norm(f - fref, axis=1)
    nref = np.linalg.norm(fref, axis=1)
    rms = float(np.sqrt(np.mean(nref ** 2)))
    return {"max_over_rms": float(dF.max() / rms),
            "median_per_atom": float(np.median(dF / np.maximum(nref, 1e-30))),
            "max_component_over_max": float(np.abs(f - fref).max() / np.abs(fref).max())}


def drift_per_atom_per_ns(ek, up, natm, dt_fs):
    H = (ek + up) / natm
    t_ns = np.arange(len(H)) * dt_fs * 1e-6
    if len(H) < 3:
        return float("nan")
    return float(np.polyfit(t_ns, H, 1)[0])


def nve_drift_leg(s, equil: int, steps: int) -> dict:
    """NVE energy drift of both forms, outside the timed region: from the
    workload's start, `equil` velocity-Verlet steps, then `steps` more whose
    total energy H(t) = K + U is fitted by a line; the slope per atom per ns
    of each form and their ratio (mixed over FP64)."""
    out = {"equil_steps": equil, "steps": steps, "dt_fs": 1.0}
    for prec, tag in ((capi.PREC_FP64, "fp64"), (capi.PREC_MIXED, "mixed")):
        d = copy.deepcopy(s.desc)
        d.precision = prec
        eng = capi.gpu_engine(d, s.itype)
        eng.set_positions(s.pos)
        eng.set_velocities(s.vel)
        eng.engforce()
        if equil:
            eng.md_vv(equil, s.dt)
        ek, up = eng.md_vv(steps, s.dt)
        eng.close()
        H = (ek + up) / s.natm
        out[tag] = {"drift_eV_per_atom_per_ns": drift_per_atom_per_ns(ek, up, s.natm, 1.0),
                    "H_rms_fluct_eV_per_atom": float(np.std(H)), "H_first_last_eV_per_atom": [float(H[0]), float(H[-1])]}
    d64 = out["fp64"]["drift_eV_per_atom_per_ns"]
    d32 = out["mixed"]["drift_eV_per_atom_per_ns"]
    out["ratio_mixed_over_fp64"] = abs(d32) / abs(d64) if d64 else None
    return out


def term_errors(s) -> dict:
    """Force error of the mixed form against the FP64 form at the workload's
    start, with the short-range term alone (Coulomb off) and the Coulomb
    terms alone (Buckingham off), each normalised by the RMS of the full
    FP64 force."""
    def forces(prec, **over):
        d = copy.deepcopy(s.desc)
        d.precision = prec
        for k, v in over.items():
            setattr(d, k, v)
        eng = capi.gpu_engine(d, s.itype)
        eng.set_positions(s.pos)
        f, _ = eng.engforce()
        eng.close()
        return f
    rms = float(np.sqrt(np.mean(np.sum(forces(capi.PREC_FP64) ** 2, axis=1))))
    out = {}
    for tag, over in (("short_range_only", {"lcoulomb": 0}), ("coulomb_only", {"lbmhft": 0})):
        dF = np.linalg.norm(forces(capi.PREC_MIXED, **over) - forces(capi.PREC_FP64, **over), axis=1)
        out[tag] = {"max_over_rms_of_full": float(dF.max() / rms)}
    return out


def cpu_baseline(s, threads: int, gpu_f64=None, gpu_t64=None, steady: int = 4):
    """The oracle on the GPU box's host cores, bounded sample: one O(N^2)
    list build, one engforce, a first VV step (it rebuilds the lists: the
    saved coordinates start at 0), then `steady` VV steps; value from their
    mean.  The oracle's engforce at the workload's positions is also the
    check of the GPU FP64 form at full size (gpu_f64, gpu_t64)."""
    sys.path.insert(0, str(ROOT / "tests"))
    import oracle_lib
    lib = oracle_lib.lib()
    o = oracle_lib.oracle(copy.deepcopy(s.desc), s.itype)
    lib.orc_set_threads(o.h, threads)
    o.set_positions(s.pos)
    o.set_velocities(s.vel)
    t0 = time.perf_counter()
    o.vnlist_build()
    t1 = time.perf_counter()
    fo, to = o.engforce()
    t2 = time.perf_counter()
    o.md_vv(1, s.dt)
    t3 = time.perf_counter()
    o.md_vv(steady, s.dt)
    t4 = time.perf_counter()
    step = (t4 - t3) / steady
    ns_day = 86400.0 / step * 1e-6 * 1.0
    out = {"value": ns_day, "unit": "ns/day", "cores": threads, "kind": "port",
           "sample": f"oracle (FP64 C restatement of the reference, OpenMP over k-vectors) on the "
                     f"same {s.natm}-ion workload: 1 O(N^2) list build ({t1 - t0:.2f} s), 1 engforce "
                     f"({t2 - t1:.2f} s), a first VV step with its list rebuild ({t3 - t2:.2f} s), "
                     f"then {steady} VV steps ({step:.2f} s each); value from their mean"}
    if gpu_f64 is not None:
        ferr = force_errors(gpu_f64, fo)
        terms = {}
        for k in ("u_bmhft", "u_coul", "u_dir", "u_rec", "u_self"):
            if abs(to[k]) > 0:
                terms[k] = abs(gpu_t64[k] - to[k]) / abs(to[k])
        for k in ("tau_nonb", "tau_coul"):
            ref = np.asarray(to[k])
            terms[k] = float(np.abs(np.asarray(gpu_t64[k]) - ref).max() / max(np.abs(ref).max(), 1e-300))
        out["gpu_fp64_vs_oracle"] = {"force": ferr, "terms_rel": terms}
    return out


def fit_leg(nsnap: int, reps: int) -> dict:
    """fit-gradients/s: 256 PIM oxide snapshots (96-1536 ions), targets from
    the plain FP64 engforce at the hidden parameters, one FP32 forward +
    adjoint gradient over all snapshots per evaluation (one launch)."""
    from mdff_amd import fit as F
    params = [("A", 1, 2), ("RHO", 1, 2), ("A", 2, 2), ("RHO", 2, 2), ("C", 2, 2), ("ALPHA", 2, 0),
              ("TTB", 2, 1), ("TTC", 2, 1), ("TTB", 2, 2), ("TTC", 2, 2)]
    snaps = configs.fit_snapshots(nsnap)
    theta_star = F.theta_of(params, configs.FIT_THETA_STAR)
    theta0 = theta_star * (1.0 + 0.03 * np.array([1, -1, 0.5, 0.7, -0.8, 1, -0.6, 0.9, 0.4, -0.5]))
    t0 = time.perf_counter()
    Fref, Tref = F.plain_targets(snaps)
    t_targets = time.perf_counter() - t0
    P = F.FitProblem(snaps, params)
    P.set_targets(Fref, Tref, 0.05)
    tune = P.autotune(theta0, capi.PREC_MIXED, reps=1)
    r32 = P.eval(theta0, capi.PREC_MIXED, grad=True, outputs=True)
    t0 = time.perf_counter()
    for _ in range(reps):
        P.eval(theta0, capi.PREC_MIXED, grad=True)
    sec = (time.perf_counter() - t0) / reps
    r64 = P.eval(theta0, capi.PREC_FP64, grad=True)
    t0 = time.perf_counter()
    P.eval(theta0, capi.PREC_FP64, grad=True)
    sec64 = time.perf_counter() - t0
    P.close()
    natm = sum(s.natm for s in snaps)
    # roofline of the fit: the reciprocal (k, atom) terms of every dipole-field
    # operator application (SCF and adjoint iterations) and the four other
    # passes (static field, forces, h, its reciprocal part), at the
    # structure-factor and gather figures of the engforce (11 + 10 flops per
    # (k, atom)); pairs left out (under a tenth of the work).  FP64 matrix peak
    # (the iterations' reciprocal field runs there in both forms).
    def nk_of(k):
        return k[2] + k[1] * (2 * k[2] + 1) + k[0] * (2 * k[1] + 1) * (2 * k[2] + 1)
    nkn = np.array([s.natm * nk_of(list(s.desc.kES)) for s in snaps], float)
    passes = r32.nscf[:, 0] + r32.nscf[:, 1] + 4
    fit_flops = float(np.sum(passes * nkn) * 21.0)
    fit_roof = {"kernel": "kf_* phase kernels (iterations: kf_sk, kf_moments)", "bound": "mfma", "achieved": round(fit_flops / sec / 1e12, 3),
                "peak": PEAK["fp64"], "unit": "TFLOP/s", "frac": round(fit_flops / sec / 1e12 / PEAK["fp64"], 4),
                "algorithmic_flops_per_launch": fit_flops, "flops_per_unit": 21.0,
                "units_per_launch": float(np.sum(passes * nkn)), "traffic": None,
                "note": "phase launches over (snapshot, block of atoms or k-vectors); launches per "
                        "evaluation: 22 + 7 per SCF or adjoint iteration of the slowest snapshot"}
    return {"metric": "fit-gradients/s", "value": round(1.0 / sec, 3), "seconds_per_gradient": sec,
            "roofline": fit_roof,
            "fp64_seconds_per_gradient": sec64, "snapshots": nsnap, "ions": natm,
            "sizes": [int(min(s.natm for s in snaps)), int(max(s.natm for s in snaps))],
            "params": len(params), "launch": {"block": tune["block"]},
            "grad_rel_diff_fp32_vs_fp64": float(np.linalg.norm(r32.grad - r64.grad) / np.linalg.norm(r64.grad)),
            "loss_at_start": r64.loss, "scf_iters_max": int(r32.nscf[:, 0].max()),
            "adjoint_iters_max": int(r32.nscf[:, 1].max()), "plain_targets_seconds": t_targets}


def extra_leg(name: str, steps: int) -> dict:
    """cfg3 (LiF 200k, NHC-3) and cfg4 (MgO PIM 12k, NHC): a few steps of
    each form; force error of the mixed form against FP64 at the start."""
    if name == "lif":
        s = configs.lif()
        eng = capi.gpu_engine(copy.deepcopy(s.desc), s.itype)
        s.pos, fmax = configs.relax_sd(eng, s.pos, iters=200)
        eng.close()
    else:
        s = configs.mgo_pim()
    out = {"natm": s.natm, "kmax": list(s.desc.kES)}
    forces = {}
    for prec, tag in ((capi.PREC_FP64, "fp64"), (capi.PREC_MIXED, "mixed")):
        d = copy.deepcopy(s.desc)
        d.precision = prec
        eng = capi.gpu_engine(d, s.itype)
        eng.set_positions(s.pos)
        eng.set_velocities(s.vel)
        f0, t0 = eng.engforce()
        forces[tag] = f0
        xi, vxi = np.zeros(3), np.zeros(3)
        _, _, _, xi, vxi = eng.md_nhcn(2, s.dt, s.temp, 0.1 * capi.TIME_UNIT, xi, vxi)
        ta = time.perf_counter()
        eng.md_nhcn(steps, s.dt, s.temp, 0.1 * capi.TIME_UNIT, xi, vxi)
        sec = (time.perf_counter() - ta) / steps
        out[tag] = {"ms_per_step": round(sec * 1e3, 3), "ns_per_day": round(86400.0 / sec * 1e-6, 3),
                    "n_scf": int(t0["n_scf"])}
        eng.close()
    out["force_error_mixed_vs_fp64"] = force_errors(forces["mixed"], forces["fp64"])
    return out


def main() -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=200)
    ap.add_argument("--warmup", type=int, default=10)
    ap.add_argument("--natm", type=int, default=24000)
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline leg")
    ap.add_argument("--cpu-threads", type=int, default=min(16, os.cpu_count() or 1))
    ap.add_argument("--relax", type=int, default=150, help="steepest-descent iterations before MD")
    ap.add_argument("--no-fit", action="store_true", help="skip the batched-fit leg")
    ap.add_argument("--fit-snapshots", type=int, default=256)
    ap.add_argument("--extra", action="store_true", help="also time the LiF 200k and MgO PIM 12k workloads")
    ap.add_argument("--drift-steps", type=int, default=10000,
                    help="NVE steps per form of the untimed drift leg (0: skip)")
    ap.add_argument("--drift-equil", type=int, default=1000, help="NVE steps before the drift fit")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py: this build runs on one GPU only (asked for {args.gpus}); "
              "the multi-GPU sharding is a design, not a measured path", file=sys.stderr)
        return 2
    s = build_system(args.natm, args.relax)
    dt_fs = 1.0
    L = float(s.desc.cell[0])
    rc = float(s.desc.cutlongrange)
    kmax = list(s.desc.kES)
    nk = kmax[2] + kmax[1] * (2 * kmax[2] + 1) + kmax[0] * (2 * kmax[1] + 1) * (2 * kmax[2] + 1)
    npairs = count_pairs(s.pos, L, rc)

    prof_steps = max(20, min(args.steps, 100))
    r64 = run_form(s, capi.PREC_FP64, args.steps, args.warmup, prof_steps)
    r32 = run_form(s, capi.PREC_MIXED, args.steps, args.warmup, prof_steps)

    ferr_all = force_errors(r32["f0"], r64["f0"])
    ferr = ferr_all["max_over_rms"]
    ms64 = r64["sec"] / args.steps * 1e3
    ms32 = r32["sec"] / args.steps * 1e3
    nsday = lambda ms: 86400.0 / (ms * 1e-3) * dt_fs * 1e-6  # noqa: E731

    # dominant kernel of the mixed form
    prof = r32["prof"]
    dom = max(prof, key=lambda k: prof[k]["ms_total"])
    units = {"k_sk": s.natm * 12**3, "k_gather": s.natm * 12**3, "k_pair_force": npairs}
    roof = None
    if dom in FLOPS_PER_UNIT and prof[dom]["ms_avg"] > 0:
        flops = FLOPS_PER_UNIT[dom] * units[dom]
        sec = prof[dom]["ms_avg"] * 1e-3
        ach = flops / sec / 1e12
        bound, kind = BOUND_OF[dom]
        roof = {"kernel": KERNEL_OF[dom], "bound": bound, "achieved": round(ach, 3), "peak": PEAK[kind],
                "unit": "TFLOP/s", "frac": round(ach / PEAK[kind], 4), "traffic": TRAFFIC.get(dom),
                "algorithmic_flops_per_launch": flops, "avg_launch_ms": prof[dom]["ms_avg"],
                "units_per_launch": units[dom], "flops_per_unit": FLOPS_PER_UNIT[dom]}

    out = {
        "metric": "ns/day mixed vs FP64 on GPU at <=1e-5 rel force err; fit-gradients/s",
        "value": round(nsday(ms32), 3),
        "unit": "ns/day",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms32, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32 pair/field math, f64 reciprocal sums and accumulation",
        "data": "synthetic (seeded random packing)",
        "config": {"workload": f"a-SiO2 {s.natm} ions, Buckingham+Ewald rc {rc} alpha {s.desc.alphaES} "
                               f"kmax {kmax[0]}, skin {s.desc.skindiff}, NVE velocity Verlet dt 1 fs",
                   "natm": s.natm, "nk": nk, "unique_pairs_in_rc": npairs,
                   "prep": f"steepest descent {args.relax} iterations (max|F| after: "
                           f"{s.extra.get('relax_fmax', float('nan')):.3g} eV/A), 300 K velocities"},
        "fp64": {"ns_per_day": round(nsday(ms64), 3), "ms_per_step": round(ms64, 4)},
        "mixed": {"ns_per_day": round(nsday(ms32), 3), "ms_per_step": round(ms32, 4),
                  "max_rel_force_err_vs_fp64": ferr,
                  "force_error_definition": "max_i |F_i(mixed) - F_i(fp64)| / RMS_i |F_i(fp64)|",
                  "force_error_vs_fp64": ferr_all},
        "speedup_mixed_vs_fp64": round(ms64 / ms32, 3),
        "pair_interactions_per_s": npairs / (ms32 * 1e-3),
        "k_terms_per_s": nk * s.natm / (ms32 * 1e-3),
        "kernel_ms_per_step_mixed": {k: round(v["ms_total"] / prof_steps, 4) for k, v in prof.items()},
        "kernel_ms_per_step_fp64": {k: round(v["ms_total"] / prof_steps, 4) for k, v in r64["prof"].items()},
        "kernel_profile_steps": prof_steps,
        "roofline": roof,
        "cpu_baseline": None,
    }
    out["mixed"]["force_error_by_term"] = term_errors(s)
    if args.drift_steps > 0:
        nd = nve_drift_leg(s, args.drift_equil, args.drift_steps)
        out["nve_drift"] = nd
        out["fp64"]["nve_drift_eV_per_atom_per_ns"] = nd["fp64"]["drift_eV_per_atom_per_ns"]
        out["mixed"]["nve_drift_eV_per_atom_per_ns"] = nd["mixed"]["drift_eV_per_atom_per_ns"]
        out["drift_ratio_mixed_over_fp64"] = nd["ratio_mixed_over_fp64"]
    if not args.no_fit:
        out["fit"] = fit_leg(args.fit_snapshots, reps=3)
    if args.extra:
        out["extra"] = {"lif_200k_nhc3": extra_leg("lif", 5), "mgo_pim_12k_nhc": extra_leg("mgo", 10)}
    if not args.no_cpu:
        try:
            out["cpu_baseline"] = cpu_baseline(s, args.cpu_threads, r64["f0"], r64["t0"])
        except Exception as e:  # the GPU result stands on its own
            out["cpu_baseline"] = {"error": str(e)}
    print(json.dumps(out))
    return 0


if __name__ == "__main__":
    sys.exit(main())
