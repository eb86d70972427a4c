"""Builds the CPU emulation of the batched fit with its matrix-core iterations,
and once more with the vector-ALU ones in their place (test infrastructure):
mdff_amd/csrc/fit.hip compiled for the host against tests/emu/hip_cpu_wave.h.
Output: tests/emu/_build/libfit_wave.so and libfit_valu.so."""
from __future__ import annotations

import subprocess
from pathlib import Path

HERE = Path(__file__).resolve().parent
ROOT = HERE.parents[1]
OUT = HERE / "_build"


def build() -> list[Path]:
    OUT.mkdir(exist_ok=True)
    src = (ROOT / "mdff_amd" / "csrc" / "fit.hip").read_text()
    subs = [
        ('#include "common.h"', '#include "hip_cpu_wave.h"'),
        ("extern __shared__ double red[];", "double* red = g_shared;"),
        ("__attribute__((ext_vector_type(4)))", "__attribute__((vector_size(32)))"),
        ("__attribute__((amdgpu_waves_per_eu(2)))", ""),
        ("__attribute__((amdgpu_waves_per_eu(LONG ? 1 : 2)))", ""),
    ]
    for a, b in subs:
        if a not in src:
            raise RuntimeError(f"fit.hip changed: {a!r} not found")
        src = src.replace(a, b)
    rule = "bool mma = fit_sk_lds(f->ncol_max) <= 65536;"
    if rule not in src:
        raise RuntimeError(f"fit.hip changed: {rule!r} not found")
    libs, jobs = [], []
    for name, text in (("wave", src), ("valu", src.replace(rule, "bool mma = false;"))):
        cpp = OUT / f"fit_{name}.cpp"
        cpp.write_text(text)
        libs.append(OUT / f"libfit_{name}.so")
        cmd = ["g++", "-std=c++20", "-O1", "-mfma", "-fPIC", "-shared", "-pthread", f"-I{HERE}", f"-I{ROOT / 'include'}",
               "-o", str(libs[-1]), str(cpp)]
        jobs.append(subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True))
    for j in jobs:
        out = j.communicate()[0]
        if j.returncode != 0:
            raise RuntimeError("CPU build of fit.hip failed:\n" + out[-4000:])
    return libs


if __name__ == "__main__":
    print(build())
