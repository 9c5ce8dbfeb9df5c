"""Build the gfx950 chemistry library ``libpele_chem_hip.so`` in-tree.

    python -m pelephysics_amd.build [--jobs N] [--mechs LiDryer drm19]

Steps: regenerate mechanism headers when the reference YAML is available,
write one instantiation unit per (mechanism, integrator) plus a launcher unit
per mechanism, compile them in parallel with hipcc for gfx950, link the
shared library next to this file.
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
INST = os.path.join(CSRC, "inst")
OBJ = os.path.join(HERE, "_build")
LIBNAME = "libpele_chem_hip.so"
LIB = os.path.join(HERE, LIBNAME)
# QSS mechanisms (quasi-steady-state species eliminated in every rate
# evaluation) are compiled table-driven
MECHS = ["LiDryer", "drm19", "dodecane_lu", "heptane_lu_88sk", "CH4_lean_qss", "LuEthylene_qss",
         "dodecane_lu_qss"]
MODES = {"bdf": ("MODE", "MODE_BDF"), "rk64": ("MODE", "MODE_RK64"),
         "adaptive": ("MODE", "MODE_ADAPTIVE"), "erk": ("MODE", "MODE_ERK"),
         "bmixed": ("BATCHED", "MODE_BATCHED_MIXED"),
         "bfp64": ("BATCHED", "MODE_BATCHED_FP64"), "cvode": ("BATCHED", "MODE_GROUP_CVODE"),
         "gfixed": ("GFIXED", "MODE_BDF"), "adjoint": ("ADJOINT", "MODE_BDF"),
         "flatten": ("FLATTEN", "MODE_BDF")}
ARCH = "gfx950"
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
CFLAGS = ["-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}",
          # no packed-FP32 instructions (v_pk_*_f32) in any kernel
          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
          "-Wno-unused-command-line-argument"]


def _write_if_changed(path: str, text: str) -> None:
    if os.path.exists(path):
        with open(path) as f:
            if f.read() == text:
                return
    with open(path, "w") as f:
        f.write(text)


# Two implementations of the small mechanisms: "<mech>" is the fully unrolled
# generated code (mech/<mech>.h), "<mech>_table" walks constant-memory tables
# (chem_table.h, compact code).  The large mechanisms are compiled from the
# tables only, under their plain name.
UNROLLED_CODE = ('#include "../mech/{m}.h"\n', "ppc::mech::{m}")
TABLE_CODE = ('#include "../tab/{m}.h"\n#include "../chem_table.h"\n', "ppc::TabMech<ppc::tab::{m}>")


def impls(m: str) -> dict:
    from .mechgen.__main__ import UNROLLED
    if m in UNROLLED:
        return {"": UNROLLED_CODE, "_table": TABLE_CODE}
    return {"": TABLE_CODE}


def write_units(mechs) -> list:
    os.makedirs(INST, exist_ok=True)
    units = []
    names = []
    for m in mechs:
        for suffix, (inc, typ) in impls(m).items():
            name = m + suffix
            names.append(name)
            inc, typ = inc.format(m=m), typ.format(m=m)
            for mode, (kind, enum) in MODES.items():
                p = os.path.join(INST, f"{name}_{mode}.hip")
                _write_if_changed(p, f'// Generated by pelephysics_amd/build.py: {name} x {mode} kernels.\n'
                                     f'{inc}#include "../launch_impl.h"\n'
                                     f'PPC_INSTANTIATE_{kind}({typ}, ppc::{enum})\n')
                units.append(p)
            p = os.path.join(INST, f"{name}_launcher.hip")
            _write_if_changed(p, f'// Generated by pelephysics_amd/build.py: launcher table for {name}.\n'
                                 f'{inc}#include "../launch.h"\n'
                                 f'PPC_DEFINE_LAUNCHER({name}, {typ})\n')
            units.append(p)
    _write_if_changed(os.path.join(INST, "registry.inc"),
                      "// Generated by pelephysics_amd/build.py: compiled mechanisms.\n" +
                      "".join(f"PPC_MECH({n})\n" for n in names))
    units.append(os.path.join(CSRC, "capi.hip"))
    units.append(os.path.join(CSRC, "manifold.hip"))
    return units


def _compile(src: str) -> str:
    rel = os.path.relpath(src, CSRC).replace(os.sep, "_")
    obj = os.path.join(OBJ, rel[:-4] + ".o")
    cmd = [HIPCC] + CFLAGS + ["-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stderr[-4000:]}")
    return obj


def build(mechs=None, jobs: int = 0, regenerate: bool = True) -> str:
    mechs = list(mechs or MECHS)
    if regenerate and os.path.isdir("/root/reference/Mechanisms"):
        from .mechgen.__main__ import generate
        generate(mechs)
    os.makedirs(OBJ, exist_ok=True)
    units = write_units(mechs)
    jobs = jobs or min(16, os.cpu_count() or 4)
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(_compile, units))
    tmp = LIB + ".tmp"
    cmd = [HIPCC, "-shared", "-fPIC", f"--offload-arch={ARCH}", "-o", tmp] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr[-4000:]}")
    os.replace(tmp, LIB)
    return LIB


def clean() -> None:
    shutil.rmtree(OBJ, ignore_errors=True)


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--jobs", type=int, default=0)
    ap.add_argument("--mechs", nargs="*", default=MECHS)
    ap.add_argument("--no-regen", action="store_true")
    a = ap.parse_args()
    print(build(a.mechs, a.jobs, regenerate=not a.no_regen), file=sys.stderr)
