"""Which mechanisms have kernels with a group of lanes per cell, and what the
others have: the table generator and the kernels' sources on synthetic
mechanisms, compiled for gfx950 without a GPU.

A group exists for 4 to 192 equations whose packed tables and areas fit the
160 KB of LDS; a mechanism beyond the packed records (254 species, 4095
reactions) gets no packed tables.  Each of these still compiles, without the
group kernels."""
import concurrent.futures as cf
import dataclasses
import os
import subprocess

import pytest

from pelephysics_amd.build import CFLAGS, CSRC, HIPCC
from pelephysics_amd.mechgen import emit_tables
from pelephysics_amd.mechgen.__main__ import load

UNITS = (("BATCHED", "MODE_BATCHED_MIXED"), ("GFIXED", "MODE_BDF"))
# (species, reactions): group sizes (cells per wave) there are
SYNTHETIC = {(2, 0): (), (4, 1): (8,), (60, 3000): (), (40, 800): (1, 2), (200, 300): (), (260, 200): ()}


def synthetic(ns, nr):
    d = load("drm19")
    el = next(r for r in d.reactions if r.kind == "elementary")
    rx = [dataclasses.replace(el, reactants={j % ns: 1.0, (j + 1) % ns: 1.0}, products={(j + 2) % ns: 1.0})
          for j in range(nr)]
    return dataclasses.replace(d, name=f"syn{ns}_{nr}", reactions=rx,
                               species=[dataclasses.replace(d.species[i % 21], name=f"S{i}") for i in range(ns)])


def _compile(args):
    src, obj = args
    r = subprocess.run([HIPCC, *CFLAGS, "-O1", "-I", CSRC, "-c", src, "-o", obj], capture_output=True, text=True)
    return r.returncode, r.stderr


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_every_mechanism_compiles(tmp_path):
    work = []
    for (ns, nr), sizes in SYNTHETIC.items():
        m = synthetic(ns, nr)
        text = emit_tables.emit(m, "a synthetic mechanism").replace('"../pack.h"', '"pack.h"')
        (tmp_path / f"{m.name}.h").write_text(text)
        assert ("kPack" in text) == (ns <= 254 and nr <= 4095)
        typ = f"ppc::TabMech<ppc::tab::{m.name}>"
        head = f'#include "{tmp_path}/{m.name}.h"\n#include "chem_table.h"\n'
        for kind, mode in UNITS:
            src = tmp_path / f"{m.name}_{mode}_{kind}.hip"
            have = "".join(f"static_assert(ppc::group_ok<{typ}, {64 // c}>() == {str(c in sizes).lower()}, "
                           f'"{c} cells per wave");\n' for c in (8, 4, 2, 1))
            src.write_text(f'{head}#include "launch_impl.h"\n{have}PPC_INSTANTIATE_{kind}({typ}, ppc::{mode})\n')
            work.append((str(src), str(src)[:-4] + ".o"))
    with cf.ThreadPoolExecutor(4) as ex:
        for (src, _), (rc, err) in zip(work, ex.map(_compile, work)):
            assert rc == 0, (os.path.basename(src), err[-2000:])


def test_committed_tables_are_packed():
    from pelephysics_amd.build import MECHS
    for name in MECHS:
        with open(os.path.join(CSRC, "tab", f"{name}.h")) as f:
            assert "kPack" in f.read()
