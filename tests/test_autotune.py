"""Autotuner bookkeeping (no GPU): candidate sets and the tuning table."""
import json

from pelephysics_amd import autotune


def test_candidates():
    for form in ("1d", "box"):
        c = autotune.candidates("drm19", "ReactorBDFAdaptiveMixed", form)
        groups = [x for x in c if x["batched_cells_per_wave"]]
        # the library's choice once per implementation, and nothing it does not read
        assert [x for x in c if not x["batched_cells_per_wave"]] == [
            {"kernels": k, "batched_cells_per_wave": 0} for k in ("drm19", "drm19_table")]
        # group kernels: the table-driven drm19 only, every size
        assert {x["kernels"] for x in groups} == {"drm19_table"}
        assert {x["batched_cells_per_wave"] for x in groups} == set(autotune.GROUPS)
        assert len(groups) == len(autotune.GROUPS) * len(autotune.GROUP_WAVES) * len(autotune.GROUP_LU)
        assert len({tuple(sorted(x.items())) for x in c}) == len(c)
    c = autotune.candidates("dodecane_lu", "ReactorBDFAdaptive")
    assert c == [{"kernels": "dodecane_lu", "batched_waves_per_simd": 0}]
    # the plain adaptive BDF of a register-resident mechanism: three builds per implementation
    c = autotune.candidates("drm19", "ReactorBDFAdaptive", "box")
    assert {(x["kernels"], x["batched_waves_per_simd"]) for x in c} == {
        (k, o) for k in ("drm19", "drm19_table") for o in autotune.PLAIN_OCCUPANCY}


def test_committed_table_holds_what_a_launch_reads():
    with open(autotune.table_path("gfx950")) as f:
        table = json.load(f)
    for name, e in table.items():
        mech, integrator, form = name.split("|")
        known = autotune.candidates(mech, integrator, form)
        keys = {k for c in known for k in c}
        entry = {k: e[k] for k in e if k.startswith("batched") or k == "kernels"}
        assert set(entry) <= keys and entry in known, name


def test_lookup_reads_the_table(tmp_path, monkeypatch):
    p = tmp_path / "t.json"
    p.write_text(json.dumps({"drm19|ReactorBDFAdaptiveMixed|box": {"kernels": "drm19_table",
                                                                    "batched_waves_per_cu": 6}}))
    monkeypatch.setenv("PELE_CHEM_TUNING", str(p))
    e = autotune.lookup("drm19", "ReactorBDFAdaptiveMixed", "box")
    assert e["kernels"] == "drm19_table" and e["batched_waves_per_cu"] == 6
    assert autotune.lookup("drm19", "ReactorBDFAdaptiveMixed", "1d") is None
