"""The C-ABI's host logic on recorders of the HIP runtime and of the mechanism
launchers (tests/host/capi_host.cpp): what a call does when something it relies
on is missing, without a GPU."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    if not os.path.exists(HIPCC) or shutil.which("g++") is None:
        pytest.skip("no hipcc or g++")
    d = tmp_path_factory.mktemp("host")
    src = os.path.join(ROOT, "tests", "host", "capi_host.cpp")
    # the host side only, linked against no HIP runtime
    for cmd in ([HIPCC, "-x", "hip", "--cuda-host-only", "-O1", "-fPIE", "-std=c++17", "--offload-arch=gfx950", "-Xclang", "-target-feature",
                 "-Xclang", "-packed-fp32-ops", "-Wno-unused-command-line-argument", "-c", src, "-o", str(d / "h.o")],
                ["g++", str(d / "h.o"), "-o", str(d / "capi_host"), "-lpthread"]):
        r = subprocess.run(cmd, capture_output=True, text=True)
        assert r.returncode == 0, r.stderr[-3000:]

    def run(scenario):
        r = subprocess.run([str(d / "capi_host"), scenario], capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, (r.returncode, r.stdout, r.stderr[-2000:])
        out = {}
        for line in r.stdout.splitlines():
            k, v = line.split(None, 1)
            out[k] = int(v) if v.lstrip("-").isdigit() else v
        return out

    return run


def test_undelivered_statistics_are_an_error(host):
    """The kernel that sums up a call hands its result to host memory.  A call
    whose result does not arrive must not return an earlier call's, and must
    leave nothing behind that spoils the next; the accumulators, which are not
    zero when they are allocated, are cleared on the call's own stream."""
    s = host("undelivered")
    assert s["create"] == 0
    assert s["first"] == 8 and s["clear_at_first"] == 1
    assert s["undelivered"] == -3  # EHIP
    assert s["next"] == 8 and s["clear_at_next"] == 1


def test_noalloc_calls_share_no_accumulators(host):
    """Overlapping pp_chem_react_1d_noalloc calls of two handles race on the
    device scratch and spoil those calls, not every later one."""
    assert host("noalloc_shared")["shared"] == 0


def test_chained_graph_follows_the_counters_layout(host):
    """The per-cell counters are one allocation whose arrays' distances depend
    on its capacity: a graph captured before it grew is not replayed after, also
    where the new allocation has the old address."""
    s = host("graph_counters")
    assert s["captures"] == 1 and s["same_address"] == 1 and s["same_layout"] == 0
    assert s["captures_after_growth"] == 2
    assert s["captures_again"] == 2  # and the new one is kept


@pytest.mark.parametrize("which", [0, 1, 2, 3])
def test_failed_growth_leaves_no_stale_capacity(host, which):
    """A buffer is freed before its larger successor is allocated.  When that
    fails (0, 3: the per-cell counters and the queue order; 1: the staging of
    host arrays; 2: the adjoint's checkpoints), a call of the old size must not
    take the missing buffer for a present one."""
    s = host(f"failed_growth{which}")
    assert s["before"] >= 0 and s["failed"] == -3 and s["after"] >= 0
    assert s["counters"] and s["staging"] and s["checkpoints"]


@pytest.mark.parametrize("mode", [3, 4, 5])
def test_mechanism_without_group_kernels(host, mode):
    """A mechanism too small or too large for a group of lanes per cell has the
    batched forms (3, 4) and ReactorCvode (5) on the one-lane kernels."""
    s = host(f"no_groups{mode}")
    for call, kernel in (("react_1d", "lane_1d"), ("box", "lane_box"), ("chained", "lane_1d"),
                         ("noalloc", "lane_1d")):
        assert s[call] == 0 and s[call + "_kernel"] == kernel and s[call + "_adaptive"] == 1, call
    assert s["rows"] == 0


def test_group_size_there_is(host):
    """A call takes the narrowest group with a lane per equation (large calls
    half of it), or the next size that the mechanism has kernels of."""
    s = host("group_size")
    assert s["drm19_1"] == 2 and s["drm19_10000"] == 4
    assert s["LuEthylene_qss_1"] == 1 and s["LuEthylene_qss_10000"] == 1


def test_workspace_bytes_limits_the_large_mechanisms(host):
    """workspace_bytes is a limit for mechanisms with more than 31 species, whose
    matrices are in device memory, and where the caller names a group size; the
    others' calls took any value before their groups kept Jacobians there."""
    s = host("small_workspace")
    assert s["small_mechanism"] == 0 and s["small_mechanism_cvode"] == 0
    assert s["workspace_lanes"] == 64 * 16  # every wave it can use (two compute units)
    assert s["large_mechanism"] == -1 and s["named_group"] == -1
