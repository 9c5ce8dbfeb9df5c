"""The group-of-lanes kernels where the library chooses them, at the counts
where a wave, a block or the choice itself has a remainder (16 or 32 cells of
four waves share a block; a call's last wave has idle groups).

* A cell's arithmetic does not depend on the cells beside it, so the first n
  cells of a larger call and a call of those n cells give the same bits.
* The larger call meets the criterion of the parity tests against the oracle,
  |x - x_ref| <= 1e-6 |x_ref| + 1e-10, and takes the steps of the
  one-lane-per-cell kernels: exactly for the fixed-step integrators, and for
  the adaptive BDF the total to 5% (the same step, order and Newton logic on a
  Newton matrix that is the same up to rounding; one wrong reaction in the
  Jacobian multiplied the steps by 25).
"""
import numpy as np
import pytest

import oracle
from pelephysics_amd import workloads as W
from test_gpu_parity import _torch, _compare_y, _oracle_1d, _run_1d

pytestmark = pytest.mark.gpu

COUNTS = (1, 3, 17, 63, 65)
ADAPTIVE = [("drm19", "ReactorBDFAdaptiveMixed"), ("drm19", "ReactorBDFBatchedFP64"), ("drm19", "ReactorCvode"),
            ("LiDryer", "ReactorBDFAdaptiveMixed"), ("CH4_lean_qss", "ReactorBDFAdaptiveMixed"),
            ("LuEthylene_qss", "ReactorBDFAdaptiveMixed"), ("LuEthylene_qss", "ReactorBDFBatchedFP64"),
            ("LuEthylene_qss", "ReactorCvode"), ("dodecane_lu_qss", "ReactorBDFAdaptiveMixed")]


def _cells(models, mech, n=66):
    m = models[mech]
    st = W.premixed(m, n, W.SEED) if mech != "LiDryer" else W.lidryer_h2air(m, n)
    return m, st, np.zeros((st.ncells, m.n_species)), np.zeros(st.ncells)


def _prefixes(run, st, neq, y, counts):
    for n in counts:
        yn = run(W.subsample(st, np.arange(n)))
        assert (yn.reshape(n, neq) == y.reshape(-1, neq)[:n]).all(), n


@pytest.mark.parametrize("mech,ident", ADAPTIVE)
def test_adaptive_counts(models, oracles, mech, ident):
    torch = _torch()
    m, st, ysrc, esrc = _cells(models, mech)
    tol = dict(rtol=1e-12, atol=1e-18) if mech == "LiDryer" else dict(rtol=1e-10, atol=1e-16)

    def run(s, ident=ident):
        z = np.zeros((s.ncells, m.n_species))
        _, y, _, R = _run_1d(torch, mech, ident, s, z, np.zeros(s.ncells), 1e-5, **tol)
        run.stats = R.stats()
        assert run.stats["nfailed"] == 0
        return y

    y = run(st)
    work = run.stats
    p = oracle.adapt_params(rtol=1e-13, atol=1e-20)
    _, oy, _, _ = _oracle_1d(oracles[mech], "adaptive", st, ysrc, esrc, 1e-5, params=p)
    _compare_y(m.n_species + 1, y, oy)
    _prefixes(run, st, m.n_species + 1, y, COUNTS)
    if ident != "ReactorCvode":  # its age limit and tolerances are its own
        run(st, "ReactorBDFAdaptive")
        assert abs(work["nsteps"] - run.stats["nsteps"]) <= 0.05 * run.stats["nsteps"]


@pytest.mark.parametrize("mech,ident,dt", [("drm19", "ReactorRK64", 1e-7), ("LiDryer", "ReactorRK64", 1e-7),
                                           ("dodecane_lu", "ReactorRK64", 1e-8),
                                           ("LuEthylene_qss", "ReactorRK64", 1e-8), ("drm19", "ReactorBDF", 1e-6)])
def test_fixed_step_counts(models, oracles, mech, ident, dt):
    torch = _torch()
    m, st, ysrc, esrc = _cells(models, mech)

    def run(s):
        z = np.zeros((s.ncells, m.n_species))
        _, y, _, R = _run_1d(torch, mech, ident, s, z, np.zeros(s.ncells), dt)
        run.steps = R.cell_steps(s.ncells)
        return y

    y = run(st)
    _, oy, _, fc = _oracle_1d(oracles[mech], "rk64" if ident == "ReactorRK64" else "bdf", st, ysrc, esrc, dt)
    assert (run.steps == fc).all()
    _compare_y(m.n_species + 1, y, oy)
    _prefixes(run, st, m.n_species + 1, y, COUNTS)


def test_rk64_on_both_sides_of_the_lane_kernel(models):
    """The call that still runs on groups and the next larger one (one cell per lane)."""
    torch = _torch()
    ncu = torch.cuda.get_device_properties(0).multi_processor_count
    m, st, _, _ = _cells(models, "drm19", 64)
    out = []
    for n in (96 * ncu, 96 * ncu + 1):
        s = W.subsample(st, np.arange(n) % st.ncells)
        _, y, _, R = _run_1d(torch, "drm19", "ReactorRK64", s, np.zeros((n, m.n_species)), np.zeros(n), 1e-7)
        y = y.reshape(n, -1)
        assert (y == y[np.arange(n) % st.ncells]).all()  # every copy of a cell alike
        out.append((y[:st.ncells], R.cell_steps(n)[:st.ncells]))
    assert (out[0][1] == out[1][1]).all()
    _compare_y(m.n_species + 1, out[0][0], out[1][0])


@pytest.mark.parametrize("mech", ["drm19", "LiDryer"])
def test_adaptive_on_both_sides_of_the_narrow_group(models, oracles, mech):
    """The largest call with a lane per equation and the next, with half as many
    lanes: both meet the criterion, and every copy of a cell is alike in each."""
    torch = _torch()
    ncu = torch.cuda.get_device_properties(0).multi_processor_count
    m, st, ysrc, esrc = _cells(models, mech, 64)
    tol = dict(rtol=1e-12, atol=1e-18) if mech == "LiDryer" else dict(rtol=1e-10, atol=1e-16)
    p = oracle.adapt_params(rtol=1e-13, atol=1e-20)
    _, oy, _, _ = _oracle_1d(oracles[mech], "adaptive", st, ysrc, esrc, 1e-6, params=p)
    for n in (256 * ncu - 1, 256 * ncu):
        s = W.subsample(st, np.arange(n) % st.ncells)
        _, y, _, R = _run_1d(torch, mech, "ReactorBDFAdaptiveMixed", s, np.zeros((n, m.n_species)), np.zeros(n), 1e-6,
                             **tol)
        assert R.stats()["nfailed"] == 0
        y = y.reshape(n, -1)
        assert (y == y[np.arange(n) % st.ncells]).all()
        _compare_y(m.n_species + 1, y[:st.ncells].reshape(-1), oy)


def test_statistics_and_cost_order_of_a_large_call(models):
    """More cells than the bookkeeping kernels have threads, an odd number of
    them: the statistics are those of the per-cell counts, and the second call,
    which visits the cells in the order of the first one's costs, integrates each
    of them once (the same state, from the same start)."""
    torch = _torch()
    from pelephysics_amd.reactor import ReactorBase
    m, st, _, _ = _cells(models, "LiDryer", 4096)
    n = 1024 * 256 + 4099
    s = W.subsample(st, np.arange(n) % st.ncells)
    R = ReactorBase.create("ReactorBDFAdaptiveMixed")
    R.init(2, n, mechanism="LiDryer", rtol=1e-6, atol=1e-10)
    dev = torch.device("cuda:0")
    y0, x0 = torch.from_numpy(s.y_1d()).to(dev), torch.from_numpy(s.rE.copy()).to(dev)
    ys, xs = torch.zeros(n * m.n_species, dtype=torch.float64, device=dev), torch.zeros(n, dtype=torch.float64, device=dev)
    y, x = y0.clone(), x0.clone()
    R.react_1d(y, ys, x, xs, 2e-6)
    first, steps = y.clone(), R.cell_steps(n)
    y.copy_(y0)
    x.copy_(x0)
    R.react_1d(y, ys, x, xs, 2e-6)
    assert torch.equal(y, first) and np.array_equal(R.cell_steps(n), steps)
    t = R.stats()
    assert (t["nsteps"], t["max_steps_cell"], t["min_steps_cell"]) == (steps.sum(), steps.max(), steps.min())
    assert t["ncells"] == n and t["nfailed"] == 0 and steps.max() > steps.min() > 0


@pytest.mark.parametrize("mech", ["drm19", "LiDryer", "dodecane_lu"])
def test_production_rate_counts(models, oracles, mech):
    """64 cells per block: the last block's remainder.  The tolerance is the mechanism tests'."""
    import torch
    from pelephysics_amd.reactor import ReactorBase
    m, st, _, _ = _cells(models, mech, 130)
    y = st.y_1d().reshape(st.ncells, -1)
    sc = torch.from_numpy(y[:, :-1] * np.array([s.imw for s in m.species]) * 1e6).cuda().contiguous()
    T = torch.from_numpy(y[:, -1].copy()).cuda()
    R = ReactorBase.create("ReactorBDF")
    R.init(2, 1, mechanism=mech)
    w = R.production_rate(sc, T)
    for c in (0, 63, 64, 129):
        wo = oracles[mech].wdot(sc[c].cpu().numpy(), float(T[c]))
        assert np.abs(w[c].cpu().numpy() - wo).max() <= 1e-10 * np.abs(wo).max(), c
    for n in (1, 63, 64, 65, 129):
        assert torch.equal(R.production_rate(sc[:n].contiguous(), T[:n].contiguous()), w[:n]), n
    # calls that fill the chip pass their arrays through LDS: every copy of a cell
    # alike, and the rates above to the same tolerance
    for n in (65535, 65536, 65537):
        i = torch.arange(n, device="cuda") % 130
        wn = R.production_rate(sc[i].contiguous(), T[i].contiguous())
        assert torch.equal(wn, wn[:130][i]), n
        assert ((wn[:130] - w).abs().amax(1) <= 1e-10 * w.abs().amax(1)).all(), n
