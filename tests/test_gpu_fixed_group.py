"""The parameters of the fixed-step ReactorBDF on drm19, whose cells run on
groups of 16 lanes (group_fixed.h), at any number of cells: substeps with the
BDF3 history and its TRPZ ramp, every scheme with several Newton iterations,
preconditioners, stale restarts, failing cells, both energy forms, sources, and
hot burnt cells, whose rates cancel to the last bits.

Criterion and rounding ensemble of test_gpu_parity; the banded fractions are the
ensemble's own, measured on the CPU."""
import numpy as np
import pytest

import oracle
from pelephysics_amd import workloads as W
from test_gpu_parity import _torch, _compare_y, _close, _hull_1d, _oracle_1d, _run_1d, _sources, _state

pytestmark = pytest.mark.gpu


def _check(models, oracles, st, ysrc, esrc, dt, reactor_type=2, max_banded=0.0, **p):
    torch = _torch()
    m = models["drm19"]
    ret, y, rX, R = _run_1d(torch, "drm19", "ReactorBDF", st, ysrc, esrc, dt, reactor_type,
                            **{f"bdf_{k}": v for k, v in p.items()})
    params = oracle.bdf_params(m.n_species, **p)
    oret, oy, orX, fc = _oracle_1d(oracles["drm19"], "bdf", st, ysrc, esrc, dt, reactor_type, params)
    assert ret == oret == p.get("nsubsteps", 1)
    assert (R.cell_steps(st.ncells) == fc).all()
    _compare_y(m.n_species + 1, y, oy, _hull_1d(models, "drm19", st, ysrc, esrc, dt, reactor_type, params),
               max_banded)
    _close("rX", rX, orX)
    return y


@pytest.mark.parametrize("precond", [1, 2])
def test_substeps_and_sources(models, oracles, precond):
    m, st = _state(models, "drm19", 100, seed=11)
    ysrc, esrc = _sources(st, m, 3, 10.0)
    _check(models, oracles, st, ysrc, esrc, 1e-6, nsubsteps=40, gmres_precond=precond)


def test_failing_cells(models, oracles):
    """Without a preconditioner no cell converges: each reports it and keeps its state."""
    torch = _torch()
    from pelephysics_amd.reactor import ReactorBase, ReactorError
    m, st = _state(models, "drm19", 100, seed=11)
    ysrc, esrc = _sources(st, m, 3, 10.0)
    p = oracle.bdf_params(m.n_species, nsubsteps=40, gmres_precond=0)
    oret, _, _, fc = _oracle_1d(oracles["drm19"], "bdf", st, ysrc, esrc, 1e-6, params=p)
    assert oret < 0 and (fc < 0).all()
    R = ReactorBase.create("ReactorBDF")
    R.init(2, st.ncells, mechanism="drm19", bdf_nsubsteps=40, bdf_gmres_precond=0)
    y = torch.from_numpy(st.y_1d()).cuda()
    with pytest.raises(ReactorError) as e:
        R.react_1d(y, torch.from_numpy(ysrc.reshape(-1).copy()).cuda(), torch.from_numpy(st.rE.copy()).cuda(),
                   torch.from_numpy(esrc).cuda(), 1e-6)
    assert e.value.code == -4 and f"{st.ncells} cell(s) failed" in str(e.value)
    assert (R.cell_steps(st.ncells) == -1).all() and np.array_equal(y.cpu().numpy(), st.y_1d())


def test_stale_restarts(models, oracles):
    """A tolerance that no cycle reaches: three restarts give three times one
    restart's increment (test_gpu_parity.py, test_bdf_gmres_stale_restarts)."""
    m, st = _state(models, "drm19", 64, seed=5)
    z = np.zeros((st.ncells, m.n_species))
    inc = {}
    for restarts in (1, 3):
        y = _check(models, oracles, st, z, np.zeros(st.ncells), 1e-7, scheme=0, gmres_tol=1e-30,
                   gmres_restarts=restarts)
        inc[restarts] = (y - st.y_1d()).reshape(st.ncells, -1)
    err = np.abs(inc[3] - 3 * inc[1]).max(1) / np.abs(inc[1]).max(1)
    assert err.max() < 1e-5, err.max()  # the rounding of three Krylov cycles that stop at 1e-30


@pytest.mark.parametrize("scheme,iters", [(0, 1), (1, 3), (2, 2), (3, 2)])
def test_schemes_e_reactor(models, oracles, scheme, iters):
    m, st = _state(models, "drm19", 64, seed=5)
    st.rE[:] = st.rE - st.p
    z = np.zeros((st.ncells, m.n_species))
    _check(models, oracles, st, z, np.zeros(st.ncells), 2e-6, reactor_type=1, nsubsteps=10, scheme=scheme,
           nonlinear_iters=iters)


# banded: 51 and 57 of 66 cells in one 1e-6 s step, 21 and 17 at 1e-7 s, none in 20 substeps
@pytest.mark.parametrize("reactor_type", [1, 2])
@pytest.mark.parametrize("dt,nsub,max_banded", [(1e-6, 1, 0.9), (1e-7, 1, 0.35), (1e-6, 20, 0.0)])
def test_hot_cells_with_sources(models, oracles, reactor_type, dt, nsub, max_banded):
    m = models["drm19"]
    g = W.drm19_grf(m, 64)
    st = W.subsample(g, np.argsort(g.T)[-64 ** 3 // 50:][::80])  # 2162 to 2200 K
    if reactor_type == 1:
        st.rE[:] = st.rE - st.p
    ysrc, esrc = _sources(st, m, 4, 10.0)
    _check(models, oracles, st, ysrc, esrc, dt, reactor_type, max_banded, nsubsteps=nsub)
