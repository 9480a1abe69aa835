"""The orbit integrator by teams of waves (small batches in the Milky Way
fields) against the integrator with one wave to 64 orbits (large batches).

Both sum every step's stages in the same order, so the results are the same
bits: positions, velocities, statuses, step counts and dense records."""

import ctypes

import numpy as np
import pytest

import galax_amd.dynamics as gd
import galax_amd.potential as gp
from galax_amd import _lib

pytestmark = pytest.mark.gpu

PID = gd.PIDController(rtol=1e-8, atol=1e-10)
# rows of a batch that a 64th of the device holds in one-wave form only
LARGE = 2304


def _with_parts(parts, f):
    prev = ctypes.c_int32()
    _lib.check(_lib.lib().gx_set_launch_fraction(parts, ctypes.byref(prev)), "gx_set_launch_fraction")
    try:
        return f()
    finally:
        _lib.check(_lib.lib().gx_set_launch_fraction(prev.value, None), "gx_set_launch_fraction")


def _orbits(n):
    rng = np.random.default_rng(n)
    r, phi = rng.uniform(0.05, 30.0, n), rng.uniform(0.0, 2 * np.pi, n)
    v = 0.2 * rng.normal(size=(n, 3))
    w = np.stack([r * np.cos(phi), r * np.sin(phi), 0.3 * rng.normal(size=n), *v.T], 1)
    t1 = rng.uniform(-150.0, 400.0, n)
    t1[2::17] = 0.0  # nothing to integrate
    w[5::31, 1] = np.nan
    return w, t1


def _pieces():
    solver = gd.OrbitSolver(stepsize_controller=PID, max_steps=None)
    w = np.array([[25.0, 0.0, 0.0, 0.0, 0.113, 0.01]])
    prog = gd.integrate_orbits(gp.MilkyWayPotential(), w, -150.0, 250.0, T=2, solver=solver, dense=True)
    track = gp.TimeDependentTranslationParameter.from_dense(prog.dense)
    return gp.CompositePotential(host=gp.MilkyWayPotential(),
                                 progenitor=gp.TranslatedPotential(gp.PlummerPotential(m_tot=1e9, r_s=0.3), track))


def _both(pot, n, solver, own_spans, T, **kw):
    """(team, one wave) results of the first n of LARGE orbits."""
    w, t1 = _orbits(LARGE)
    ts = None
    if T > 1:  # save times at both ends, repeated, and beyond the end
        ts = np.sort(np.random.default_rng(T).uniform(0.0, 1.0, (LARGE, T)), 1)
        ts[:, 0], ts[:, -1] = 0.0, 1.0
        ts[::3, 1] = ts[::3, 2] if T > 3 else 0.0
        ts[::7, -1] = 1.1
        ts = ts * (t1[:, None] if own_spans else 300.0)

    def run(m):
        return gd.integrate_orbits(pot, w[:m], 0.0 if not own_spans else np.zeros(m), t1[:m] if own_spans else 300.0,
                                   ts=None if ts is None else ts[:m], solver=solver, **kw)

    team = run(n)
    one = _with_parts(64, lambda: run(LARGE))
    return team, one


def _same(team, one, n):
    for k in ("out", "status", "nsteps", "naccept"):
        np.testing.assert_array_equal(getattr(team, k).cpu().numpy(), getattr(one, k).cpu().numpy()[:n])


@pytest.mark.parametrize("field", ["milky way", "pieces"])
@pytest.mark.parametrize("n, own_spans, T", [(1, True, 1), (63, True, 9), (64, False, 40), (65, False, 2),
                                             (2000, True, 5)])
@pytest.mark.parametrize("control", ["pid", "limits", "fixed"])
def test_teams_give_the_bits_of_single_waves(field, n, own_spans, T, control):
    pot = gp.MilkyWayPotential() if field == "milky way" else _pieces()
    kw = {}
    if control == "pid":
        solver = gd.OrbitSolver(stepsize_controller=PID, max_steps=None)
    elif control == "limits":
        pid = gd.PIDController(rtol=1e-8, atol=1e-10, pcoeff=0.3, icoeff=0.4, dtmin=0.5, force_dtmin=n % 2 == 0,
                               dtmax=9.0)
        solver = gd.OrbitSolver(stepsize_controller=pid, max_steps=40)
    else:
        solver = gd.OrbitSolver(stepsize_controller=gd.ConstantStepSize(), max_steps=None)
        kw = {"dt0": 2.3}
    _same(*_both(pot, n, solver, own_spans, T, **kw), n)


@pytest.mark.parametrize("n", [1, 64, 130])
@pytest.mark.parametrize("cap", [7, 400])
def test_team_records_are_those_of_single_waves(n, cap):
    """Dense records, also where the capacity has to be raised."""
    solver = gd.OrbitSolver(stepsize_controller=PID, max_steps=None)
    team, one = _both(gp.MilkyWayPotential(), n, solver, True, 3, dense=cap)
    _same(team, one, n)
    a, b = team.dense.nrec.cpu().numpy(), one.dense.nrec.cpu().numpy()[:n]
    np.testing.assert_array_equal(a, b)
    x, y = team.dense.rec.cpu().numpy(), one.dense.rec.cpu().numpy()
    x, y = x.reshape(n, -1, x.shape[-1] if x.ndim > 2 else 50), y.reshape(LARGE, -1, y.shape[-1] if y.ndim > 2 else 50)
    for i in range(n):
        np.testing.assert_array_equal(x[i, :a[i]], y[i, :a[i]])
