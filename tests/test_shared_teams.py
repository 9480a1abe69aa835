"""A batch as one system by teams of waves (the Milky Way, up to 32,768
orbits), at the edges of a team's 64 orbits and over several workgroups,
against the oracle's shared step sequence.

Both take the same decisions; their step sizes differ by the rounding of the
batch's error norm, a few units in the last place a step, which some hundred
steps and the orbits' divergence over 300 Myr leave below 1e-10."""

import numpy as np
import pytest

import galax_amd.dynamics as gd
import galax_amd.potential as gp
import oracle

pytestmark = pytest.mark.gpu


def _batch(n):
    rng = np.random.default_rng(n)
    r, phi = rng.uniform(4.0, 20.0, n), rng.uniform(0.0, 2 * np.pi, n)
    return np.stack([r * np.cos(phi), r * np.sin(phi), 0.3 * rng.normal(size=n), -0.2 * np.sin(phi),
                     0.2 * np.cos(phi), 0.02 * rng.normal(size=n)], 1)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 640])
@pytest.mark.parametrize("control", ["pid", "stopped", "fixed"])
@pytest.mark.parametrize("t1", [300.0, -120.0])
def test_shared_teams_against_the_oracle(n, control, t1):
    kw = {}
    if control == "fixed":
        solver = gd.OrbitSolver(stepsize_controller=gd.ConstantStepSize(), max_steps=None)
        kw = {"dt0": 2.3}
    else:
        solver = gd.OrbitSolver(stepsize_controller=gd.PIDController(rtol=1e-8, atol=1e-10),
                                max_steps=12 if control == "stopped" else None)
    w0 = _batch(n)
    # at the start twice, inside steps, several in one step, at the end
    ts = t1 * np.array([0.0, 0.0, 0.001, 0.0011, 0.2, 0.37, 0.9, 1.0])
    res = gd.integrate_orbits(gp.MilkyWayPotential(), w0, 0.0, t1, ts=ts, solver=solver, shared=True, **kw)
    ref, st, ns, na = oracle.integrate(gp.MilkyWayPotential(), solver, w0, 0.0, t1, ts=ts, shared=True, **kw)
    for got, want in ((res.status, st), (res.nsteps, ns), (res.naccept, na)):
        np.testing.assert_array_equal(got.cpu().numpy(), want)
    out = res.out.cpu().numpy()
    np.testing.assert_array_equal(np.isfinite(out), np.isfinite(ref))
    d, scale = np.nan_to_num(out - ref), np.nan_to_num(ref)
    for s in (slice(0, 3), slice(3, 6)):
        assert np.linalg.norm(d[..., s]) <= 1e-10 * np.linalg.norm(scale[..., s])


def test_shared_teams_stop_together_at_a_lost_orbit():
    w0 = _batch(200)
    w0[130, 1] = np.nan
    solver = gd.OrbitSolver(stepsize_controller=gd.PIDController(rtol=1e-8, atol=1e-10), max_steps=None)
    res = gd.integrate_orbits(gp.MilkyWayPotential(), w0, 0.0, 100.0, ts=[0.0, 50.0, 100.0], solver=solver,
                              dt0=1.0, shared=True)
    assert len(set(res.status.cpu().tolist())) == 1 and res.status[0] != 0
    assert np.all(np.isnan(res.out.cpu().numpy()[:, 1:]))
