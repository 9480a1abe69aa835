"""The kernels whose workgroups exchange values, at the sizes that fill the
device, against the oracle at the bounds of their smaller tests: a shared step
sequence of up to 512 workgroups (256 meet in one round of loads) with a
ragged last one, and N-body systems of up to 256 workgroups of 16 bodies."""

import numpy as np
import pytest

import galax_amd.dynamics as gd
import galax_amd.potential as gp
import oracle
from galax_amd.units import G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [16_384, 16_449, 32_768])
@pytest.mark.parametrize("control", ["pid", "fixed"])
def test_shared_steps_of_a_full_device(n, control):
    rng = np.random.default_rng(n)
    r, phi = rng.uniform(4.0, 20.0, n), rng.uniform(0.0, 2 * np.pi, n)
    w0 = np.stack([r * np.cos(phi), r * np.sin(phi), 0.3 * rng.normal(size=n), -0.2 * np.sin(phi), 0.2 * np.cos(phi),
                   0.02 * rng.normal(size=n)], 1)
    kw = {} if control == "pid" else {"dt0": 2.3}
    ctl = gd.PIDController(rtol=1e-8, atol=1e-10) if control == "pid" else gd.ConstantStepSize()
    solver = gd.OrbitSolver(stepsize_controller=ctl, max_steps=None)
    ts = np.array([0.0, 3.7, 20.0])
    print(f"[case] shared {control} n={n}", flush=True)
    res = gd.integrate_orbits(gp.MilkyWayPotential(), w0, 0.0, 20.0, ts=ts, solver=solver, shared=True, **kw)
    ref, st, ns, na = oracle.integrate(gp.MilkyWayPotential(), solver, w0, 0.0, 20.0, ts=ts, shared=True, **kw)
    for got, want in ((res.status, st), (res.nsteps, ns), (res.naccept, na)):
        np.testing.assert_array_equal(got.cpu().numpy(), want)
    d = res.out.cpu().numpy() - ref
    for s in (slice(0, 3), slice(3, 6)):
        assert np.linalg.norm(d[..., s]) <= 1e-10 * np.linalg.norm(ref[..., s])


@pytest.mark.parametrize("n", [2048, 2049, 4096])
def test_bodies_on_every_workgroup(n):
    rng = np.random.default_rng(n)
    w0 = np.concatenate([[8.0, 0.0, 0.2] + 0.05 * rng.normal(size=(n, 3)), [0.0, 0.23, 0.0] + 0.002 * rng.normal(size=(n, 3))], 1)
    m = rng.uniform(0.01, 1.0, n) * (4e6 / n)
    mw = gp.MilkyWayPotential()
    solver = gd.OrbitSolver(gd.Dopri8(), stepsize_controller=gd.ConstantStepSize(), max_steps=None)
    ts = np.array([0.33, 1.0])
    print(f"[case] nbody n={n}", flush=True)
    soln = gd.solve_nbody(gd.NBodyField(masses=m, eps=0.05, external_potential=mw), (w0[:, :3], w0[:, 3:]), 0.0, 1.0,
                          saveat=ts, solver=solver, dt0=0.5)
    ref, st, ns, _ = oracle.nbody_integrate(mw, G * m, 0.05, solver, w0, 0.0, 1.0, ts=ts, dt0=0.5)
    assert soln.status == 0 and st == 0 and soln.nsteps == ns == 2
    got = np.concatenate([np.transpose(soln.ys[0], (1, 0, 2)), np.transpose(soln.ys[1], (1, 0, 2))], -1)
    rel = np.abs(got - ref) / np.abs(ref).max(axis=(1, 2), keepdims=True)
    assert rel.max() < 1e-12
