"""Small self-gravitating systems on either side of the number of bodies that
changes the kernel, in a table field, against the oracle, at the bound of the
larger systems' fixed-step tests."""

import numpy as np
import pytest

import galax_amd.dynamics as gd
import galax_amd.potential as gp
import oracle
from galax_amd.units import G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 4, 5, 6, 8, 9, 12])
@pytest.mark.parametrize("method", [gd.Dopri8(), gd.Dopri5()], ids=["dopri8", "dopri5"])
def test_a_few_bodies_against_the_oracle(n, method):
    rng = np.random.default_rng(n)
    w0 = np.concatenate([[8.0, 0.0, 0.2] + 0.5 * rng.normal(size=(n, 3)), [0.0, 0.22, 0.0] + 0.01 * rng.normal(size=(n, 3))], 1)
    m = rng.uniform(1e4, 1e6, n)
    ext = gp.NFWPotential(m=5e11, r_s=12.0)
    solver = gd.OrbitSolver(method, stepsize_controller=gd.ConstantStepSize(), max_steps=None)
    ts = np.array([0.0, 3.3, 7.0, 20.0])
    print(f"[case] nbody few n={n}", flush=True)
    soln = gd.solve_nbody(gd.NBodyField(masses=m, eps=0.1, external_potential=ext), (w0[:, :3], w0[:, 3:]), 0.0, 20.0,
                          saveat=ts, solver=solver, dt0=0.5)
    ref, st, ns, na = oracle.nbody_integrate(ext, G * m, 0.1, solver, w0, 0.0, 20.0, ts=ts, dt0=0.5)
    assert (soln.status, soln.nsteps, soln.naccept) == (st, ns, na) and st == 0
    got = np.concatenate([np.transpose(soln.ys[0], (1, 0, 2)), np.transpose(soln.ys[1], (1, 0, 2))], -1)
    rel = np.abs(got - ref) / np.abs(ref).max(axis=(1, 2), keepdims=True)
    assert rel.max() < 1e-12
