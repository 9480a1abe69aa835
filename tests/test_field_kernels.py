"""The Milky Way's field kernels (alone and with a rotating group) at the edges
of a workgroup, on positions of every alignment, with a time for all points or
for each, far out and at the centre, against the oracle.

Bound: some 30 rounded operations a value, each within two units in the last
place (7e-15), times the halo's cancellation between 0.05 and 60 kpc (below
10): 1e-13 of a row's norm.  Within 1e-4 kpc of the centre the halo's share
cancels against itself, in the oracle as here, and only finiteness is left to
compare."""

import numpy as np
import pytest

import galax_amd.potential as gp
import oracle
from test_rotating_group import _group

pytestmark = pytest.mark.gpu
FIELDS = {"milky way": lambda: gp.MilkyWayPotential(), "group": lambda: _group("bpppppp")}


def _points(n):
    rng = np.random.default_rng(n)
    d = rng.normal(size=(n, 3))
    return d / np.linalg.norm(d, axis=1, keepdims=True) * 10.0 ** rng.uniform(-1.3, 1.78, (n, 1))


@pytest.mark.parametrize("field", list(FIELDS))
@pytest.mark.parametrize("n", [1, 63, 255, 256, 257, 1000])
@pytest.mark.parametrize("each", [False, True])
def test_field_kernels_against_the_oracle(field, n, each):
    import torch

    pot, x = FIELDS[field](), _points(n)
    t = np.linspace(-30.0, 70.0, n) if each else 11.0
    # a view one double into its storage: aligned to 8 bytes only
    q = torch.empty(3 * n + 1, dtype=torch.float64, device="cuda")[1:].view(n, 3)
    q.copy_(torch.from_numpy(x))
    tt = torch.from_numpy(t).cuda() if each else t
    for what in ("acceleration", "gradient") + (("hessian",) if field == "milky way" else ()):
        got = getattr(pot, what)(q, tt).cpu().numpy().reshape(n, -1)
        ref = oracle.evaluate(pot, what, x, t).reshape(n, -1)
        assert np.all(np.linalg.norm(got - ref, axis=1) <= 1e-13 * np.linalg.norm(ref, axis=1)), what


def test_fields_far_out_and_at_the_centre():
    pot = gp.MilkyWayPotential()
    r = np.array([1e-9, 0.9e-4, 1.1e-4, 1e-3, 1e9, 1e90])
    x = r[:, None] * np.array([0.6, -0.64, 0.48])
    got, ref = pot.hessian(x, 0.0).reshape(6, 9), oracle.evaluate(pot, "hessian", x, 0.0).reshape(6, 9)
    assert np.all(np.isfinite(got))
    far = r > 1e-4
    # at 1e-4 kpc the halo's difference holds 1e-5 of its terms' digits, and is 1e-4 of the Hessian
    assert np.all(np.linalg.norm(got - ref, axis=1)[far] <= 1e-11 * np.linalg.norm(ref, axis=1)[far])
    acc = pot.acceleration(np.array([[0.0, 0.0, 0.0], [np.nan, 1.0, 1.0], [1.0, np.inf, 0.0]]), 0.0)
    assert np.all(acc[0] == 0.0) and np.all(np.isnan(acc[1]))
