"""Which form of the integrator takes a batch does not show in its results:
batches beyond what the device holds in teams, where the device chooses by
the batch's spans, and the one-wave form's queue (fixed first tickets, tickets
taken several at a time, lanes that take many orbits), against the same orbits
by teams, row by row and bit by bit.

A 64th of the device holds 512 orbits in teams and 2,048 in the one-wave form;
all of it takes every batch here by teams."""

import ctypes

import numpy as np
import pytest

import galax_amd.dynamics as gd
import galax_amd.potential as gp
from galax_amd import _lib
from test_orbit_teams import PID, _orbits, _pieces, _with_parts

pytestmark = pytest.mark.gpu


def _queue(head, chunk, f):
    lib, h, c = _lib.lib(), ctypes.c_int64(), ctypes.c_int32()
    _lib.check(lib.gx_set_queue_policy(head, chunk, ctypes.byref(h), ctypes.byref(c)), "gx_set_queue_policy")
    try:
        return f()
    finally:
        _lib.check(lib.gx_set_queue_policy(h.value, c.value, None, None), "gx_set_queue_policy")


def _same(a, b):
    for k in ("out", "status", "nsteps", "naccept"):
        np.testing.assert_array_equal(getattr(a, k).cpu().numpy(), getattr(b, k).cpu().numpy())
    if a.dense is not None:
        n, m = a.dense.nrec.cpu().numpy(), b.dense.nrec.cpu().numpy()
        np.testing.assert_array_equal(n, m)
        x, y = a.dense.rec.cpu().numpy(), b.dense.rec.cpu().numpy()
        used = np.arange(min(x.shape[1], y.shape[1]))[None, :] < n[:, None]
        np.testing.assert_array_equal(x[:, :used.shape[1]][used], y[:, :used.shape[1]][used])


@pytest.mark.parametrize("field", ["milky way", "pieces"])
@pytest.mark.parametrize("n", [513, 1025, 2048, 2049])
@pytest.mark.parametrize("spans", ["own", "equal", "none"])
@pytest.mark.parametrize("T, ordered", [(1, True), (3, False), (300, True)])
def test_the_device_chooses_between_equal_results(field, n, spans, T, ordered):
    pot = gp.MilkyWayPotential() if field == "milky way" else _pieces()
    solver = gd.OrbitSolver(stepsize_controller=PID, max_steps=None)
    w, t1 = _orbits(n)
    t1 = {"own": t1, "equal": np.full(n, 120.0), "none": np.zeros(n)}[spans]
    order = np.argsort(-np.abs(t1), kind="stable") if ordered else None

    def run():
        return gd.integrate_orbits(pot, w, np.zeros(n), t1, T=T if T > 1 else None, solver=solver, order=order)

    _same(_with_parts(64, run), run())


@pytest.mark.parametrize("control, dense", [("pid", False), ("pid", True), ("fixed", False)])
@pytest.mark.parametrize("field", ["milky way", "pieces"])
@pytest.mark.parametrize("head, chunk", [(0, 1), (64, 1), (512, 5), (1_000_000, 3)])
def test_one_waves_take_orbit_after_orbit(field, control, dense, head, chunk):
    if dense and field == "pieces":
        pytest.skip("no dense form of its own")
    pot = gp.MilkyWayPotential() if field == "milky way" else _pieces()
    kw = {"dense": 400} if dense else {}
    if control == "pid":
        solver = gd.OrbitSolver(stepsize_controller=PID, max_steps=None)
    else:
        solver, kw = gd.OrbitSolver(stepsize_controller=gd.ConstantStepSize(), max_steps=None), {"dt0": 2.3}
    n = 6001
    w, t1 = _orbits(n)
    order = np.random.default_rng(head).permutation(n)

    def run():
        return gd.integrate_orbits(pot, w, np.zeros(n), t1, T=4, solver=solver, order=order, **kw)

    one = _with_parts(64, lambda: _queue(head, chunk, run))
    _same(one, run())
