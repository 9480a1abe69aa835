"""What the adjoint asks of memory."""

import pytest

from galax_amd import _lib


@pytest.mark.parametrize("K", [1, 8, 64, 500])
def test_a_workspace_serves_every_smaller_batch(K):
    """A program sizes its workspace once, for its largest batch and longest
    span: no smaller one may need more."""
    if not _lib.LIB_PATH.exists():
        pytest.skip("libgalaxhip.so not built")
    size = _lib.lib().gx_adjoint_workspace_bytes
    ns = [0, 1, 127, 1000, 24_028, 25_001, 76_000, 132_701, 160_037, 200_000, 5_000_000]
    steps = [0, 1, 49, 490, 1000, 3000, 10_000, 400_000]
    table = [[int(size(n, m, K)) for m in steps] for n in ns]
    for i, row in enumerate(table):
        assert row == sorted(row)
        if i:
            assert all(a <= b for a, b in zip(table[i - 1], row))


@pytest.mark.parametrize("n, steps, K", [(0, 10, 64), (1, 1, 64), (1000, 490, 64), (160_037, 490, 64), (77, 3000, 8)])
def test_the_caller_says_how_much_memory_is_taken(n, steps, K):
    """A limit is kept where the checkpoints fit in it, and what is taken for
    it is what the same limit again would take."""
    if not _lib.LIB_PATH.exists():
        pytest.skip("libgalaxhip.so not built")
    within = _lib.lib().gx_adjoint_workspace_within
    least = int(within(n, steps, K, 0))
    assert least == 56 * n * (steps // K + 2 + K) + 256 or n == 0
    every = 56 * n * (steps // K + 2) * K + 256
    for limit in (0, least, every - 1, every, every + 1, 1 << 40):
        got = int(within(n, steps, K, limit))
        assert got == (every if limit >= every or n == 0 else least)
        assert int(within(n, steps, K, got)) == got


def _problem(n):
    import numpy as np

    import galax_amd.potential as gp
    from galax_amd import workloads

    rng = np.random.default_rng(n)
    t0 = -rng.uniform(1.0, 300.0, n)
    ts = np.stack([0.37 * t0, np.zeros(n)], 1)
    return gp.MilkyWayPotential(), workloads.disk_ics(n, 3), t0, ts, rng.normal(size=(n, 2, 6))


@pytest.mark.gpu
@pytest.mark.parametrize("method", ["dopri8", "dopri5"])
def test_gradients_do_not_depend_on_the_memory_given(method, monkeypatch):
    """Every step's state kept, checkpoints on request, and checkpoints where
    the states do not fit on the device: the same bits."""
    import numpy as np
    import torch

    import galax_amd.dynamics as gd
    from galax_amd import _abi
    from galax_amd.adjoint import adjoint_orbits

    n, K = 300, 16
    pot, w0, t0, ts, cot = _problem(n)
    meth = gd.Dopri8() if method == "dopri8" else gd.Dopri5()
    empty, sizes, refuse = torch.empty, [], []

    def spy(shape, *a, **kw):
        if isinstance(shape, int):
            sizes.append(8 * shape)
            if refuse and len(sizes) == 1:
                raise torch.cuda.OutOfMemoryError("no room")
        return empty(shape, *a, **kw)

    monkeypatch.setattr(torch, "empty", spy)

    def run(**kw):
        del sizes[:]
        wb, raw, st = adjoint_orbits(pot, w0, t0, 0.0, torch.as_tensor(cot), dt0=1.0, ts=ts, method=meth, ntheta=12,
                                     max_steps=302, K=K, **kw)
        assert int(st.abs().sum()) == 0
        return wb.cpu().numpy(), raw.cpu().numpy(), list(sizes)

    within = _lib.lib().gx_adjoint_workspace_within
    least, every = (int(within(n, 302, K, b)) for b in (0, _abi.GX_ADJOINT_STATES_BYTES))
    assert least < every
    first = run()
    assert first[2] == [every]
    small = run(workspace_bytes=0)
    assert small[2] == [least]
    refuse.append(True)
    fallback = run()
    assert fallback[2] == [every, least]
    for other in (small, fallback):
        for a, b in zip(first[:2], other[:2]):
            np.testing.assert_array_equal(a, b)


@pytest.mark.gpu
def test_too_small_a_workspace_is_refused():
    import ctypes

    import torch

    import galax_amd.dynamics as gd
    from galax_amd import _abi

    pot, w0, t0, _, cot = _problem(64)
    d = [torch.as_tensor(x, device="cuda").contiguous() for x in (w0, t0, 0 * t0, cot[:, :1])]
    cfg = gd.OrbitSolver(gd.Dopri8(), stepsize_controller=gd.ConstantStepSize(), max_steps=None).cfg(dt0=1.0)
    lib = _lib.lib()
    least = int(lib.gx_adjoint_workspace_within(64, 302, 16, 0))
    ws, wb = torch.empty(least, dtype=torch.uint8, device="cuda"), torch.empty((64, 6), dtype=torch.float64, device="cuda")

    def call(nbytes):
        return lib.gx_adjoint_within(pot._handle(), ctypes.addressof(cfg), *(_lib.ptr(x) for x in d[:3]), 1, None, 1,
                                     _abi.GX_TS_FINAL, 64, _lib.ptr(d[3]), _lib.ptr(wb), None, 0, 302, 16, None,
                                     _lib.ptr(ws), nbytes, _lib.stream_ptr())

    for nbytes in (-1, 0, 255, least - 1):
        assert call(nbytes) == _abi.GX_EINVAL
    assert call(least) == _abi.GX_OK
    torch.cuda.synchronize()
