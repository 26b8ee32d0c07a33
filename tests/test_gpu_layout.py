"""Copies between a caller's packed arrays and the solver's pitched planes
(csrc/layout2d.hip): what goes up comes down with the same bytes, on rows that
fill their pitch (multiples of 32), just miss it and just pass it, with the
energy given and formed on the device; the BC -1 ghost tables; the flux batch's
rows that its fast solver leaves to the IEEE one, at the edges of its blocks."""
import numpy as np
import pytest

import cases
from _libs import make_config
from conftest import parity

pytestmark = pytest.mark.gpu
GAMMA, EPS = 1.4, 1e-9
SIZES = [(1, 1), (3, 32), (32, 31), (5, 33), (64, 64), (1, 50), (50, 1), (257, 190)]


@pytest.fixture(scope="module")
def hg():
    import hydrogrp
    hydrogrp.lib()
    return hydrogrp


def _energy(s):
    t = 0.5 * s["u"] * s["u"] + s["p"] / (GAMMA - 1.0) / s["rho"]
    return t + 0.5 * s["v"] * s["v"]


@pytest.mark.parametrize("m,n", SIZES)
def test_state_and_fraction_round_trip(hg, m, n):
    s = cases.smooth_random(m, n, m + n)
    c = hg.Solver2D(m, n, make_config(t_all=0.1, h_x=1 / m, h_y=1 / n, bc_x=-4, bc_y=-4, split=1))
    try:
        for e in (None, _energy(s) + 0.25):
            c.upload(s["rho"], s["u"], s["v"], s["p"], e)
            for _ in range(2):                         # a download leaves the state alone
                got = np.asarray(c.download()).reshape(5, m, n)
                for f, w in enumerate((s["rho"], s["u"], s["v"], s["p"], _energy(s) if e is None else e)):
                    assert np.array_equal(got[f], w.reshape(m, n)), (f, e is None)
        a = np.random.default_rng(m).random((m, n))
        c.set_fluids(1.67, a)
        assert np.array_equal(np.asarray(c.download_fraction()).reshape(m, n), a)
        assert np.array_equal(np.asarray(c.download()).reshape(5, m, n)[:4], got[:4])
    finally:
        c.close()


def test_batch_round_trip(hg):
    states = [cases.smooth_random(m, n, m + n) for m, n in SIZES]
    b = hg.Batch2D([(m, n, 1.0 / m, 1.0 / n) for m, n in SIZES],
                   make_config(t_all=0.1, bc_x=-4, bc_y=-4, split=1))
    try:
        b.upload(states)
        for got, s, (m, n) in zip(b.download(), states, SIZES):
            for f, w in enumerate((s["rho"], s["u"], s["v"], s["p"], _energy(s))):
                assert np.array_equal(got[f], w.reshape(m, n)), (m, n, f)
    finally:
        b.close()


@pytest.mark.parametrize("m,n", [(6, 32), (32, 6), (7, 33)])
def test_initial_state_ghosts(hg, oracle, m, n):
    init = cases.smooth_random(m, n, 3)
    cfg = make_config(t_all=0.04, h_x=1 / m, h_y=1 / n, bc_x=-1, bc_y=-1, split=1)
    fo, npo, tpo, co, _ = oracle.split2d(m, n, init, cfg)
    fg, npg, tpg, cg, _ = hg.run_split2d(m, n, init, cfg)
    assert (co[5], npo, tpo[npo - 1]) == (cg[5], npg, tpg[npg - 1])
    assert parity(fg[:, npg - 1], fo[:, npo - 1]).max() <= 1e-10      # glibc's pow against the device's


@pytest.mark.parametrize("direction,nxy", [(0, (1.0, 0.0)), (1, (0.0, 1.0))])
@pytest.mark.parametrize("count", [1, 127, 128, 129])
def test_flux_batch_outside_the_fast_range(hg, oracle_devpow, count, direction, nxy):
    """Every other row has a pressure, velocity or gamma that the fast solver
    does not take; all rows against the oracle with the device's pow, each to
    1e-13 of its largest entry (the arithmetic is the same: rounding only)."""
    L, R = (np.array(A) for A in cases.interface_pairs(count, 31))
    rng = np.random.default_rng(count)
    for A in (L, R):
        A[:, 11:15] = 0.0 if direction == 0 else -0.0
    for k in range(0, count, 2):
        A = (L, R)[rng.integers(2)]
        kind = rng.integers(4)
        if kind == 0:
            A[k, 6] = np.nan
        elif kind == 1:
            A[k, 3], A[k, 6] = 1e-40, 1e-40
        elif kind == 2:
            L[k, 4:6] = R[k, 4:6] = 1e35
        else:
            L[k, 0] = R[k, 0] = 1.0 + 2.0 ** -22
    got = hg.flux_batch(L, R, 1e-3, EPS, direction)
    want = np.array([[rc, *o] for rc, o in (oracle_devpow.flux2d(L[k], R[k], 1e-3, EPS, *nxy) for k in range(count))])
    assert np.array_equal(got[:, 0] != 0, want[:, 0] != 0)
    ok = want[:, 0] == 0
    scale = np.abs(want[ok, 1:]).max(axis=1, keepdims=True)
    fin = np.isfinite(scale[:, 0])
    assert np.array_equal(np.isfinite(got[ok, 1:]), np.isfinite(want[ok, 1:]))
    assert np.all(np.abs(got[ok, 1:] - want[ok, 1:])[fin] <= 1e-13 * scale[fin])
