"""The steps' interface solver and the IEEE one on the device.

Runs that continue past the steps' fallback (redo_face, redo_face_tf,
redo_face_t, redo_iface: sides, ghosts and previous slopes built again from
memory), over enough steps that the previous slopes count.  Densities and
pressures in units of 2^-140 are out of the fast solver's range everywhere; so
are slopes over cells of 2^-150, and there every operation scales by powers of
two exactly, so that the run has the bits of one over cells of 1.  eps lies
below all that is compared with it (and the runs end by their number of steps).
And interface batches through both solvers, values next to powers of two among
them."""
import numpy as np
import pytest

import cases
from _libs import make_config

pytestmark = pytest.mark.gpu
UNIT, EPS, TOL = 2.0 ** -140, 1e-100, 1e-12
ENDS = [(-2, -7), (-24, -4), (-4, -2), (-7, -24), (-1, -1)]


@pytest.fixture(scope="module")
def hg():
    import hydrogrp
    hydrogrp.lib()
    return hydrogrp


def _scaled(s, unit):
    return {k: (a * unit if k in ("rho", "p") else a) for k, a in s.items()}


def _run(hg, m, n, s, cfg, converge, frac=None, gamma_b=1.67, g2d=False, form=None, sweeps=None):
    c = hg.Solver2D(m, n, cfg)
    try:
        c.set_newton(TOL, converge=converge)
        if g2d:
            c.set_interface_solver(True)
        if form is not None:
            c.set_unsplit_form(form)
        if sweeps is not None:
            c.set_sweeps(*sweeps)
        c.upload(s["rho"], s["u"], s["v"], s["p"])
        if frac is not None:
            c.set_fluids(gamma_b, frac)
        res = c.solve(np.array([0.0, cfg[1]]), 2)
        assert res.status == 0 and res.k >= 9
        return np.asarray(c.download()).reshape(5, m, n), None if frac is None else c.download_fraction()
    finally:
        c.close()


def _config(m, n, ends, h=1.0, **kw):
    return make_config(t_all=10.0, N=9, h_x=h / m, h_y=h / n, bc_x=ends[0], bc_y=ends[1], eps=EPS, **kw)


@pytest.mark.parametrize("ends", ENDS)
@pytest.mark.parametrize("converge", [False, True])
def test_split(hg, oracle_devpow, ends, converge):
    m, n = 17, 22
    s = _scaled(cases.smooth_random(m, n, 7), UNIT)
    cfg = _config(m, n, ends, split=1)
    want, k, _, _, st = oracle_devpow.split2d(m, n, s, cfg, newton_tol=TOL, converge=converge)
    assert st == 0
    for sweeps in ((3, 4), (0, 0), (4, 2)):
        assert np.array_equal(_run(hg, m, n, s, cfg, converge, sweeps=sweeps)[0], want[:, k - 1]), sweeps


@pytest.mark.parametrize("ends", ENDS[:4])
@pytest.mark.parametrize("converge", [False, True])
def test_two_fluids(hg, ends, converge):
    m, n = 17, 22
    s, frac = cases.smooth_random(m, n, 8), np.random.default_rng(1).random((m, n))
    frac[:5], frac[12:] = 0.0, 1.0
    (one, fa), (small, fb) = (_run(hg, m, n, s, _config(m, n, ends, h, split=1), converge, frac)
                              for h in (1.0, 2.0 ** -150))
    assert np.array_equal(one, small) and np.array_equal(fa, fb)
    # a second gas out of the fast solver's range, of which there is none: the single-fluid run
    lone, _ = _run(hg, m, n, s, _config(m, n, ends, split=1), converge)
    pure, _ = _run(hg, m, n, s, _config(m, n, ends, split=1), converge, np.ones((m, n)), 1.0 + 2.0 ** -22)
    assert np.array_equal(lone, pure)


@pytest.mark.parametrize("ends", ENDS)
@pytest.mark.parametrize("g2d", [False, True], ids=["Q1D", "G2D"])
def test_unsplit(hg, oracle_devpow, ends, g2d):
    m, n = 17, 22
    s = _scaled(cases.smooth_random(m, n, 9), UNIT)
    cfg = _config(m, n, ends, split=0)
    for converge in (False, True):
        want, k, _, _, st = oracle_devpow.unsplit2d(m, n, s, cfg, newton_tol=TOL, converge=converge, g2d=g2d)
        assert st == 0
        for form in (hg.UNSPLIT_TILE, hg.UNSPLIT_STRIP):
            assert np.array_equal(_run(hg, m, n, s, cfg, converge, g2d=g2d, form=form)[0], want[:, k - 1]), (converge, form)


def test_batch(hg):
    sizes = [(17, 22), (5, 9), (30, 3)]
    states = [cases.smooth_random(m, n, m) for m, n in sizes]
    out = []
    for h in (1.0, 2.0 ** -150):
        cfg = make_config(t_all=10.0, N=9, bc_x=-2, bc_y=-7, eps=EPS, split=1)
        b = hg.Batch2D([(m, n, h / m, h / n) for m, n in sizes], cfg)
        try:
            b.set_newton(TOL)
            b.upload(states)
            b.run()
            assert not b.results()[1].any()
            out.append(b.download())
        finally:
            b.close()
    assert all(np.array_equal(a, b) for a, b in zip(*out))


@pytest.mark.parametrize("bc", [-4, -7, -2, -24, -1])
def test_ensemble(hg, bc):
    cells = np.array([1, 2, 63, 64, 65, 130])
    rng = np.random.default_rng(abs(bc))
    x = np.concatenate([(np.arange(m) + 0.5) / m for m in cells])
    rho, u, p = (b + 0.2 * np.sin(2 * np.pi * (x + rng.random())) for b in (1.0, 0.05, 1.0))
    out = []
    for h in (1.0, 2.0 ** -150):
        e = hg.Ensemble1D(cells, h / cells, make_config(t_all=10.0, N=9, bc_x=bc, eps=EPS))
        try:
            e.upload(rho, u, p)
            e.run()
            steps, status, _ = e.results()
            out.append((e.download(), steps, status))
        finally:
            e.close()
    (one, *r1), (small, *r2) = out
    assert all(np.array_equal(a, b) for a, b in zip(r1, r2)) and np.all(r1[0][1:] >= 9)
    assert np.array_equal(one, small, equal_nan=True)


@pytest.mark.parametrize("direction,nxy", [(0, (1.0, 0.0)), (1, (0.0, 1.0))])
@pytest.mark.parametrize("near", [False, True])
def test_batches_through_both_solvers(hg, direction, nxy, near):
    """flux_batch runs the steps' solver, flux_general_batch the IEEE one: the same
    bits.  near: values a few ulps from powers of two, where reciprocals lie next
    to the middle of two doubles."""
    n, rng = 100000, np.random.default_rng(5)
    L, R = (np.array(A) for A in cases.interface_pairs(n, 51))
    for A in (L, R):
        A[:, 11:15] = 0.0
        if near:
            for q, sign in ((3, 1), (6, 1), (4, 0), (5, 0), (7, 0), (8, 0), (9, 0), (10, 0)):
                x = 2.0 ** rng.integers(-2, 3, n) * (1.0 - rng.integers(-9, 40, n) * 2.0 ** -53)
                A[:, q] = x if sign else x * rng.choice([-1.0, 0.0, 1.0], n)
    got = hg.flux_batch(L, R, 1e-3, 1e-9, direction)
    want = hg.flux_general_batch(L, R, 1e-3, 1e-9, *nxy)
    ok = want[:, 0] == 0
    assert np.array_equal(got[:, 0] != 0, ~ok) and ok.mean() > 0.5
    assert np.array_equal(got[ok, 1:9], want[ok, 1:9])
