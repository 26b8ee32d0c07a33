"""Grids of few cells in x: the X sweep's lines of 4 and 8 lanes
(csrc/sweep2d.hpp x_lanes) at the edges of their layout, and the size rule that
takes them, for one grid, a batch and two fluids; the unsplit step's tile of 9 x 6
cells (csrc/unsplit2d.hip tile_shape)."""
import numpy as np
import pytest

import cases
from _libs import make_config
from conftest import parity

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hg():
    import hydrogrp
    hydrogrp.lib()
    return hydrogrp


def _config(m, n, **kw):
    return make_config(h_x=1 / m, h_y=1 / n, bc_x=-2, bc_y=-7, split=1, **kw)


@pytest.mark.parametrize("m,n", [(2, 16), (3, 15), (4, 64), (5, 63), (6, 65), (8, 130)])
def test_layout_edges(hg, oracle, m, n):
    init = cases.smooth_random(m, n, m + 100 * n)
    cfg = _config(m, n, t_all=0.03)
    fo, npo, tpo, co, st = oracle.split2d(m, n, init, cfg)
    first = None
    for xv in (0, 2, 4):
        fg, npg, tpg, cg, res = hg.run_split2d(m, n, init, cfg, sweeps=(xv, 0))
        assert (co[5], npo, tpo[npo - 1], st) == (cg[5], npg, tpg[npg - 1], res.status), xv
        first = fg[:, npg - 1] if first is None else first
        assert np.array_equal(fg[:, npg - 1], first), xv
    assert parity(first, fo[:, npo - 1]).max() <= 1e-10      # glibc's pow against the device's


# 769 blocks of 16 lanes and more: the lanes that give the fewest blocks; below, 4 lanes on up to 3 cells
@pytest.mark.parametrize("m,n,w,lanes", [(1, 12305, 4, 4), (3, 12305, 4, 4), (4, 12305, 4, 8), (7, 12305, 4, 8),
                                         (9, 12305, 4, 4), (15, 12305, 4, 16), (16, 8192, 4, 8), (22, 8192, 4, 16),
                                         (1, 49, 4, 4), (3, 64, 4, 4), (3, 32, 3, 16), (3, 304, 4, 4), (4, 304, 3, 16)])
def test_size_rule(hg, m, n, w, lanes):
    s0 = cases.smooth_random(m, n, m)
    cfg = _config(m, n, t_all=1.0)
    out = []
    for two, xv in ((False, None), (False, 0), (True, None)):
        c = hg.Solver2D(m, n, cfg)
        try:
            if xv is None and not two:
                assert c.sweep_kernel(0) == f"sweep_x_kernel<{w}, 0, {lanes}>"
            if xv is not None:
                c.set_sweeps(xv, 0)
            c.upload(s0["rho"], s0["u"], s0["v"], s0["p"])
            if two:
                c.set_fluids(1.67, np.ones((m, n)))           # all of it fluid a: the single-fluid operations
                assert c.sweep_kernel(0) == f"sweep_x_tf_kernel<0, {lanes}>"
            c.bench(3)
            out.append(np.asarray(c.download()).reshape(5, m, n))
        finally:
            c.close()
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])


def test_batch_of_thin_grids(hg):
    sizes = [(1, 9000), (2, 5001), (3, 4099), (8, 700)]
    states = [cases.smooth_random(m, n, m + n) for m, n in sizes]
    out = []
    for xv in (None, 0, 2, 4):
        cfg = make_config(t_all=1.0, N=4, bc_x=-4, bc_y=-4, split=1)
        b = hg.Batch2D([(m, n, 0.01, 0.01) for m, n in sizes], cfg)
        try:
            if xv is not None:
                b.set_sweeps(xv, 0)
            b.upload(states)
            b.run()
            out.append(b.download())
        finally:
            b.close()
    for got in out[1:]:
        assert all(np.array_equal(a, g) for a, g in zip(out[0], got))


# 3073 tiles of 7 x 8 and more, and a quarter fewer of 9 x 6: the unsplit step's second tile shape
@pytest.mark.parametrize("g2d", [False, True], ids=["Q1D", "G2D"])
@pytest.mark.parametrize("m,n,shape", [(8, 12289, 2), (9, 12293, 2), (8, 12288, 1), (10, 12289, 1), (7, 24577, 1)])
def test_unsplit_tile_shape(hg, m, n, shape, g2d):
    s0 = cases.smooth_random(m, n, m)
    for bx, by in ((-2, -7), (-24, -1)):
        cfg = make_config(t_all=1.0, h_x=1 / m, h_y=1 / n, bc_x=bx, bc_y=by, split=0)
        out = []
        for form in (hg.UNSPLIT_TILE, hg.UNSPLIT_STRIP):
            c = hg.Solver2D(m, n, cfg)
            try:
                if g2d:
                    c.set_interface_solver(True)
                c.set_unsplit_form(form)
                if form == hg.UNSPLIT_TILE:
                    assert c.sweep_kernel(2) == f"unsplit_step_{'g2d_' if g2d else ''}kernel<12, {shape}, 0>"
                c.upload(s0["rho"], s0["u"], s0["v"], s0["p"])
                c.bench_unsplit(3)
                out.append(np.asarray(c.download()))
            finally:
                c.close()
        assert np.array_equal(out[0], out[1]), (bx, by)


@pytest.mark.parametrize("m,n", [(1, 33), (1, 64), (2, 33), (2, 64), (3, 33)])
def test_round_trip_of_few_rows(hg, m, n):
    """Grids of one or two rows come down row by row (csrc/layout2d.hip): any of the fields alone, too."""
    s = cases.smooth_random(m, n, m + n)
    c = hg.Solver2D(m, n, _config(m, n, t_all=0.1))
    try:
        c.upload(s["rho"], s["u"], s["v"], s["p"])
        got = np.asarray(c.download()).reshape(5, m, n)
        for f, k in enumerate(("rho", "u", "v", "p")):
            assert np.array_equal(got[f], s[k].reshape(m, n)), k
        a = np.random.default_rng(n).random((m, n))
        c.set_fluids(1.67, a)
        assert np.array_equal(np.asarray(c.download_fraction()).reshape(m, n), a)
        p = np.empty((m, n))
        assert hg.lib().hgrp2d_download(c._h, None, None, None, hg._p(p), None) == 0
        assert np.array_equal(p, s["p"].reshape(m, n))
    finally:
        c.close()
