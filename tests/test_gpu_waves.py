"""The wave-parallel sweeps (csrc/sweep2d_body.hpp wave_sweep) at the edges of
their layout: lines that end with a wave's last updated cell, one before and one
after it, groups of lines that fill a block or leave waves idle; and the launch
variant that a grid's size selects."""
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


@pytest.mark.parametrize("m,n", [(1, 1), (14, 15), (15, 16), (16, 17), (7, 8), (31, 4), (32, 33), (63, 14), (61, 46)])
def test_layout_edges(hg, oracle, m, n):
    init = cases.smooth_random(m, n, m + 100 * n)
    cfg = make_config(t_all=0.03, h_x=1 / m, h_y=1 / n, bc_x=-2, bc_y=-7, split=1)
    fo, npo, tpo, co, st = oracle.split2d(m, n, init, cfg)
    first = None
    for sweeps in (None, (0, 0), (1, 1), (2, 3), (3, 4), (4, 2), (5, 1)):
        fg, npg, tpg, cg, res = hg.run_split2d(m, n, init, cfg, sweeps=sweeps)
        assert (co[5], npo, tpo[npo - 1], st) == (cg[5], npg, tpg[npg - 1], res.status), sweeps
        first = fg[:, npg - 1] if first is None else first
        assert np.array_equal(fg[:, npg - 1], first), sweeps
    assert parity(first, fo[:, npo - 1]).max() <= 1e-10      # glibc's pow against the device's


@pytest.mark.parametrize("m,n,w", [(1, 1, 3), (384, 384, 3), (512, 512, 4), (100, 1000, 3), (1000, 1000, 4)])
def test_default_variant(hg, m, n, w):
    s = hg.Solver2D(m, n, make_config(t_all=0.1, h_x=1 / m, h_y=1 / n, bc_x=-4, bc_y=-4, split=1))
    try:
        assert s.sweep_kernel(0) == f"sweep_x_kernel<{w}, 0, 16>" and s.sweep_kernel(1) == f"sweep_y_kernel<{w}, 0, 16>"
    finally:
        s.close()


@pytest.mark.parametrize("m,n", [(1, 1), (14, 15), (15, 16), (16, 17), (31, 4), (33, 46)])
def test_two_fluid_layout_edges(hg, oracle, m, n):
    """Cells that are all fluid a run as the single fluid, bit for bit."""
    s0 = cases.smooth_random(m, n, m + 100 * n)
    cfg = make_config(t_all=1.0, h_x=1 / m, h_y=1 / n, bc_x=-2, bc_y=-7, split=1)
    out = []
    for two in (False, True):
        c = hg.Solver2D(m, n, cfg)
        try:
            c.upload(s0["rho"], s0["u"], s0["v"], s0["p"])
            if two:
                c.set_fluids(1.67, np.ones((m, n)))        # all of it fluid a: the single-fluid operations
            c.bench(7)
            out.append(np.asarray(c.download()).reshape(5, m, n))
            if two:
                assert np.array_equal(c.download_fraction().reshape(m, n), np.ones((m, n)))
        finally:
            c.close()
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("g2d", [False, True], ids=["Q1D", "G2D"])
@pytest.mark.parametrize("m,n", [(1, 1), (6, 7), (7, 8), (8, 9), (14, 31), (15, 33), (2, 40)])
def test_unsplit_tile_edges(hg, oracle, m, n, g2d):
    init = cases.smooth_random(m, n, m + 100 * n)
    for bx, by in ((-4, -4), (-2, -7), (-24, -1)):
        cfg = make_config(t_all=0.03, h_x=1 / m, h_y=1 / n, bc_x=bx, bc_y=by, split=0)
        tp = np.array([0.0, cfg[1]])
        fo, npo, tpo, co, st = oracle.unsplit2d(m, n, init, cfg, time_plot=tp, g2d=g2d)
        tile, strip = (hg.run_unsplit2d(m, n, init, cfg, time_plot=tp, g2d=g2d, form=f)
                       for f in (hg.UNSPLIT_TILE, hg.UNSPLIT_STRIP))
        for fg, npg, tpg, cg, res in (tile, strip):
            assert (co[5], npo, tpo[npo - 1], st) == (cg[5], npg, tpg[npg - 1], res.status), (bx, by)
            assert parity(fg[:, npg - 1], fo[:, npo - 1]).max() <= 1e-10, (bx, by)      # glibc's pow against the device's
        assert np.array_equal(tile[0][:, npo - 1], strip[0][:, npo - 1])
