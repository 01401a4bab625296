"""Stages of small grids by blocks of one wave per face (k_block_yx,
k_block_z) against the march: a fixed march segment selects the march, and
both evaluate the same faces, sums and updates with the same operations, so
the states are equal bit for bit.  Sizes at the edges of the blocks: one row
to several blocks of rows, 63 / 64 columns and one more, one to several
blocks along z, every scheme, flux, time recipe and boundary kind."""
import numpy as np
import pytest

from sonicsolver_amd import workloads as wl
from sonicsolver_amd._native import Grid, SonicError, make_desc

pytestmark = pytest.mark.gpu

SIZES = [(8, 8), (9, 13), (63, 10), (64, 11), (65, 12), (66, 64), (67, 9), (128, 31), (130, 130),
         (200, 90), (8, 8, 8), (64, 9, 12), (66, 12, 15), (24, 30, 22), (40, 40, 40)]
RECIPES = [("weno5", "hllc", "ssprk3"), ("weno5", "rusanov", "rk4"), ("teno5", "hllc", "euler"),
           ("weno3", "roe", "ssprk3"), ("weno7", "steger", "ssprk3"), ("weno7", "hllc", "rk4"),
           ("weno3", "laxwendroff", "euler"), ("teno5", "laxfriedrichs", "ssprk3")]


@pytest.mark.parametrize("bc", ["transmissive", "periodic"])
@pytest.mark.parametrize("scheme,flux,time", RECIPES)
def test_blocks_equal_march(scheme, flux, time, bc):
    for k, n in enumerate(SIZES):
        h = [1.0 / m for m in n] + [1.0] * (3 - len(n))
        desc = make_desc(n=n, bc=(bc,) * 3, d=h, scheme=scheme, flux=flux, time=time)
        q = wl.smooth_field(n, seed=k + 1, amp=0.1)
        print(n, scheme, flux, time, bc, flush=True)
        with Grid(desc) as g:
            g.upload(q)
            dts = g.run(3, 0.2)
            blocks = g.download()
            g.upload(q)
            g.set_march_segment(5)
            march_dts = g.run(3, 0.2)
            assert np.array_equal(g.download(), blocks), n
            assert np.array_equal(march_dts, dts), n


@pytest.mark.parametrize("scheme,flux,time", [("weno5", "hllc", "ssprk3"),
                                              ("teno5", "rusanov", "rk4"),
                                              ("weno3", "laxwendroff", "euler"),
                                              ("weno7", "roe", "ssprk3")])
@pytest.mark.parametrize("n", [(502, 499), (600, 613), (640, 601), (1000, 333), (65, 61, 70),
                               (64, 64, 64)])
def test_stacked_waves_equal_single(n, scheme, flux, time):
    """Blocks of four waves that share the y faces between them, with the last
    block's waves full, partly filled and without rows."""
    h = [1.0 / m for m in n] + [1.0] * (3 - len(n))
    q = wl.smooth_field(n, seed=5, amp=0.1)
    for bc in ("transmissive", "periodic"):
        with Grid(make_desc(n=n, bc=(bc,) * 3, d=h, scheme=scheme, flux=flux, time=time)) as g:
            g.upload(q)
            dts = g.run(2, 0.2)
            stacked = g.download()
            g.upload(q)
            g.set_march_segment(7)
            assert np.array_equal(g.run(2, 0.2), dts)
            assert np.array_equal(g.download(), stacked)


def test_fault_keeps_the_step_start():
    """Two halves that move apart until a near-vacuum turns non-physical in
    some stage: both paths stop at the same step and stage, with the state at
    the start of that step."""
    n = (65, 40)
    x = np.arange(n[0])
    u = np.where(x < n[0] // 2, -2.0, 2.0)
    q = wl.conserved(np.ones(n[::-1]), u + np.zeros(n[::-1]), 0.0, 0.0, 0.4)
    seen = []
    for seg in (0, 6):
        with Grid(make_desc(n=n, d=(0.1, 0.1, 1.0), flux="hllc")) as g:
            if seg:
                g.set_march_segment(seg)
            g.upload(q)
            with pytest.raises(SonicError):
                g.run(200, 0.5)
            flags, step, phase = g.fault()
            print(seg, flags, step, phase, flush=True)
            assert flags and step > 1 and phase < 4
            seen.append((step, phase, g.clock(), g.download()))
    assert seen[0][:3] == seen[1][:3]
    assert np.array_equal(seen[0][3], seen[1][3])
