"""The fused y / x stage launch against the separate sweeps.

Both form every face, sum and update by the same functions in the same
order, so their states are compared bit for bit, at the sizes where the
launch's columns, helper lane, row segments and ring wrap end."""
import numpy as np
import pytest

from sonicsolver_amd import Grid, make_desc, workloads as wl

pytestmark = pytest.mark.gpu

# (n, bc): one column block and its edges, two blocks whose 63-column form
# needs no third (126) and whose 64-column form does (127, 128), remainders of
# the 32-row segments, the smallest grids, ends of every kind
CASES = [((4, 4), "transmissive"), ((31, 33), "periodic"), ((63, 32), "none"),
         ((64, 5), "transmissive"), ((65, 97), "none_lo"), ((126, 40), "periodic"),
         ((127, 31), "transmissive"), ((128, 70), "none_hi"), ((193, 64), "transmissive"),
         ((4, 9, 5), "periodic"), ((64, 33, 7), "transmissive"), ((129, 12, 6), "none"),
         ((24, 40, 300), "periodic")]


@pytest.mark.parametrize("scheme,flux,time", [("weno5", "hllc", "ssprk3"), ("teno5", "rusanov", "rk4"),
                                              ("weno3", "roe", "euler"),
                                              ("weno7", "laxwendroff", "ssprk3")])
@pytest.mark.parametrize("n,bc", CASES)
def test_fused_launch_equals_separate_sweeps(n, bc, scheme, flux, time):
    print(f"fused yx {n} {bc} {scheme}/{flux}/{time}", flush=True)
    q = wl.smooth_field(n)
    desc = make_desc(n=n, bc=(bc,) * 3, d=tuple(1.0 / x for x in n) + (1.0,) * (3 - len(n)),
                     scheme=scheme, flux=flux, time=time)
    out = []
    for walk, seg in ((0, 0), (-1, 0), (-1, 32), (-1, 3)):
        with Grid(desc) as g:
            g.set_x_walk(walk)
            g.set_march_segment(seg)
            g.upload(q)
            dts = g.run(3, 0.3)
            out.append((g.download(), dts))
    for state, dts in out[1:]:
        assert np.array_equal(state, out[0][0])
        assert np.array_equal(dts, out[0][1])


@pytest.mark.parametrize("n", [(70, 33), (40, 20, 9)])
def test_boundary_nodes_follow_the_path_taken(n):
    """An upload is handed back as it is until the boundary is prepared;
    then every zeroGradient boundary node holds its inner neighbour.  Steps
    may change between the fused launch and the separate sweeps, whose
    ghosts are stored."""
    q = wl.smooth_field(n)
    desc = make_desc(n=n, bc=("transmissive", "none_hi", "periodic"),
                     d=tuple(1.0 / x for x in n) + (1.0,) * (3 - len(n)))
    shape = (5,) + tuple(reversed(n + (1,) * (3 - len(n))))
    with Grid(desc) as g:
        g.upload(q)
        assert np.array_equal(g.download(), q)
        g.prepare()
        s = g.download().reshape(shape)
        assert np.array_equal(s[:4, :, 1:, 0], q.reshape(shape)[:4, :, 1:, 1])
        assert np.array_equal(s[:4, :, 0, :], s[:4, :, 1, :])
        np.testing.assert_allclose(s[4, :, 1:, -1], q.reshape(shape)[4, :, 1:, -2], rtol=1e-15)
        g.run(6, 0.3)
        ref = g.download()
        g.upload(q)
        for walk in (-1, 0, -1):
            g.set_x_walk(walk)
            g.run(2, 0.3)
        assert np.array_equal(g.download(), ref)
