"""Whole 1D steps in one launch against the launch-per-stage path (chosen
with set_x_walk): the same faces and updates, so states, dt sequences and
clocks are equal bit for bit, at the sizes where the launch's tiles begin
and end."""
import numpy as np
import pytest

from sonicsolver_amd import Grid, SonicError, make_desc, workloads as wl

pytestmark = pytest.mark.gpu

# nodes a block advances are 64 - 2 halo stages: 46 (WENO5, SSPRK3), 40
# (TENO5, RK4), 60 (WENO3, Euler), 32 (WENO7, RK4)
RECIPES = [("weno5", "hllc", "ssprk3"), ("teno5", "rusanov", "rk4"), ("weno3", "roe", "euler"),
           ("weno7", "laxwendroff", "rk4"), ("weno5", "steger", "euler")]
SIZES = [4, 5, 31, 33, 40, 46, 47, 61, 64, 92, 93, 200, 1001]


@pytest.mark.parametrize("scheme,flux,time", RECIPES)
@pytest.mark.parametrize("bc", ["transmissive", "periodic", "none", "none_lo", "none_hi"])
def test_whole_step_launch_equals_stages(bc, scheme, flux, time):
    for n in SIZES:
        print(f"step1d {n} {bc} {scheme}/{flux}/{time}", flush=True)
        q = wl.smooth_field((n,))
        desc = make_desc(n=(n,), bc=(bc,) * 3, d=(1.0 / n, 1.0, 1.0), scheme=scheme, flux=flux,
                         time=time)
        out = []
        for walk in (0, -1):
            with Grid(desc) as g:
                g.set_x_walk(walk)
                g.upload(q)
                a = g.run(4, 0.3)
                b = g.run(5, 0.3, max_dt=0.9 * a[-1])   # from the folded scan
                g.prepare()
                c = g.compute_dt(0.3)                   # op by op after whole steps
                g.begin()
                for s in range(g.stage_count()):
                    g.stage(s)
                g.commit()
                d = g.run(1, 0.2)                       # another CFL number: scanned again
                out.append((np.concatenate([a, b, [c], d]), g.download(), g.clock()))
        assert np.array_equal(out[0][0], out[1][0])
        assert np.array_equal(out[0][1], out[1][1])
        assert out[0][2] == out[1][2]


def test_fault_is_reported_as_by_the_stages():
    kw, q = wl.riemann_1d(1200, (1.0, -3.0, 1.0), (1.0, 3.0, 1.0), 0.5)
    desc = make_desc(n=(kw["n"][0], 1, 1), active=(1, 0, 0), d=(kw["d"][0], 1.0, 1.0),
                     scheme="weno5", flux="hllc", time="ssprk3")
    got = []
    for walk in (0, -1):
        with Grid(desc) as g:
            g.set_x_walk(walk)
            g.upload(q)
            with pytest.raises(SonicError):
                g.run(40, 0.5)
            got.append((g.fault(), g.clock(), g.download()))
            # a new state starts clean, from accumulators the fault left behind
            kw1, q1 = wl.riemann_1d(1200, (1.0, 0.0, 1.0), (0.5, 0.0, 0.5), 0.5)
            g.upload(q1)
            got[-1] += (g.run(6, 0.5), g.download())
    assert got[0][0] == got[1][0]
    for k in (1, 2, 3, 4):
        assert np.array_equal(got[0][k], got[1][k])
