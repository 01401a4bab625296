"""The x walk and the march length may change between the stages of a step:
the fused launch, which trusts the boundary that the stage before wrote, and
the separate sweeps, which store none, follow each other in every order, and
the results do not depend on it (bit for bit)."""
import numpy as np
import pytest

from sonicsolver_amd import Grid, make_desc, workloads as wl

pytestmark = pytest.mark.gpu


def _steps(g, steps, before_stage):
    for k in range(steps):
        g.prepare()
        g.compute_dt(0.3)
        g.begin()
        for s in range(g.stage_count()):
            before_stage(k, s)
            g.stage(s)
        g.commit()


def _state(desc, q, before_stage):
    with Grid(desc) as g:
        g.upload(q)
        _steps(g, 4, lambda k, s: before_stage(g, k, s))
        g.set_x_walk(-1)
        g.set_march_segment(0)
        g.run(2, 0.3)
        return g.download(), g.clock()


@pytest.mark.parametrize("time", ["ssprk3", "rk4"])
@pytest.mark.parametrize("n,bc", [((70, 45), "transmissive"), ((33, 20), "periodic"),
                                  ((64, 31), "none_lo"), ((40, 20, 9), "transmissive"),
                                  ((20, 12, 10), "none_hi")])
def test_walk_changes_between_stages(n, bc, time):
    q = wl.smooth_field(n)
    desc = make_desc(n=n, bc=(bc,) * 3, d=tuple(1.0 / x for x in n) + (1.0,) * (3 - len(n)),
                     scheme="weno5", flux="hllc", time=time)
    ref = _state(desc, q, lambda g, k, s: None)
    for walks in ((0, -1), (-1, 0), (1, -1, 0), (-1, 0, 0, -1, 1)):
        print(f"walks {walks} {n} {bc} {time}", flush=True)
        got = _state(desc, q, lambda g, k, s: g.set_x_walk(walks[(4 * k + s) % len(walks)]))
        assert np.array_equal(got[0], ref[0]), walks
        assert got[1] == ref[1]


def test_march_length_changes_between_stages():
    """On a grid narrower than 32 nodes the march length decides between the
    fused launch (long segments) and the separate sweeps (short ones)."""
    n = (24, 100, 100)
    q = wl.smooth_field(n)
    desc = make_desc(n=n, bc=("transmissive",) * 3, d=tuple(1.0 / x for x in n))
    ref = _state(desc, q, lambda g, k, s: None)
    for order in ((1, 32), (32, 1)):
        got = _state(desc, q, lambda g, k, s: g.set_march_segment(order[s % 2]))
        assert np.array_equal(got[0], ref[0]), order
        assert got[1] == ref[1]
