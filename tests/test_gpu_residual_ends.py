"""A residual between steps leaves everything that the steps read as it was:
the ghosts that an end without a condition holds since the upload are stored
in every state buffer, the residual's scratch buffer among them."""
import numpy as np
import pytest

from sonicsolver_amd import Grid, make_desc, workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("time", ["euler", "ssprk3", "rk4"])
@pytest.mark.parametrize("bc", ["none", "none_lo", "none_hi", "transmissive"])
@pytest.mark.parametrize("n,walk", [((101,), -1), ((101,), 0), ((70, 33), -1), ((70, 33), 1),
                                    ((20, 12, 9), -1)])
def test_run_is_the_same_after_a_residual(n, walk, bc, time):
    print(f"residual {n} walk {walk} {bc} {time}", flush=True)
    q = wl.smooth_field(n)
    desc = make_desc(n=n, bc=(bc,) * 3, d=tuple(1.0 / x for x in n) + (1.0,) * (3 - len(n)),
                     scheme="weno5", flux="hllc", time=time)
    out = []
    for residual in (False, True):
        with Grid(desc) as g:
            g.set_x_walk(walk)
            g.upload(q)
            dts = []
            r = []
            for k in range(4):   # each buffer is the scratch once
                if residual:
                    r.append(g.residual())
                    assert np.array_equal(r[-1], g.residual())
                dts.append(g.run(1 + k % 2, 0.3))
            out.append((g.download(), np.concatenate(dts), g.clock()))
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])
    assert out[0][2] == out[1][2]
