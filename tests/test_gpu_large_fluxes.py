"""y fluxes that are finite, each of them, while their sum is not, are no
fault: the launches that take the y and x faces together agree with the y
march, which tests them one by one.  Only a uniform stream gets there: a face
area is at most 1.3e154 (its square has to be finite), and the smallest
differences between states of 1e153 overflow the weights."""
import numpy as np
import pytest

from sonicsolver_amd import Grid, make_desc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,seg", [((40, 30), 0), ((40, 30), 8), ((600, 600), 0), ((40, 12, 6), 0)])
def test_finite_y_fluxes_with_an_overflowing_sum(n, seg):
    print(f"large y fluxes {n} segment {seg}", flush=True)
    # y fluxes of mass, momentum and energy 3.6, 5.3 and 6.8 times 2e153 times
    # the y faces' area of 1.3e154
    rho, v, p = 3.0, 1.2, 1.0
    node = np.array([rho, 0.0, rho * v, 0.0, p / 0.4 + 0.5 * rho * v * v]) * 2e153
    q = np.repeat(node[:, None], int(np.prod(n)), axis=1)
    desc = make_desc(n=n, bc=("periodic",) * 3, d=(1.3e154, 1.0, 1.0), scheme="weno5", flux="hllc")
    out = []
    for walk in (0, -1):
        with Grid(desc) as g:
            g.set_x_walk(walk)
            g.set_march_segment(seg)
            g.upload(q)
            g.run(2, 0.3)
            out.append(g.download())
    assert np.array_equal(out[0], out[1])
