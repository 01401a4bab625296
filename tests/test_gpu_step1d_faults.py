"""What stops a whole-step launch of a 1D grid, and what the record says
then, against the launch-per-stage path (set_x_walk(0))."""
import numpy as np
import pytest

from sonicsolver_amd import Grid, SonicError, make_desc, workloads as wl

pytestmark = pytest.mark.gpu

# Thin gas whose face just beyond an end without a condition, no face of the
# grid, turns non-physical while every face of the grid is sound (found by a
# search with the oracle): recipe, CFL number, steps, then rho, u and p.
BEYOND_THE_END = [
    ("weno7", "rusanov", "rk4", 0.3, 10,
     [3.81e-06, 3.98e-06, 4.19e-06, 4.43e-06, 4.7e-06, 4.97e-06, 5.24e-06, 5.48e-06],
     [1960.0, 1960.0, 1900.0, 1870.0, 1920.0, 1950.0, 1980.0, 2010.0],
     [1.4, 3.14, 5.19, 5.18, 3.1, 1.34, 0.566, 0.0774]),
    ("weno5", "rusanov", "euler", 0.3, 10,
     [4.45e-06, 3.61e-06, 3.29e-06, 3.45e-06, 4.08e-06, 5.09e-06, 6.15e-06, 6.69e-06],
     [873.0, 1140.0, 1260.0, 1310.0, 1470.0, 1780.0, 2090.0, 2160.0],
     [0.892, 0.345, 0.417, 1.34, 3.47, 2.58, 0.673, 0.222]),
    ("weno3", "hllc", "ssprk3", 0.3, 10,
     [0.000103, 0.000101, 7.35e-05, 6.97e-05, 0.00012, 0.000158, 8.89e-05, 5.69e-05, 9.09e-05],
     [253.0, 261.0, 262.0, 254.0, 245.0, 246.0, 255.0, 262.0, 259.0],
     [0.48, 0.346, 0.355, 0.704, 2.11, 4.78, 4.68, 2.1, 0.252]),
    ("weno5", "hllc", "rk4", 0.5, 7,
     [1.59e-06, 1.68e-06, 1.81e-06, 1.95e-06, 2.05e-06, 2.09e-06, 2.03e-06, 1.91e-06, 1.74e-06,
      1.58e-06],
     [-3380.0, -3500.0, -3490.0, -3340.0, -3090.0, -2790.0, -2500.0, -2310.0, -2260.0, -2360.0],
     [0.0951, 0.208, 0.641, 1.03, 0.716, 0.45, 0.535, 1.05, 1.51, 1.01]),
    ("weno7", "hllc", "ssprk3", 0.5, 8,
     [2.7e-06, 2.75e-06, 2.82e-06, 2.91e-06, 2.99e-06, 3.06e-06, 3.11e-06, 3.13e-06, 3.11e-06,
      3.06e-06],
     [321.0, 326.0, 337.0, 351.0, 367.0, 381.0, 391.0, 396.0, 398.0, 397.0],
     [0.954, 1.25, 1.17, 0.937, 0.911, 1.14, 1.36, 1.24, 0.964, 0.17]),
]


@pytest.mark.parametrize("case", BEYOND_THE_END, ids=lambda c: "-".join(c[:3]))
@pytest.mark.parametrize("mirror", [False, True])
def test_faces_beyond_an_end_stop_nothing(case, mirror):
    scheme, flux, time, cfl, steps, rho, u, p = case
    rho, u, p = (np.array(x) for x in (rho, u, p))
    if mirror:
        rho, u, p = rho[::-1], -u[::-1], p[::-1]
    q = np.stack([rho, rho * u, 0 * u, 0 * u, p / 0.4 + 0.5 * rho * u * u])
    n = len(rho)
    print(f"beyond the end {scheme}/{flux}/{time} mirror {mirror}", flush=True)
    desc = make_desc(n=(n,), bc=("none",) * 3, d=(1.0 / n, 1.0, 1.0), scheme=scheme, flux=flux,
                     time=time)
    out = []
    for walk in (0, -1):
        with Grid(desc) as g:
            g.set_x_walk(walk)
            g.upload(q)
            dts = g.run(steps, cfl)
            out.append((dts, g.download(), g.clock(), g.fault()))
    assert out[0][3] == out[1][3] == (0, 0, -1)
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])
    assert out[0][2] == out[1][2]


def _no_pressure_at(q, k):
    q = q.copy()
    q[4, k] = -1.0
    return q


@pytest.mark.parametrize("time", ["euler", "ssprk3", "rk4"])
@pytest.mark.parametrize("node,phase", [(1, 6), (200, 7)])
def test_a_fault_before_the_run_is_kept(node, phase, time):
    """Raised by the ghost fill (phase 6) or the CFL scan (7) of the state a
    run starts from, or by the residual or the scan before the run, a fault
    stops the run's first step like every launch: flags, step and phase stay
    as they were recorded, and nothing advances."""
    n = 401
    kw, q = wl.riemann_1d(n - 1, (1.0, 0.0, 1.0), (0.5, 0.0, 0.5), 0.5)
    bad = _no_pressure_at(q, node)
    desc = make_desc(n=(n, 1, 1), active=(1, 0, 0), d=(kw["d"][0], 1.0, 1.0), time=time)

    def run(g):
        with pytest.raises(SonicError):
            g.run(3, 0.4)

    def scan(g):
        with pytest.raises(SonicError):
            g.prepare()
            g.compute_dt(0.4)

    def residual(g):
        with pytest.raises(SonicError):
            g.residual()

    for before in (None, scan, residual):
        got = []
        for walk in (0, -1):
            with Grid(desc) as g:
                g.set_x_walk(walk)
                g.upload(q)
                g.run(2, 0.4)
                g.upload(bad)
                if before:
                    before(g)
                first = g.fault() if before else None
                run(g)
                got.append((g.fault(), g.clock(), g.download()[:, 2:-2]))
                if before:
                    assert got[-1][0] == first
                # a sound state runs again from the accumulators left behind
                g.upload(q)
                got[-1] += (g.run(4, 0.4), g.download())
        assert got[0][0] == got[1][0]
        if before is not residual:
            assert got[1][0][2] == phase
        assert got[0][1] == got[1][1]
        for k in (2, 3, 4):
            assert np.array_equal(got[0][k], got[1][k])
