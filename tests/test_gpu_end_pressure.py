"""A node next to a zeroGradient end whose pressure vanishes: the boundary
closure rebuilds the end's energy from that pressure and stops where it is
not positive (SF_thermodynamicClosure.cpp:219-281).  Its rounding differs
from the state check's by some units in the last place, so a step is placed
there by bisection on dt, and the fused launches, which close the ends
themselves, have to refuse the steps that the ghost fill of the separate
sweeps refuses."""
import numpy as np
import pytest

from sonicsolver_amd import Grid, make_desc

pytestmark = pytest.mark.gpu


def _state(rng, n):
    N = int(np.prod(n))
    rho = 1 + 0.3 * rng.random(N)
    u, v = 3 + rng.random(N), 0.5 * rng.normal(size=N)
    p = 0.5 + 0.5 * rng.random(N)
    return np.stack([rho, rho * u, rho * v, 0 * u, p / 0.4 + 0.5 * rho * (u * u + v * v)])


def _fault(g, q, dt):
    """The fault of one Euler step with this dt."""
    g.upload(q)
    try:
        g.run(1, 100.0, max_dt=dt)
    except RuntimeError:
        pass
    return g.fault()


@pytest.mark.parametrize("n,seeds", [((12, 10), 150), ((40,), 150), ((9, 7, 6), 60)])
def test_fused_launches_refuse_what_the_fill_refuses(n, seeds):
    desc = make_desc(n=n, bc=("transmissive",) * 3, d=(0.1,) * len(n) + (1.0,) * (3 - len(n)),
                     scheme="weno5", flux="hllc", time="euler")
    between = placed = 0
    with Grid(desc) as sep, Grid(desc) as fused:
        sep.set_x_walk(0)
        for seed in range(seeds):
            q = _state(np.random.default_rng(seed), n)
            low, high = 1e-3, 0.2
            if _fault(sep, q, low)[0] or not _fault(sep, q, high)[0]:
                continue
            while np.nextafter(low, high) < high:
                mid = 0.5 * (low + high)
                if _fault(sep, q, mid)[0]:
                    high = mid
                else:
                    low = mid
            placed += 1
            for t in range(-8, 12):
                dt = low + t * np.spacing(low)
                a, b = _fault(sep, q, dt), _fault(fused, q, dt)
                assert a[0] == b[0], (seed, dt, a, b)
                between += a[2] == 6   # the fill refused what the stage passed
    print(f"end pressure {n}: {placed} states, {between} steps refused by the fill", flush=True)
    assert placed > 5 and between > 0
