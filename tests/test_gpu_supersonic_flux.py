"""HLLC where the whole fan leaves the face: the flux is the upwind side's own
physical flux, whose mass component is that side's normal momentum, bit for
bit; the others are products of it and quotients by the density.  With one
Newton step those are within 40 units in the last place of a double (the
squared reciprocal root's 20, twice), and two such factors and the pressure
stay within 200 of the largest component."""
import numpy as np
import pytest

from sonicsolver_amd._native import face_flux, riemann_flux
from tests import hllc_fan as hf

pytestmark = pytest.mark.gpu


def _stream(count, seed, axis, sign):
    rng = np.random.default_rng(seed)
    q = []
    for _ in range(count):
        rho, p = rng.uniform(0.1, 2.0), rng.uniform(0.1, 5.0)
        u = rng.uniform(-1, 1, 3)
        u[axis] = sign * np.sqrt(1.4 * p / rho) * rng.uniform(1.6, 6.0)
        q.append(hf.conserved(rho, u, p))
    return np.array(q)


@pytest.mark.parametrize("sign", [1.0, -1.0])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_supersonic_mass_flux_is_the_momentum(axis, sign):
    n = hf.NORMALS[axis]
    q = _stream(500, 7 + axis, axis, sign)
    print(f"supersonic hllc axis {axis} sign {sign}", flush=True)
    ref = np.array([hf.euler_flux(a, n) for a in q])
    tol = 200 * 2.0 ** -52 * np.abs(ref).max(axis=1, keepdims=True)
    for scheme in ("weno5", "teno5"):
        out, flags = face_flux(scheme, "hllc", axis, np.repeat(q[:, None], 6, axis=1))
        assert not flags.any()
        assert np.array_equal(out[:, 0], q[:, 1 + axis]), scheme
        assert (np.abs(out - ref) <= tol).all(), scheme
    # between two different streams: the upwind one's
    other = q.copy()
    other[:, 0] *= 1.01
    qL, qR = (q, other) if sign > 0 else (other, q)
    out, flags = riemann_flux("hllc", axis, qL, qR)
    assert not flags.any()
    assert np.array_equal(out[:, 0], q[:, 1 + axis])
    assert (np.abs(out - ref) <= tol).all()
