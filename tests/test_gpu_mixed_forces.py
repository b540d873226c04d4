"""The mixed form's hourglass forces beside large stress forces: the two kinds
meet in float64, so the small one keeps the precision of its own size."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_hourglass_forces_under_large_pressure(lulesh_gpu):
    """A regular lattice of exact spacing under one pressure: the stress
    forces are exact in float32 and cancel on every inner node, which only
    the hourglass forces of random velocities move.  They are 10^-7 of the
    stress forces, an ulp of float32."""
    nx, dt, p0 = 6, 1e-6, 2.0 ** 20
    en = nx + 1
    rng = np.random.default_rng(5)
    k, j, i = (a.ravel().astype(np.float64) for a in np.meshgrid(*[np.arange(en)] * 3,
                                                               indexing="ij"))
    moved = {}
    for mixed in (False, True):
        d = lulesh_gpu.Domain(nx, mixed=mixed)
        if not moved:
            vel = {f: rng.uniform(-1, 1, d.num_node) for f in ("xd", "yd", "zd")}
        one = np.ones(d.num_elem)
        d.upload_state({"x": i * 0.25, "y": j * 0.25, "z": k * 0.25, **vel, "e": 0 * one,
                        "p": p0 * one, "q": 0 * one, "v": one, "ss": one, "time": 0.0,
                        "deltatime": dt})
        volo, mass = d.get("volo").reshape(nx, nx, nx), d.get("nodalMass").reshape(en, en, en)
        assert d.step(1) == (0, 1)
        moved[mixed] = {f: (d.get(f) - vel[f]).reshape(en, en, en)[1:-1, 1:-1, 1:-1]
                        for f in vel}
        d.close()
    # On the lattice an element's four hourglass modes of the velocity are sums
    # of its corners' differences from corner 0, and a corner's force is coef
    # times a sum of the four.  Each takes fewer than 24 roundings of float32
    # (coefficient and cube root among them) of values below coef times four
    # times the sum of the differences; the eight corners of a node add in
    # float64.
    coef = 0.03 * volo / np.cbrt(volo)
    for f in vel:
        u = vel[f].reshape(en, en, en)
        diff = np.zeros((nx, nx, nx))
        for c in np.ndindex(2, 2, 2):
            diff += np.abs(u[c[0]:c[0] + nx, c[1]:c[1] + nx, c[2]:c[2] + nx] -
                           u[:nx, :nx, :nx])
        bound = np.zeros((en, en, en))
        for c in np.ndindex(2, 2, 2):
            bound[c[0]:c[0] + nx, c[1]:c[1] + nx, c[2]:c[2] + nx] += 4 * coef * diff
        bound = (24 * 2.0 ** -24 * bound / mass * dt)[1:-1, 1:-1, 1:-1]
        assert np.all(np.abs(moved[True][f] - moved[False][f]) <= bound), f
        assert np.max(np.abs(moved[False][f])) > 100 * np.max(bound)
