"""The fused build's EOS in reciprocal volumes."""
import math
from fractions import Fraction

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# separate kernels, and k_eos_dt_nat beyond the last-level cache
@pytest.mark.parametrize("nx,every", [(48, 1), (104, 10)])
def test_sound_speed_is_the_rounded_root(lulesh_gpu, nx, every):
    """ss of the 2.0 step is the root of 2/3 (e + v p), correctly rounded: the
    sum in one rounding, the product in one."""
    d = lulesh_gpu.Domain(nx, fused=True)
    st = d.download_state()
    rng = np.random.default_rng(nx)
    st["e"] = 10.0 ** rng.uniform(0, 7, d.num_elem)
    st["deltatime"] = 1e-8
    d.upload_state(st)
    d.step(2)
    e, p, v, ss = (d.get(f)[::every] for f in ("e", "p", "vnew", "ss"))
    d.close()
    assert np.all(p > 0.0) and len(set(v)) > 1000
    wrong = 0
    for i in range(len(e)):
        s = (2.0 / 3.0) * float(Fraction(v[i]) * Fraction(p[i]) + Fraction(e[i]))
        wrong += math.sqrt(s) != ss[i]
    assert wrong == 0


PARAMETERS = [{"eosvmax": 1.02}, {"eosvmin": 0.97}, {"refdens": 1.3},
              {"eosvmax": 1.02, "eosvmin": 0.97, "refdens": 0.7}]


def blast(lulesh_gpu, nx, fused, parameters):
    d = lulesh_gpu.Domain(nx, fused=fused)
    for name, value in parameters.items():
        d.set_parameter(name, value)
    return d


@pytest.mark.parametrize("parameters", PARAMETERS)
def test_volume_limits_and_density(lulesh_gpu, parameters):
    """Both ends of the clamped volumes and a density other than 1 against
    the bit-identical build, within the reference's tolerance."""
    a, b = (blast(lulesh_gpu, 14, fused, parameters) for fused in (True, False))
    assert a.step(60, raise_on_error=False) == b.step(60, raise_on_error=False)
    v = b.get("vnew")
    if "eosvmax" in parameters:
        assert np.count_nonzero(v == parameters["eosvmax"]) > 0
    if "eosvmin" in parameters:
        assert np.count_nonzero(v == parameters["eosvmin"]) > 0
    for f in ("x", "xd", "e", "p", "q", "ql", "qq", "v", "vnew", "ss"):
        x, y = a.get(f), b.get(f)
        assert np.max(np.abs(x - y)) <= 1e-10 * np.max(np.abs(y)), f
    a.close()
    b.close()


@pytest.mark.parametrize("parameters", PARAMETERS)
def test_volume_limits_beyond_the_cache(lulesh_gpu, parameters):
    """The EOS after the sweep of kinematics and limiter against the separate
    kernels, bit for bit."""
    a, b = (blast(lulesh_gpu, 104, True, parameters) for _ in range(2))
    b.set_eos_bands(1)
    assert a.step(40, raise_on_error=False) == b.step(40, raise_on_error=False)
    v = b.get("vnew")
    for limit in ("eosvmax", "eosvmin"):
        if limit in parameters:
            assert np.count_nonzero(v == parameters[limit]) > 0
    for f in ("x", "xd", "e", "p", "q", "ql", "qq", "v", "vnew", "ss", "delv"):
        assert np.array_equal(a.get(f).view(np.uint64), b.get(f).view(np.uint64)), f
    a.close()
    b.close()
