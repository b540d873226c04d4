"""The fused sweep with two and three planes per block, the last chunk of the
37 planes shorter or not."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,planes", [(36, 2), (36, 3), (35, 2), (35, 3)])
def test_fused_sweep_in_chunks(lulesh_gpu, nx, planes):
    a = lulesh_gpu.Domain(nx, fused=True)
    a.set_sweep_shape(32, 8, planes, 2)
    b = lulesh_gpu.Domain(nx)
    assert a.step(37) == b.step(37)
    for f in ("x", "y", "z", "xd", "yd", "zd", "e", "p", "q", "v", "ss", "delv_zeta"):
        x, y = a.get(f), b.get(f)
        assert np.max(np.abs(x - y)) <= 1e-10 * np.max(np.abs(y)), f
    a.close()
    b.close()
