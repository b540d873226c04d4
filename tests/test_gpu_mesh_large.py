"""Meshes of more than 2^20 elements, whose blocks run in launch order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fused", [False, True])
def test_mesh_beyond_a_million_elements(lulesh_gpu, oracle, fused):
    """A cube given as lists against the cube itself: the same bits, fused
    within the reference's tolerance."""
    nx = 102
    assert nx ** 3 > 1 << 20
    a = lulesh_gpu.Domain.from_mesh(oracle.cube_mesh(nx), fused=fused)
    b = lulesh_gpu.Domain(nx, ic_mode=1)
    assert a.step(12) == b.step(12)
    for f in ("x", "y", "z", "xd", "yd", "zd", "e", "p", "q", "ql", "qq", "v", "vnew", "ss"):
        x, y = a.get(f), b.get(f)
        if fused:
            assert np.max(np.abs(x - y)) <= 1e-10 * np.max(np.abs(y)), f
        else:
            assert np.array_equal(x.view(np.uint64), y.view(np.uint64)), f
    a.close()
    b.close()
