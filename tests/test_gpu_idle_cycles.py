"""Cycles queued past the end of a run: their kernels may load, and change
nothing."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("x", "y", "z", "xd", "yd", "zd", "e", "p", "q", "ql", "qq", "v", "vnew", "ss",
          "delv", "delv_xi", "delx_zeta", "vdov", "arealg")


@pytest.mark.parametrize("kind,fused", [("mesh", False), ("mesh", True), ("cube", False),
                                        ("cube", True), ("mixed", False)])
def test_cycles_past_the_end(lulesh_gpu, oracle, kind, fused):
    """Also on a state that would be an error if they ran."""
    if kind == "mesh":
        d = lulesh_gpu.Domain.from_mesh(oracle.cube_mesh(9), max_cycles=7, fused=fused)
    else:
        d = lulesh_gpu.Domain(9, max_cycles=7, fused=fused, mixed=kind == "mixed")
    assert d.step(40) == (0, 7)
    x = d.get("x")
    d.set("x", -x)  # every volume below 0
    before = {f: d.get(f) for f in FIELDS}
    for n in (1, 3, 40):
        assert d.step(n) == (0, 0)
    for f in FIELDS:
        assert np.array_equal(d.get(f).view(np.uint64), before[f].view(np.uint64)), f
    s = d.stats()
    assert s.cycle == 7 and s.done == 1
    d.close()
