"""The kernels at the sizes where their work is cut: tiles and planes of the
sweeps, blocks of the Q/EOS kernel and their shares of the EOS repetitions.

The bit-identical build against the oracle, bit for bit; the build with fused
multiply-adds within the reference's tolerance, 1e-10 of each field's
max-norm (tests/test_gpu_fused.py)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NODE = ("x", "y", "z", "xd", "yd", "zd")
ELEM = ("e", "p", "q", "ql", "qq", "v", "vnew", "delv", "vdov", "arealg", "ss",
        "delv_xi", "delv_eta", "delv_zeta", "delx_xi", "delx_eta", "delx_zeta")
ORACLE = tuple(f for f in NODE + ELEM if f not in ("vnew",))


def differing(dom, orc):
    return [f for f in ORACLE if not np.array_equal(dom.get(f).view(np.uint64),
                                                    orc.get(f).view(np.uint64))]


# 6^3: less than one Q/EOS block; 7^3, 8^3: a partial and a full last one
@pytest.mark.parametrize("nx", [1, 6, 7, 8])
@pytest.mark.parametrize("num_reg,cost", [(1, 0), (1, 3), (5, 0), (11, 1), (21, 30)])
def test_repetitions_shared_over_a_block(lulesh_gpu, oracle, nx, num_reg, cost):
    """Elements with none, light and heavy counts of extra EOS evaluations,
    one class or both present, against the oracle bit for bit."""
    d = lulesh_gpu.Domain(nx, num_reg=num_reg, cost=cost, max_cycles=12)
    o = oracle.Oracle(nx, num_reg=num_reg, cost=cost, cbrt_mode=1, threads=4)
    rc, n = d.step(12, raise_on_error=False)
    assert rc == o.run(12)
    assert n == o.cycle
    assert differing(d, o) == []
    d.close()


# one tile owns 31 x 7 nodes of the 32 x 8 shape; 36: two planes per block
@pytest.mark.parametrize("nx,mode", [(1, 1), (2, 2), (6, 2), (7, 2), (29, 1), (30, 2),
                                     (31, 2), (36, 2), (61, 2), (62, 1)])
def test_fused_step_at_tile_edges(lulesh_gpu, nx, mode):
    """The fused step and the bit-identical one of the same domain agree on
    every field within the reference's tolerance."""
    a = lulesh_gpu.Domain(nx, ic_mode=mode)
    b = lulesh_gpu.Domain(nx, ic_mode=mode, fused=True)
    ra, rb = a.step(37, raise_on_error=False), b.step(37, raise_on_error=False)
    assert ra == rb
    for f in NODE + ELEM:
        x, y = a.get(f), b.get(f)
        s = np.max(np.abs(x))
        assert np.max(np.abs(x - y)) <= 1e-10 * s, f
    a.close()
    b.close()
