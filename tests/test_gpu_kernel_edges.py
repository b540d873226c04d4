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


# the sweep of kinematics and limiter serves domains beyond the last-level
# cache: tiles of 16 x 16 columns, full, one column over and one short
@pytest.mark.parametrize("nx,mode,step,limit", [(104, 2, 3, None), (112, 1, 2, None),
                                                (113, 2, 35, None), (127, 2, 40, 33)])
def test_limiter_sweep_is_the_separate_kernels(lulesh_gpu, nx, mode, step, limit):
    """Bit for bit the fused step whose kinematics and limiter are separate
    kernels (the region-sorted schedule), in every field, also those that
    only a call's last cycle stores: a call that ends inside a replayed
    graph's length, past it, and at the cycle limit before its own end."""
    more = {} if limit is None else {"max_cycles": limit}
    a = lulesh_gpu.Domain(nx, ic_mode=mode, fused=True, **more)
    b = lulesh_gpu.Domain(nx, ic_mode=mode, fused=True, **more)
    b.set_eos_bands(1)
    assert a.step(step) == b.step(step)
    bad = [f for f in NODE + ELEM
           if not np.array_equal(a.get(f).view(np.uint64), b.get(f).view(np.uint64))]
    assert bad == []
    a.close()
    b.close()


# tiles in XCD order: fewer than eight, a multiple of eight and not; the last
# chunk of the columns whole and short
@pytest.mark.parametrize("nx,planes", [(1, 1), (5, 2), (31, 7), (61, 64), (62, 20)])
@pytest.mark.parametrize("mode", ["exact", "fused", "mixed"])
def test_planes_per_block_change_no_bits(lulesh_gpu, nx, planes, mode):
    """A domain swept with the planes per block of its own choice against
    one with the given number: each element's and each node's arithmetic is
    the same whichever block does it."""
    a = lulesh_gpu.Domain(nx, fused=mode == "fused", mixed=mode == "mixed")
    b = lulesh_gpu.Domain(nx, fused=mode == "fused", mixed=mode == "mixed")
    b.set_sweep_shape(32, 8, planes, 3 if mode == "mixed" else 2)
    assert a.step(20) == b.step(20)
    bad = [f for f in NODE + ELEM if not np.array_equal(a.get(f), b.get(f))]
    assert bad == []
    a.close()
    b.close()


# Q/EOS blocks of 64 elements up to 55^3, of 128 up to 70^3, of 256 beyond;
# the last block full (4^3, 64^3), partial and short
@pytest.mark.parametrize("nx", [4, 5, 55, 56, 57, 64, 70, 71])
@pytest.mark.parametrize("mode", ["exact", "fused", "mixed"])
def test_small_q_eos_blocks_change_no_bits(lulesh_gpu, nx, mode):
    """Against the region-sorted schedule, which shares no evaluations."""
    a = lulesh_gpu.Domain(nx, fused=mode == "fused", mixed=mode == "mixed")
    b = lulesh_gpu.Domain(nx, fused=mode == "fused", mixed=mode == "mixed")
    b.set_eos_bands(1)
    assert a.step(20) == b.step(20)
    bad = [f for f in NODE + ELEM if not np.array_equal(a.get(f), b.get(f))]
    assert bad == []
    sa, sb = a.stats(), b.stats()
    assert (sa.time, sa.dtcourant, sa.dthydro) == (sb.time, sb.dtcourant, sb.dthydro)
    a.close()
    b.close()


# one thread below 4 MB in all (8^3, 29^3), several beyond; fields of one slot
# (4 MB) and of more: the elements of 80^3 in one, its nodes in two
@pytest.mark.parametrize("nx,mode", [(1, "exact"), (8, "exact"), (29, "exact"), (37, "exact"),
                                     (80, "exact"), (128, "exact"), (8, "mixed"),
                                     (37, "mixed"), (101, "mixed"), (8, "mesh"),
                                     (37, "mesh"), (81, "mesh")])
def test_state_there_and_back(lulesh_gpu, oracle, nx, mode):
    """Every value of a state is found in its place, with the state and by
    field; values that float32 holds."""
    if mode == "mesh":
        d = lulesh_gpu.Domain.from_mesh(oracle.cube_mesh(nx), max_cycles=5)
    else:
        d = lulesh_gpu.Domain(nx, mixed=mode == "mixed")
    st = {"time": 0.25, "deltatime": 0.125}
    for t, f in enumerate(("x", "y", "z", "xd", "yd", "zd", "e", "p", "q", "v", "ss")):
        n = d.num_node if t < 6 else d.num_elem
        st[f] = np.arange(n, dtype=np.float64) + 7 * t
    d.upload_state(st)
    back = d.download_state()
    assert all(np.array_equal(back[f], st[f]) for f in st)
    for f in ("z", "ss"):
        assert np.array_equal(d.get(f), st[f])
        d.set(f, st[f][::-1].copy())
        assert np.array_equal(d.get(f), st[f][::-1])
    d.close()


# 75^3 beside the others: chunks of 256 elements; without it 64.  Planes per
# tile follow the members left, to the last one alone.
@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("sizes", [[75, 30, 5], [31, 12, 44, 1, 16]])
def test_ensemble_cut_anew_as_members_stop(lulesh_gpu, sizes, fused):
    """Members of a default ensemble against runs of their own, bit for bit."""
    b = lulesh_gpu.Batch(sizes, fused=fused)
    b.run()
    for m, nx in enumerate(sizes):
        d = lulesh_gpu.Domain(nx, fused=fused)
        rc, cycles = d.run()
        assert b.stats(m)[0] == rc and b.stats(m)[1].cycle == cycles
        bad = [f for f in NODE + ELEM[:10] if not np.array_equal(
            b.get(m, f).view(np.uint64), d.get(f).view(np.uint64))]
        assert bad == []
        d.close()
    b.close()


# element blocks of at most 512: one, one and a bit, and several on each XCD
@pytest.mark.parametrize("nx,cycles", [(1, 8), (2, 20), (8, 20), (9, 20), (17, 40), (33, 20)])
@pytest.mark.parametrize("fused", [False, True])
def test_mesh_forces_by_blocks(lulesh_gpu, oracle, nx, cycles, fused):
    """A cube given as lists against the cube itself with the same initial
    conditions: the same bits, fused within the reference's tolerance."""
    a = lulesh_gpu.Domain.from_mesh(oracle.cube_mesh(nx), fused=fused)
    b = lulesh_gpu.Domain(nx, ic_mode=1)
    assert a.step(cycles) == b.step(cycles)
    for f in NODE + ELEM[:11]:
        x, y = a.get(f), b.get(f)
        if fused:
            assert np.max(np.abs(x - y)) <= 1e-10 * np.max(np.abs(y)), f
        else:
            assert np.array_equal(x.view(np.uint64), y.view(np.uint64)), f
    a.close()
    b.close()


# tiles of 16 x 8 columns own 15 x 7 nodes: one tile, its edge, several; 33^3
# the largest in one round, 34^3 swept
@pytest.mark.parametrize("nx,mode,hgcoef", [(1, 2, None), (2, 1, None), (6, 2, None),
                                            (7, 2, 0.0), (14, 2, None), (15, 1, None),
                                            (16, 2, None), (30, 2, None), (33, 2, None),
                                            (33, 1, 0.0), (34, 2, None)])
def test_plane_blocks_are_the_sweep(lulesh_gpu, nx, mode, hgcoef):
    """The forces of a small domain by blocks of one node plane, bit for bit
    the sweep's, with and without hourglass forces."""
    a = lulesh_gpu.Domain(nx, ic_mode=mode)
    b = lulesh_gpu.Domain(nx, ic_mode=mode)
    b.set_sweep_shape(32, 8, 4, 2)
    if hgcoef is not None:
        a.set_parameter("hgcoef", hgcoef)
        b.set_parameter("hgcoef", hgcoef)
    ra, rb = a.step(37, raise_on_error=False), b.step(37, raise_on_error=False)
    assert ra == rb
    bad = [f for f in NODE + ELEM
           if not np.array_equal(a.get(f).view(np.uint64), b.get(f).view(np.uint64))]
    assert bad == []
    a.close()
    b.close()


# 36^3 the largest whose repetitions are shared, 37^3 one wave per block
@pytest.mark.parametrize("nx", [1, 4, 5, 36, 37])
@pytest.mark.parametrize("form", [0, 1])
@pytest.mark.parametrize("fused", [False, True])
def test_learned_q_outside_its_range_is_the_limiter(lulesh_gpu, nx, form, fused):
    """With no input in the network's range every element keeps the plain
    limiter: the plain step, bit for bit, in the learned Q kernels."""
    import learned_q
    net, _ = learned_q.load(learned_q.NET_FILE if form == 0 else learned_q.NET_FILE_STANDIN)
    a = lulesh_gpu.Domain(nx, fused=fused)
    b = lulesh_gpu.Domain(nx, fused=fused)
    b.set_learned_q(net, 1e-30, form=form)
    assert a.step(20) == b.step(20)
    bad = [f for f in NODE + ELEM if not np.array_equal(a.get(f), b.get(f))]
    assert bad == []
    sa, sb = a.stats(), b.stats()
    assert (sa.time, sa.dtcourant, sa.dthydro) == (sb.time, sb.dtcourant, sb.dthydro)
    a.close()
    b.close()
