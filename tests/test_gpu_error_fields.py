"""What an error inside a call leaves of the intermediate fields where the
fused step's kinematics and limiter are one sweep (domains beyond the
last-level cache): the values of the last cycle whose kinematics ran, as from
the separate kernels (the region-sorted schedule), which store them in every
cycle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NX = 104  # the sweep serves domains from 102^3 on
FIELDS = ("delv", "delv_xi", "delv_eta", "delv_zeta", "delx_xi", "delx_eta", "delx_zeta",
          "vdov", "arealg")


def pair(lulesh_gpu):
    a = lulesh_gpu.Domain(NX, fused=True)
    b = lulesh_gpu.Domain(NX, fused=True)
    b.set_eos_bands(1)
    return a, b


def differing(a, b):
    return [f for f in FIELDS
            if not np.array_equal(a.get(f).view(np.uint64), b.get(f).view(np.uint64))]


# 20 cycles queued one by one, 40 of which a replayed graph holds 32
@pytest.mark.parametrize("step", [20, 40])
def test_q_stop_inside_a_call(lulesh_gpu, step):
    """An error of the EOS: the gradients of the failed cycle."""
    a, b = pair(lulesh_gpu)
    a.step(4)
    b.step(4)
    # the largest q passes it three cycles on (it grows up to the 14th cycle,
    # to 2.6 times this), and the cycle after that stops
    limit = 1.5 * float(np.max(a.get("q")))
    got = []
    for d in (a, b):
        d.set_parameter("qstop", limit)
        got.append(d.step(step, raise_on_error=False))
    assert got[0] == got[1] and got[0][0] == lulesh_gpu.QSTOP_ERROR
    assert 2 <= got[0][1] < min(step, 32)  # inside the call, and inside its graph
    assert differing(a, b) == []
    a.close()
    b.close()


def set_fold(d):
    """Constant velocities that fold one element: its xi edges shrink through
    nothing while its twist keeps the volume, so that the Jacobian at its
    centre turns over first."""
    en, h, cycles = NX + 1, 1.125 / NX, 10.5
    st = d.download_state()
    rng = np.random.default_rng(1)
    for f in ("xd", "yd", "zd"):
        st[f] = rng.uniform(-1e-3, 1e-3, d.num_node) * h / 1e-7
    st["e"] = np.zeros(d.num_elem)
    st["deltatime"] = 1e-7
    v = {f: st[f].reshape(en, en, en) for f in ("xd", "yd", "zd")}
    c = NX // 2
    for s3 in (-1, 1):
        for s2 in (-1, 1):
            for s1 in (-1, 1):
                at = (c + (s3 > 0), c + (s2 > 0), c + (s1 > 0))
                v["xd"][at] += (-0.5 * s1 + 0.25 * s1 * s2) * h / (cycles * 1e-7)
                v["zd"][at] += 0.25 * s2 * s3 * h / (cycles * 1e-7)
    d.set_parameter("dtfixed", 1e-7)
    for name in ("qlc_monoq", "qqc_monoq", "hgcoef"):
        d.set_parameter(name, 0.0)
    d.upload_state(st)


@pytest.mark.parametrize("step", [20, 40])
def test_jacobian_turned_over_inside_a_call(lulesh_gpu, step):
    """An error of the force sweep: the gradients of the cycle before, whose
    nodes are in the other copy."""
    a, b = pair(lulesh_gpu)
    got = []
    for d in (a, b):
        set_fold(d)
        got.append(d.step(step, raise_on_error=False))
    assert got[0] == got[1] and got[0][0] == lulesh_gpu.VOLUME_ERROR
    assert 8 <= got[0][1] <= 16
    # no volume turned over: it was the sweep's error, in the last cycle
    assert np.min(b.get("vnew")) > 0.0
    for f in ("x", "v", "vnew", "ql", "qq"):
        assert np.array_equal(a.get(f).view(np.uint64), b.get(f).view(np.uint64))
    assert differing(a, b) == []
    # an error in a call's first cycle leaves what the calls before left
    for d in (a, b):
        d.upload_state({**{f: d.get(f) for f in ("x", "y", "z", "xd", "yd", "zd", "e", "p", "q",
                                                 "v", "ss")}, "time": 0.0, "deltatime": 1e-7})
        assert d.step(1, raise_on_error=False)[0] == lulesh_gpu.VOLUME_ERROR
    assert differing(a, b) == []
    a.close()
    b.close()


def test_volume_turned_over_inside_a_call(lulesh_gpu):
    """An error of the kinematics, in the sweep that limits as well: the same
    code in the same cycle as from the separate kernels."""
    en, h, cycles = NX + 1, 1.125 / NX, 6.5
    a, b = pair(lulesh_gpu)
    got = []
    for d in (a, b):
        st = d.download_state()
        xd = np.zeros((en, en, en))
        xd[:, :, NX // 2] = h / (cycles * 1e-7)  # a node plane overtakes the next
        st.update(xd=xd.ravel(), e=np.zeros(d.num_elem), deltatime=1e-7)
        d.set_parameter("dtfixed", 1e-7)
        for name in ("qlc_monoq", "qqc_monoq", "hgcoef"):
            d.set_parameter(name, 0.0)
        d.upload_state(st)
        got.append(d.step(20, raise_on_error=False))
    assert got == [(lulesh_gpu.VOLUME_ERROR, 7)] * 2
    for f in ("x", "xd", "e", "p", "q", "v", "ss"):
        assert np.array_equal(a.get(f).view(np.uint64), b.get(f).view(np.uint64)), f
    a.close()
    b.close()
