"""State transfers on both sides of the sizes where their route changes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("x", "y", "z", "xd", "yd", "zd", "e", "p", "q", "v", "ss")


# the largest field below and above 16 KB, the state below and above 10 MB
@pytest.mark.parametrize("nx", [11, 12, 48, 49])
@pytest.mark.parametrize("shared", [False, True])
def test_state_there_and_back(lulesh_gpu, nx, shared):
    d = lulesh_gpu.Domain(nx)
    rng = np.random.default_rng(nx)
    st = {f: rng.standard_normal(d.num_node if t < 6 else d.num_elem)
          for t, f in enumerate(FIELDS)}
    if shared:  # one array for several fields
        st["yd"] = st["zd"] = st["xd"]
        st["p"] = st["e"]
    st.update(time=0.25, deltatime=0.125)
    d.upload_state(st)
    back = d.download_state()
    assert all(np.array_equal(back[f], st[f]) for f in st)
    d.close()
