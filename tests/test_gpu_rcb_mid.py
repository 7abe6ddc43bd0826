"""RCB orders where the middle kernel takes over from the global rounds and
hands on to the tail, against the global rounds alone."""
import numpy as np
import pytest

from parrsb_amd import meshgen as M

pytestmark = pytest.mark.gpu


def _order(vtx, xyz, nv, bounds, parts):
    import parrsb_amd as pa
    b, p = np.asarray(bounds), np.asarray(parts)
    with pa.Device() as d:
        d.set_mesh(vtx, xyz, nv)
        d.set_segments(b[:-1], np.diff(b), p, np.r_[0, np.cumsum(p)[:-1]])
        d.prepartition(1)
        return d.order()


@pytest.mark.parametrize("parts", [2, 3, 7, 64, 1500])
@pytest.mark.parametrize("n", [1024, 1025, 2049, 8191, 8192, 8193, 16400, 20000])
def test_mid_kernel_equals_global_rounds(n, parts, monkeypatch):
    """Sizes either side of both kernels' limits; a lattice, so that many
    ranks are equal and the order among them is the stable sort's."""
    print("rcb", n, parts, flush=True)
    vtx, xyz, nv = M.box_hex(28, 28, 28, jitter=0.0)
    vtx, xyz = vtx[:n], xyz[:n]
    got = _order(vtx, xyz, nv, [0, n], [parts])
    monkeypatch.setenv("PARRSB_AMD_RCB_TAIL", "0")
    assert np.array_equal(got, _order(vtx, xyz, nv, [0, n], [parts]))


@pytest.mark.parametrize("mesh", ["hex", "quads"])
def test_several_segments(mesh, monkeypatch):
    """Segments that need global rounds, the middle kernel, the tail alone and
    nothing, one of them with more ranks than elements."""
    vtx, xyz, nv = (M.box_hex(33, 30, 29, jitter=0.1, seed=3) if mesh == "hex"
                    else M.holed_quads(190, 180, seed=5))
    n = vtx.shape[0]
    for parts in ([4, 3, 1, 2, 9, 5], [4, 3, 1, 2, 9, 2]):
        b = [0, 11000, 11003 if parts[-1] == 5 else 19000, 19001, 20000, 27000, n]
        print("rcb segments", mesh, parts, flush=True)
        monkeypatch.delenv("PARRSB_AMD_RCB_TAIL", raising=False)
        got = _order(vtx, xyz, nv, b, parts)
        monkeypatch.setenv("PARRSB_AMD_RCB_TAIL", "0")
        assert np.array_equal(got, _order(vtx, xyz, nv, b, parts))
