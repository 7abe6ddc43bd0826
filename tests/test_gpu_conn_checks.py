"""Connectivity on the device against the oracle where its sweeps end early or
not, and where the face check has to find a broken face from either side."""
import numpy as np
import pytest

from parrsb_amd import meshgen as M

pytestmark = pytest.mark.gpu


def _both(oracle, xyz, ndim, tol=0.2):
    import parrsb_amd as pa
    rc, ref = oracle.conn_mesh(xyz, ndim, tol)
    try:
        ids = pa.conn_mesh(xyz, ndim, tol)
        return rc, ref, 0, ids
    except pa.ParrsbError as e:
        return rc, ref, e.rc, None


@pytest.mark.parametrize("corner", range(8))
@pytest.mark.parametrize("elem", [0, 13, 26])
def test_broken_face_is_found(oracle, elem, corner, monkeypatch):
    """One corner of a first, inner or last element moves away from its
    vertex: every face at it is left with three common corners."""
    monkeypatch.setenv("PARRSB_VERBOSE_LEVEL", "0")
    vtx, xyz, nv = M.box_hex(3, 3, 3, jitter=0.0)
    x = xyz.copy()
    x[elem, corner] += 0.4 / 3
    print("conn", elem, corner, flush=True)
    rc, ref, rd, ids = _both(oracle, x, 3)
    assert rd == rc
    if rc == 0:
        assert np.array_equal(ids.ravel(), np.asarray(ref).ravel())


@pytest.mark.parametrize("order", ["lattice", "shuffled"])
@pytest.mark.parametrize("name", ["one", "box", "skew", "noise", "quads"])
def test_sweeps(oracle, name, order, monkeypatch):
    """skew: planes of one axis overlap along it, so points separate only in a
    later sweep; noise: corners of a vertex apart by a tenth of the limit."""
    monkeypatch.setenv("PARRSB_VERBOSE_LEVEL", "0")
    rng = np.random.default_rng(3)
    ndim = 3
    if name == "one":
        xyz = M.box_hex(1, 1, 1, jitter=0.0)[1]
    elif name == "box":
        xyz = M.box_hex(9, 7, 5, jitter=0.0)[1]
    elif name == "skew":
        xyz = M.box_hex(7, 6, 5, jitter=0.0)[1]
        xyz[..., 0] += 0.37 * xyz[..., 1] + 0.19 * xyz[..., 2]
    elif name == "noise":
        xyz = M.box_hex(8, 8, 8, jitter=0.0)[1]
        xyz += rng.uniform(-0.01 / 8, 0.01 / 8, size=xyz.shape)
    else:
        xyz, ndim = M.holed_quads(40, 30, seed=2, rmax=5.0)[1], 2
    if order == "shuffled":
        xyz = xyz[rng.permutation(xyz.shape[0])]
    print("conn", name, order, flush=True)
    rc, ref, rd, ids = _both(oracle, xyz, ndim)
    assert rd == rc
    if rc == 0:
        assert np.array_equal(ids.ravel(), np.asarray(ref).ravel())
