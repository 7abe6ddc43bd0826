"""Connectivity on the device against the oracle where its sweeps end early or
not, and where the face check has to find a broken face from either side."""
import time

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


@pytest.mark.parametrize("spokes", [63, 64, 65, 130])
def test_vertices_of_many_elements(oracle, spokes, monkeypatch):
    """A wheel of quads: its hub is shared by `spokes` elements, either side of
    the longest list that the end of the sweeps looks through."""
    monkeypatch.setenv("PARRSB_VERBOSE_LEVEL", "0")
    t = np.arange(2 * spokes) * np.pi / spokes
    rim = np.stack([np.cos(t), np.sin(t)], 1)
    k = 2 * np.arange(spokes)
    # preprocessor order: hub, rim, rim, rim around the element
    xyz = np.stack([np.zeros((spokes, 2)), rim[k], rim[k + 1], rim[(k + 2) % (2 * spokes)]], 1)
    print("conn wheel", spokes, flush=True)
    rc, ref, rd, ids = _both(oracle, xyz, 2, 1e-3)
    assert rd == rc
    if rc == 0:
        assert np.array_equal(ids.ravel(), np.asarray(ref).ravel())


def test_points_that_stay_together_cost_no_serial_walk(monkeypatch):
    """On a warped mesh no coordinate separates the points, so all sweeps run
    over one long segment: about three times a lattice that one sweep takes
    apart (1.0 ms; with one thread's walk over 4,096 points after each of two
    sweeps it was 7.4)."""
    import parrsb_amd as pa
    monkeypatch.setenv("PARRSB_VERBOSE_LEVEL", "0")
    took = {}
    for name, xyz, rc in (("lattice", M.box_hex(24, 24, 24, jitter=0.0)[1], 0),
                          ("warped", M.warped_box_hex(24, seed=3)[1], 1)):
        print("conn time", name, flush=True)
        n, nv = xyz.shape[:2]
        with pa.Device() as d:
            dx = d.upload(np.ascontiguousarray(xyz))
            dv = d.upload(np.zeros((n, nv), dtype=np.int64))
            for _ in range(5):
                t0 = time.perf_counter()
                assert pa.lib().parrsb_amd_conn_mesh_dev(dv, dx, n, 3, 0.2) == rc
                took[name] = min(took.get(name, 1.0), time.perf_counter() - t0)
            pa.Device.free(dx), pa.Device.free(dv)
    assert took["warped"] < 5 * took["lattice"], took
