"""Blocks of closed handles are reused by later ones: results do not depend on
what a block held before, on its size class, or on which thread asks."""
import threading

import numpy as np
import pytest

from parrsb_amd import meshgen as M

pytestmark = pytest.mark.gpu


def _part(mesh, P):
    import parrsb_amd as pa
    vtx, xyz, nv = mesh
    b = vtx.shape[0]
    with pa.Device() as d:
        d.set_mesh(vtx, xyz, nv)
        d.set_segments([0], [b], [P], [0])
        d.prepartition(1)
        d.level_laplacian()
        out = d.fiedler(1, precision=64)
        d.fiedler_sort()
        return d.order(), out["lambda"].copy()


MESHES = [lambda: M.box_hex(5, 4, 3), lambda: M.box_hex(20, 18, 16, jitter=0.1, seed=2),
          lambda: M.quad_grid(70, 50), lambda: M.warped_box_hex(22, seed=6)]


def test_reused_blocks_give_the_same_results():
    meshes = [m() for m in MESHES]
    first = [_part(m, 4) for m in meshes]
    # every order of sizes, more closes than the pool keeps idle blocks for
    for k in range(24):
        i = (7 * k + k // 4) % len(meshes)
        o, lam = _part(meshes[i], 4)
        assert np.array_equal(o, first[i][0]) and np.array_equal(lam, first[i][1]), (k, i)


def test_threads_share_the_pool():
    meshes = [m() for m in MESHES]
    first = [_part(m, 4) for m in meshes]
    bad = []

    def work(i):
        for _ in range(4):
            o, lam = _part(meshes[i], 4)
            if not (np.array_equal(o, first[i][0]) and np.array_equal(lam, first[i][1])):
                bad.append(i)

    ts = [threading.Thread(target=work, args=(i,)) for i in range(len(meshes))]
    for t in ts:
        t.start()
    for t in ts:
        t.join(100)
    assert not bad and not any(t.is_alive() for t in ts)


def test_memory_left_by_a_call_goes_back(monkeypatch):
    """After the last close the device gets everything back on request, and
    with a bound of 0 at once."""
    import parrsb_amd as pa
    mesh = MESHES[1]()
    before = pa.device_memory()[0]
    first = _part(mesh, 4)
    live, idle, peak = pa.device_memory()
    assert live == before and 0 < idle <= 4 << 30 and peak >= live + idle
    assert pa.release_memory() == idle
    assert pa.device_memory() == (live, 0, live) and pa.release_memory() == 0
    monkeypatch.setenv("PARRSB_AMD_POOL_MB", "0")
    o, lam = _part(mesh, 4)
    assert np.array_equal(o, first[0]) and np.array_equal(lam, first[1])
    assert pa.device_memory()[:2] == (live, 0)
