"""Calls that run short of device memory (PARRSB_AMD_MEM_LIMIT_MB): they
succeed wherever their buffers fit at the sizes they need, fail with 2
otherwise, and leave nothing behind that a later call could trip over."""
import numpy as np
import pytest

from parrsb_amd import meshgen as M

pytestmark = pytest.mark.gpu


def _peak(call):
    """Most device memory of a call that starts from an empty pool."""
    import parrsb_amd as pa
    pa.release_memory()
    live = pa.device_memory()[0]
    out = call()
    peak = pa.device_memory()[2]
    pa.release_memory()
    return out, peak - live


@pytest.mark.parametrize("opt", [dict(), dict(rsb_algo=1), dict(partitioner=1)])
def test_calls_short_of_memory(opt, monkeypatch):
    import parrsb_amd as pa
    vtx, xyz, nv = M.box_hex(30, 25, 20, jitter=0.1, seed=4)

    def call():
        return pa.part_mesh(vtx, xyz, nv, 12, **opt)[0]
    ref, peak = _peak(call)
    mb = peak >> 20
    done = 0
    for limit in sorted({1, 2, *range(3, mb + 2, max(1, mb // 24)), mb + 1}):
        print("limit", opt, limit, "of", mb, flush=True)
        live = pa.device_memory()[0] >> 20
        monkeypatch.setenv("PARRSB_AMD_MEM_LIMIT_MB", str(limit + live))
        try:
            got = call()
            done += 1
            assert np.array_equal(got, ref)
        except pa.ParrsbError as e:
            assert e.rc == 2
        monkeypatch.delenv("PARRSB_AMD_MEM_LIMIT_MB")
        assert np.array_equal(call(), ref)
        pa.release_memory()
    assert done >= 1


def test_room_to_grow_is_not_needed(monkeypatch):
    """A handle whose level buffers grow: with the memory for one level at its
    exact sizes and not an eighth more, the next, larger level still runs."""
    import parrsb_amd as pa
    vtx, xyz, nv = M.box_hex(64, 64, 32, jitter=0.1, seed=6)
    n = vtx.shape[0]

    def call(two):
        with pa.Device() as d:
            d.set_mesh(vtx, xyz, nv)
            for cut in ([0, n // 2], [0]) if two else ([0],):
                # the first level solves one half only, so the second is larger
                d.set_segments(cut, np.diff(cut + [n]), [2] + [1] * (len(cut) - 1),
                               [0, 2][:len(cut)])
                d.prepartition(1)
                d.level_laplacian()
                out = d.fiedler(len(cut), precision=64, max_passes=1)
            return out["lambda"][0]
    one, peak1 = _peak(lambda: call(False))
    two, peak2 = _peak(lambda: call(True))
    assert one == pytest.approx(two, rel=1e-6)
    # what the second level needs beside the first one's retired buffers
    limit = (peak1 >> 20) + 40
    print("room", peak1 >> 20, peak2 >> 20, limit, flush=True)
    assert limit << 20 < peak2
    live = pa.device_memory()[0] >> 20
    monkeypatch.setenv("PARRSB_AMD_MEM_LIMIT_MB", str(limit + live))
    assert call(True) == two


def test_graph_build_gives_its_sort_arrays_back_before_the_graph(monkeypatch):
    """Most bytes per corner of a quality report, when the rows are counted:
    keys, slots, flags and offsets of the sort 20, its output and scratch 24,
    groups 5, row lengths and offsets 2, centroids and ranks 4.5, in blocks up
    to an eighth larger: at most 62.5.  The graph's entries (13) come after
    the first 16 of them have gone; beside them it would be 68.5 at least."""
    import parrsb_amd as pa
    vtx, _, nv = M.box_hex(64, 64, 64, jitter=0.0)
    n = vtx.shape[0]
    monkeypatch.setenv("PARRSB_AMD_POOL_MB", "0")
    with pa.Device() as d:
        dv = d.upload(np.ascontiguousarray(vtx))
        dp = d.upload(np.arange(n, dtype=np.int32) * 8 // n)
    q, peak = _peak(lambda: pa.quality_dev(dp, dv, n, nv, 8))
    pa.Device.free(dv), pa.Device.free(dp)
    print("bytes per corner", peak / vtx.size, flush=True)
    assert q["components"] == 8
    assert peak < 64 * vtx.size
