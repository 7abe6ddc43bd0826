"""Level kernels at the sizes where their forms change: LDS sorts, LDS sets of
neighbouring segments, 32- and 64-bit quality keys."""
import time

import numpy as np
import pytest

from parrsb_amd import meshgen as M

pytestmark = pytest.mark.gpu


def _dev():
    import parrsb_amd as pa
    return pa.Device()


@pytest.mark.parametrize("n", [1, 2, 2047, 2048, 2049, 8191, 8192, 8193, 9000])
def test_fiedler_sort_is_the_stable_sort(n):
    """Values with many ties, both zeros, infinities; a second segment with
    one rank keeps its order."""
    print("fsort", n, flush=True)
    vtx, xyz, nv = M.box_hex(24, 24, 24, jitter=0.0)
    vtx, xyz = vtx[:n + 50], xyz[:n + 50]
    rng = np.random.default_rng(n)
    f = rng.integers(-20, 20, n + 50) * 0.125
    f[rng.random(n + 50) < 0.1] = -0.0
    f[rng.random(n + 50) < 0.01] = np.inf
    f[rng.random(n + 50) < 0.01] = -np.inf
    with _dev() as d:
        d.set_mesh(vtx, xyz, nv)
        d.set_segments([0, n], [n, 50], [2, 1], [0, 2])
        d.set_fiedler_values(f)
        d.fiedler_sort()
        o, g = d.order(), d.fiedler_values()
    want = np.r_[np.argsort(f[:n], kind="stable"), np.arange(n, n + 50)]
    assert np.array_equal(o, want) and np.array_equal(g, f[want])


@pytest.mark.parametrize("size", [1, 2, 25, 26, 40])
def test_fiedler_sort_of_many_small_segments(size):
    """Segments so small that a workgroup each takes longer than device-wide
    sorts: the stable order on both sides of the rule (65,536 elements: LDS
    from 26 elements a segment on), and no more than a few times one large
    segment's time for segments of one element, where a workgroup each took
    2.3 ms of device time against 0.1."""
    print("fsort small", size, flush=True)
    vtx, xyz, nv = M.box_hex(32, 32, 64, jitter=0.0)
    rng = np.random.default_rng(size)
    f = rng.integers(-3, 3, vtx.shape[0]) * 0.25
    took = {}
    with _dev() as d:
        d.set_mesh(vtx, xyz, nv)
        n = vtx.shape[0]
        for ln in (size, n):
            start = np.arange(0, n, ln)
            cnt = np.minimum(ln, n - start)
            for _ in range(4):
                d.set_segments(start, cnt, np.full(start.size, 2), 2 * np.arange(start.size))
                d.set_fiedler_values(f)
                at = d.order()  # the elements' own order; also waits
                t0 = time.perf_counter()
                d.fiedler_sort()
                got = d.order()
                took[ln] = min(took.get(ln, 1.0), time.perf_counter() - t0)
            want = np.concatenate([b + np.argsort(f[b:b + c], kind="stable")
                                   for b, c in zip(start, cnt)])
            assert np.array_equal(got, at[want])
    if size == 1:
        assert took[size] < 6 * took[n], took


def _sort_large(n, cuts):
    """Fiedler sort of n elements in segments too large for LDS: checks the
    stable order, returns the least time of four."""
    vtx, xyz, nv = M.box_hex(128, 64, n // 8192 + 1, jitter=0.0)
    vtx, xyz = vtx[:n], xyz[:n]
    f = np.random.default_rng(n).integers(-20000, 20000, n) * 0.125
    cnt, took = np.diff(cuts + [n]), 1.0
    with _dev() as d:
        d.set_mesh(vtx, xyz, nv)
        for _ in range(4):
            d.set_segments(cuts, cnt, [2] * len(cuts), 2 * np.arange(len(cuts)))
            d.set_fiedler_values(f)
            at = d.order()
            t0 = time.perf_counter()
            d.fiedler_sort()  # waits
            took = min(took, time.perf_counter() - t0)
        want = np.concatenate([b + np.argsort(f[b:b + c], kind="stable")
                               for b, c in zip(cuts, cnt)])
        assert np.array_equal(d.order(), at[want])
    return took


@pytest.mark.parametrize("n", [262144, 262145, 1048576, 1048577])
def test_device_wide_sorts_either_side_of_their_forms(n):
    """64-bit values merge up to 2^20 elements, segment numbers up to 2^18."""
    print("fsort large", n, flush=True)
    _sort_large(n, [0, n // 3, n // 2])


def test_device_wide_sort_times_do_not_jump():
    """100,000 elements against 65,000: the onesweep form takes 235 us there,
    the merge sort 90 (85 for 65,000)."""
    print("fsort times", flush=True)
    took = {n: _sort_large(n, [0]) for n in (65000, 100000)}
    assert took[100000] < 1.8 * took[65000], took


@pytest.mark.parametrize("size", [1, 3, 40, 700])
def test_neighbour_counts_of_small_segments(size):
    """Segments of one to a few elements: a workgroup's set of pairs overflows
    its LDS, and the common set has to grow."""
    print("neighbours", size, flush=True)
    vtx, xyz, nv = M.box_hex(17, 16, 15, jitter=0.0)
    n = vtx.shape[0]
    start = np.arange(0, n, size)
    ln = np.minimum(size, n - start)
    with _dev() as d:
        d.set_mesh(vtx, xyz, nv)
        d.set_segments(start, ln, np.ones_like(start), np.arange(start.size))
        got = d.neighbors(start.size)
        rowptr, col, _ = d.graph()
    seg = np.arange(n) // size
    pairs = np.stack([np.repeat(seg, np.diff(rowptr)), seg[col]], 1)
    pairs = np.unique(pairs[pairs[:, 0] != pairs[:, 1]], axis=0)
    assert np.array_equal(got, np.bincount(pairs[:, 0], minlength=start.size))


@pytest.mark.parametrize("mesh", ["apart", "box"])
def test_neighbour_counts_of_a_segment_per_element(mesh):
    """300,000 elements that share nothing, and a box whose 18.6M pairs do not
    fit the set's first size: a set of at most 128 MiB to begin with, doubled
    once for the box."""
    import parrsb_amd as pa
    print("neighbours", mesh, flush=True)
    if mesh == "apart":
        n, nv = 300000, 4
        vtx = np.arange(1, 4 * n + 1, dtype=np.int64).reshape(n, nv)
        xyz = np.zeros((n, nv, 2))
    else:
        vtx, xyz, nv = M.box_hex(90, 90, 90, jitter=0.0)
        n = vtx.shape[0]
    pa.release_memory()
    with _dev() as d:
        d.set_mesh(vtx, xyz, nv)
        e = np.arange(n)
        d.set_segments(e, np.ones_like(e), np.ones_like(e), e)
        live = pa.device_memory()[0]
        got = d.neighbors(n)
        took = pa.device_memory()[0] - live
        rowptr = d.graph()[0]
    assert np.array_equal(got, np.diff(rowptr))
    assert took <= (144 << 20 if mesh == "apart" else 600 << 20), took


@pytest.mark.parametrize("shift", [0, 1 << 20, 1 << 40])
@pytest.mark.parametrize("parts", [1, 2, 37, 1000])
@pytest.mark.parametrize("mesh", ["hex", "quads"])
def test_quality(oracle, mesh, parts, shift):
    """Parts in bricks and scattered, vertex ids that need 32 and 64 bits,
    tiles of the component search that end inside the mesh."""
    import parrsb_amd as pa
    print("quality", mesh, parts, shift, flush=True)
    vtx, xyz, nv = (M.box_hex(19, 13, 11, jitter=0.0) if mesh == "hex"
                    else M.holed_quads(61, 57, seed=3, rmax=7.0))
    n = vtx.shape[0]
    rng = np.random.default_rng(parts)
    for part in ((np.arange(n) * parts // n).astype(np.int32),
                 rng.integers(0, parts, n).astype(np.int32)):
        want = oracle.quality(part, vtx, nv, parts)
        assert pa.quality(part, vtx + shift, nv, parts) == want
