"""Level kernels at the sizes where their forms change: LDS sorts, LDS sets of
neighbouring segments, 32- and 64-bit quality keys."""
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
