"""Results read back through pinned memory or, above its size, by copies:
arrays just below and above the limit of 8,192 words."""
import numpy as np
import pytest

from parrsb_amd import meshgen as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 1365, 1366, 8192, 8193])
def test_arrays_around_the_pinned_limit(n):
    import parrsb_amd as pa
    print("read back", n, flush=True)
    vtx, xyz, nv = M.quad_grid(n, 1)
    with pa.Device() as d:
        d.set_mesh(vtx, xyz, nv)  # centroids: 6 n words
        c = xyz.reshape(n, nv, -1)
        ref = c[:, 0].copy()
        for k in range(1, nv):
            ref += c[:, k]
        assert np.array_equal(d.centroids()[:, :c.shape[2]], ref / nv)
        d.set_segments([0], [n], [1], [0])
        assert np.array_equal(np.sort(d.order()), np.arange(n))  # n words
