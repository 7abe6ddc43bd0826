"""The running lists of a Lanczos pass, taken up two iterations after their
compaction is queued, against the graph replays, which wait for each: the
same results to the bit, at pass lengths around the first compactions."""
import numpy as np
import pytest

from parrsb_amd import meshgen as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("max_iter", [7, 8, 10, 11, 12, 26, 27, 50])
@pytest.mark.parametrize("prec", [64, 32])
def test_delayed_lists_equal_waiting(prec, max_iter, monkeypatch):
    import parrsb_amd as pa
    print("lists", prec, max_iter, flush=True)
    vtx, xyz, nv = M.warped_box_hex(24, seed=3)
    b = np.array([0, 2, 9, 21, 67, 1091, 1092, 6000, 13824])
    nseg = b.size - 1
    res = []
    for graph in ("0", "1"):
        monkeypatch.setenv("PARRSB_AMD_LZ_GRAPH", graph)
        with pa.Device() as d:
            d.set_mesh(vtx, xyz, nv)
            d.set_segments(b[:-1], np.diff(b), np.full(nseg, 2), 2 * np.arange(nseg))
            d.prepartition(1)
            d.level_laplacian()
            out = d.fiedler(nseg, precision=prec, max_iter=max_iter, max_passes=5)
            res.append((out, d.fiedler_values()))
    (o0, f0), (o1, f1) = res
    for k in ("niter", "npass", "lambda", "rnorm", "resid"):
        assert np.array_equal(o0[k], o1[k], equal_nan=True), k
    assert np.array_equal(f0, f1)
