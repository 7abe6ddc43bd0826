"""Fused Lanczos iterations against the separate finishing launches: the same
sums in the same order, so every result has the same bits."""
import numpy as np
import pytest

from parrsb_amd import meshgen as M

pytestmark = pytest.mark.gpu


def _solve(vtx, xyz, nv, bounds, prec):
    """Fiedler solve of the segments [bounds[i], bounds[i+1]) of the input
    order, two virtual ranks each."""
    import parrsb_amd as pa
    b = np.asarray(bounds)
    nseg = b.size - 1
    with pa.Device() as d:
        d.set_mesh(vtx, xyz, nv)
        d.set_segments(b[:-1], np.diff(b), np.full(nseg, 2), 2 * np.arange(nseg))
        d.prepartition(1)
        d.level_laplacian()
        out = d.fiedler(nseg, precision=prec, max_passes=6)
        return out, d.fiedler_values()


CASES = {
    # a pass shorter than rsb_max_iter, one row past a tile, a whole number
    # of tiles, and many segments that stop at different iterations
    "tiny": lambda: (M.box_hex(3, 2, 2), [0, 12]),
    "tile_plus_one": lambda: (M.box_hex(41, 25, 1), [0, 1025]),
    "tiles": lambda: (M.box_hex(32, 16, 16, jitter=0.1), [0, 8192]),
    "uneven": lambda: (M.warped_box_hex(24, seed=3), [0, 2, 67, 1091, 1092, 6000, 13824]),
    "quads": lambda: (M.holed_quads(150, 140, seed=4, rmax=9.0), None),
}


@pytest.mark.parametrize("tiles", ["lds", "global"])
@pytest.mark.parametrize("prec,fold", [(64, "0"), (32, "0"), (32, "4096")])
@pytest.mark.parametrize("name", list(CASES))
def test_fused_iterations_equal_separate_launches(name, prec, fold, tiles, monkeypatch):
    print("fused", name, prec, fold, tiles, flush=True)
    (vtx, xyz, nv), bounds = CASES[name]()
    n = vtx.shape[0]
    bounds = bounds or [0, n // 3, n // 3 + 1200, n]
    monkeypatch.setenv("PARRSB_AMD_LZ_FOLD_TILES", fold)
    if tiles == "global":
        monkeypatch.setenv("PARRSB_AMD_NO_TILES", "1")
    res = {}
    for fuse in ("1024", "0"):
        monkeypatch.setenv("PARRSB_AMD_LZ_FUSE_TILES", fuse)
        res[fuse] = _solve(vtx, xyz, nv, bounds, prec)
    (of, ff), (ou, fu) = res["1024"], res["0"]
    for k in ("niter", "npass", "lambda", "rnorm", "resid"):
        assert np.array_equal(of[k], ou[k], equal_nan=True), k
    assert np.array_equal(ff, fu)


@pytest.mark.parametrize("prec,fold", [(64, "0"), (32, "0"), (32, "4096")])
@pytest.mark.parametrize("dims", [(64, 64, 128), (128, 64, 127), (128, 64, 128)])
def test_fused_iterations_of_large_segments(dims, prec, fold, monkeypatch):
    """Segments of 512, 1,016 and 1,024 tiles, the last the fused form's limit,
    and the same cut at 513 tiles (at one for the first): the sums of a
    segment take one round of a workgroup's loads, folded two above 512."""
    print("fused large", dims, prec, fold, flush=True)
    (vtx, xyz, nv), n = M.box_hex(*dims, jitter=0.1, seed=1), int(np.prod(dims))
    res = {}
    monkeypatch.setenv("PARRSB_AMD_LZ_FOLD_TILES", fold)
    for fuse in ("1024", "0"):
        monkeypatch.setenv("PARRSB_AMD_LZ_FUSE_TILES", fuse)
        import parrsb_amd as pa
        with pa.Device() as d:
            d.set_mesh(vtx, xyz, nv)
            for b in ([0, n], [0, 513 * 1024 - 100, n] if n > 513 * 1024 else [0, 1000, n]):
                nseg = len(b) - 1
                d.set_segments(b[:-1], np.diff(b), [2] * nseg, 2 * np.arange(nseg))
                d.prepartition(1)
                d.level_laplacian()
                out = d.fiedler(nseg, precision=prec, max_iter=12, max_passes=2)
                res.setdefault(fuse, []).append((out, d.fiedler_values()))
    for (of, ff), (ou, fu) in zip(res["1024"], res["0"]):
        for k in ("niter", "npass", "lambda", "rnorm", "resid"):
            assert np.array_equal(of[k], ou[k], equal_nan=True), k
        assert np.array_equal(ff, fu)


@pytest.mark.parametrize("n", [1, 2, 50, 63, 64, 65, 128])
def test_tridiagonal_solves_over_wide_ranges(n, oracle):
    """Entries over 300 decades, zero off-diagonals and a zero diagonal leave
    the plain divide's range: the QL solve keeps the oracle's bits, and the
    multisection solve's eigenvalue agrees with it to rounding of the largest
    entry."""
    import parrsb_amd as pa
    rng = np.random.default_rng(n)
    for kind in range(4):
        if kind == 0:
            d, e = 10.0 ** rng.uniform(-150, 150, n), 10.0 ** rng.uniform(-150, 150, n - 1)
        elif kind == 1:
            d, e = rng.uniform(0.1, 4, n), np.where(rng.random(n - 1) < 0.3, 0.0, 0.5)
        elif kind == 2:
            d, e = np.zeros(n), rng.uniform(0.1, 1, n - 1)
        else:
            d, e = np.full(n, 2.0), np.full(n - 1, -1.0)
        print("tridiagonal", n, kind, flush=True)
        lam, y = pa.test_tqli(d, e)
        rc, ev, z = oracle.tqli(d, e)
        k = int(np.argmin(np.abs(ev)))
        assert lam == ev[k] and np.array_equal(y, z[k]), kind
        if kind in (1, 3):
            fast, _ = pa.test_tqli(d, e, fast=True)
            assert abs(fast - lam) <= 1e-12 * (np.abs(d).max() + 1.0)
