"""The FP32 path's sums against FP64 sums of the same data, where an iteration
shrinks the residual most: one iteration from a start close to an eigenvector,
|r_0| = rho |r_1|.  Its r_1 is formed again in FP64."""
import numpy as np
import pytest

from parrsb_amd import meshgen as M

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


@pytest.fixture(scope="module")
def problem():
    vtx, xyz, nv = M.box_hex(13, 10, 9, jitter=0.1, seed=2)
    import parrsb_amd as pa
    n = vtx.shape[0]
    with pa.Device() as d:
        d.set_mesh(vtx, xyz, nv)
        rowptr, col, w = d.graph()
    A = np.zeros((n, n))
    A[np.repeat(np.arange(n), np.diff(rowptr)), col] = w
    L = np.diag(A.sum(1)) - A
    lam, V = np.linalg.eigh(L)
    return (vtx, xyz, nv), L, lam, V


def _step(L, r):
    """r - alpha L r and the ratio of the norms, in FP64."""
    w = L @ r
    r1 = r - (r @ r) / (r @ w) * w
    return r1, np.linalg.norm(r) / np.linalg.norm(r1)


@pytest.mark.parametrize("fold", ["0", "4096"])
@pytest.mark.parametrize("rho", [4.0, 10.0, 100.0, 1000.0])
def test_residual_norm_within_the_sums_bound(problem, rho, fold, monkeypatch):
    """Folded, |r_1|^2 comes from r.r, r.w and w.w, each within 2^-24 of the sum
    of its terms' magnitudes: relative error 2^-24 (2 rho + 1)^2, half of it in
    the norm.  Summed from the stored r_1 instead there is only the rounding
    of r_0, w (27 terms a row) and alpha, each at most a few 2^-24 |r_0|."""
    import parrsb_amd as pa
    (vtx, xyz, nv), L, lam, V = problem
    n = vtx.shape[0]
    rng = np.random.default_rng(int(rho))
    # v_2 and as much of the next eigenvectors as leaves r_1 at |r_0| / rho
    mix = V[:, 2:40] @ rng.standard_normal(38)
    lo, hi = 1e-9, 1e3
    for _ in range(100):
        e = np.sqrt(lo * hi)
        lo, hi = (e, hi) if _step(L, V[:, 1] + e * mix)[1] > rho else (lo, e)
    x = (V[:, 1] + e * mix).astype(np.float32)
    monkeypatch.setenv("PARRSB_AMD_LZ_FOLD_TILES", fold)
    with pa.Device() as d:
        d.set_mesh(vtx, xyz, nv)
        d.set_segments([0], [n], [2], [0])
        d.level_laplacian()
        dx = d.upload(x)
        d._chk(pa.lib().rsbgpu_set_start(d.h, dx))
        out = d.fiedler(1, precision=32, max_iter=1, max_passes=1, tol=1e-30, init_mode=1)
        pa.Device.free(dx)
    r0 = x.astype(np.float64)
    r0 -= r0.mean()
    r0 /= np.linalg.norm(r0)
    r1, ratio = _step(L, r0)
    first, _, last = out["rnorm"]
    err = abs(last / first / np.linalg.norm(r1) - 1)
    bound = EPS * 64 * ratio + (EPS * (2 * ratio + 1) ** 2 / 2 if fold != "0" else 0)
    print("rho %.3g fold %s error %.2e bound %.2e" % (ratio, fold, err, bound), flush=True)
    assert out["niter"][0] == 1
    assert err < bound
