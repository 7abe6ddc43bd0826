"""The coarse end of the V-cycle in one workgroup (k_mg_low) against the
oracle, at the sizes where its form changes: a level of 64 / 65 rows (one
wave or the workgroup), of 1024 / 1025 rows (one or two rows per thread) and
of 2048 / 2050 rows (the workgroup or a launch per step), and factors that
are no powers of two.  With four and five levels above k_mg_low (33,920 and
67,200 elements) the way up takes k_mg_prolong_c first and evaluates the last
three in k_mg_up0."""
import numpy as np
import pytest

import parrsb_amd as pa
from parrsb_amd import meshgen as M


@pytest.mark.gpu
@pytest.mark.parametrize("dims,factor", [((4, 4, 8), 2), ((2, 5, 13), 2), ((8, 8, 32), 2),
                                         ((5, 10, 41), 2), ((8, 16, 32), 2), ((10, 10, 41), 2),
                                         ((1, 1, 2), 2), ((1, 1, 3), 7), ((6, 7, 20), 3),
                                         ((16, 20, 30), 5), ((16, 20, 106), 2), ((10, 24, 280), 2),
                                         ((16, 24, 170), 3)])
def test_low_levels_match_oracle(oracle, dims, factor):
    print("mg low", dims, factor, flush=True)
    vtx, xyz, nv = M.box_hex(*dims)
    n = vtx.shape[0]
    with pa.Device() as d:
        d.set_mesh(vtx, xyz, nv)
        d.set_segments([0], [n], [2], [0])
        d.prepartition(1)
        order = d.order()
        d.level_laplacian()
        out = d.fiedler_mg(1, factor=factor)
        f = d.fiedler_values()
    fo, it, npass = oracle.fiedler_mg(vtx, nv, order, factor=factor)
    # FP64 on both sides, sums in other orders: the same steps to rounding
    assert abs(f @ fo - 1) < 1e-8
    assert out["npass"][0] == npass
    assert abs(out["niter"][0] - it) <= 1
