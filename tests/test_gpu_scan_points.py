"""The blurred line scan at the sizes where its kernels split the work: points
go in segments of 16 (two halves of 8), four to a matrix reduction, cells 1024
to a workgroup, workgroups' partial sums 64 to a wavefront."""
from __future__ import annotations

import numpy as np
import pytest

import srs_amd as S
from srs_amd import workloads as W
from oracle.oracle import PHILOX_KEY1, RNG_GLIBC, RNG_PHILOX, Fields, Oracle, grid_dict

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_xy,points", [(9, [1, 4, 7, 8, 9, 15, 16, 17, 24, 33, 1024]), (33, [1, 8, 17, 130])])
def test_blur_at_segment_edges(n_xy, points):
    """Every point against the oracle's sum over all cells.  A weight is at most
    eight products from a closed form (some 20 ulps) and all terms of a sum
    are positive, so 1e-12 as for the other scans.  One cell's value is then
    NaN: exactly the points that reach it are, as in the oracle."""
    g = S.box_grid(W.spark_box_spec(h=1.0 / n_xy, n_xy=n_xy))
    aij, nij = S.assemble_operator(g)
    p = W.spark_params(dt=W.stable_dt(aij, 0.22))
    cen = g.centroids() - np.array([0.5, 0.5, 0.3])
    n = g.n_ele
    rng = np.random.default_rng(3)
    X = S.equilibrium_state(g, p.reals)[0]
    X[5 * n:] *= rng.uniform(1.0, 4.0, n)
    bad = X.copy()
    bad[5 * n + int(np.argmin(cen[:, 0]))] = np.nan
    with S.Context(0) as ctx:
        mid = ctx.add_mesh_grid(g, aij, nij, perm=W.kuhn_block_order(g))
        ctx.add_realization(mid, g.ryr_ele, g.ryr_jsr, g.ryr_nb, g.lcc_ele, p, seed=1, stream=0)
        ctx.finalize()
        for k in points:
            d = S.read_scan_parameters(None)
            d.axis, d.offset1, d.offset2 = 0, 0.03, -0.2
            d.x_min, d.x_max, d.res_x_f, d.res_x_ca = -0.8, 1.2, 2.0 / (k + 0.5), 0.5
            for q, size in enumerate((1.0, 1.0, 0.6)):
                d.domain[q] = size
            d.pad_min, d.pad_max, d.pad_res = -1.5, 1.5, 0.5
            sid, nf, _ = ctx.add_scan(mid, cen, d)
            assert nf == k
            for state in (X, bad):
                ctx.state_set(0, state)
                got = ctx.scan_sample(0, sid)[2]
                ref = Oracle().linescan(d, cen, g.V0, state[:n], state[5 * n:])[2]
                ok = np.isfinite(ref)
                np.testing.assert_array_equal(np.isfinite(got), ok)
                np.testing.assert_allclose(got[ok], ref[ok], rtol=1e-12, atol=0)
