"""The single-launch step's gating workgroup at the edges of what it holds:
more RyRs and more channel elements than it has threads, coupled RyRs, and
each of its register budgets (by the number of tiles, or asked for)."""
from __future__ import annotations

import numpy as np
import pytest

import srs_amd as S
from oracle.oracle import RNG_PHILOX, Oracle, grid_dict
from srs_amd import workloads as W
from tests.helpers import fast_gating, initial_fields

pytestmark = pytest.mark.gpu


# 2,160 elements (17 tiles of 128) and 37,752 (295 tiles: more than 256)
@pytest.mark.parametrize("n_xy,rows,occ,a_star", [(9, 14, 0, 0.0), (9, 14, 6, 0.05), (9, 1, 0, 0.05), (22, 14, 0, 0.05),
                                                  (22, 3, 6, 0.0), (22, 3, 0, 0.0)])
def test_gating_workgroup_matches_oracle(n_xy, rows, occ, a_star):
    """120 gated steps in two calls, 128-element tiles (128 threads gate up
    to 196 RyRs and update up to a few hundred channel elements): fields,
    channel states and residual order equal the oracle's bit for bit."""
    spec = W.spark_box_spec(h=1.0 / n_xy, n_xy=n_xy, ryr_rows=rows, ryr_cols=rows)
    g = S.box_grid(spec)
    aij, nij = S.assemble_operator(g)
    p = fast_gating(W.spark_params(dt=W.stable_dt(aij, 0.22)))
    p.setr(RYR_A_STAR=a_star, RYR_PHI_M=2.0 if rows == 3 else 0.0, RYR_K_PLUS=20.0, RYR_K_MINUS=400.0)
    p.seti(INIT_RYR=0)
    X0, bnd = S.equilibrium_state(g, p.reals)
    pr = W.Prepared(g, aij, nij, X0, bnd, p)
    F = initial_fields(pr, seed=11)
    with S.Context(0) as ctx:
        ctx.tune(tile=128, occupancy=occ)
        mid = ctx.add_mesh_grid(g, aij, nij, perm=S.morton_order(g))
        ctx.add_realization(mid, g.ryr_ele, g.ryr_jsr, g.ryr_nb, g.lcc_ele, p, seed=77, stream=2)
        ctx.finalize()
        ctx.state_set(0, F.X)
        ctx.channels_set(0, F.ryr_state, F.lcc_state, F.lccv_state, F.R)
        ctx.globals_set(0, F.gv[0], F.gv[1])
        ctx.explicit_step(101, S.STEP_GRAPH)
        ctx.explicit_step(19)
        X, ch = ctx.state_get(0), ctx.channels_get(0)
    Fo = Oracle().steps(grid_dict(g, aij, nij), p.reals, F.copy(), 120, p.reals[1], gating=True, rng_kind=RNG_PHILOX,
                        key=77, stream=2)
    assert np.array_equal(ch[0], Fo.ryr_state) and np.array_equal(ch[1], Fo.lcc_state)
    assert np.array_equal(ch[2], Fo.lccv_state)
    assert np.array_equal(X, Fo.X)
    assert not np.array_equal(ch[0], F.ryr_state)  # the RyRs did move
