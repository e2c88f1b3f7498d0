"""Field transfers between the caller's layout and the device's: a pinned
buffer holds 1,048,576 doubles, so fields of more than 174,762 elements cross
in parts, through two buffers in turn."""
from __future__ import annotations

import numpy as np
import pytest

import srs_amd as S
from srs_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_xy,group,members", [(9, 1, 1), (9, 4, 3), (59, 1, 1), (59, 2, 2)])
def test_fields_come_back_as_they_were_set(n_xy, group, members):
    """state_set then state_get returns every bit for each member of a
    realization group, in a shuffled element order, below and above the
    buffers' size; a step then reads what was set (two contexts with
    different orders agree)."""
    spec = W.spark_box_spec(h=1.0 / n_xy, n_xy=n_xy)
    g = S.box_grid(spec)
    aij, nij = S.assemble_operator(g)
    p = W.spark_params(dt=W.stable_dt(aij, 0.22))
    p.seti(INIT_RYR=-1)
    X0, _ = S.equilibrium_state(g, p.reals)
    rng = np.random.default_rng(5)
    states = [X0 * rng.uniform(0.9, 1.0, X0.shape) for _ in range(members)]
    after = []
    for perm in (None, rng.permutation(g.n_ele).astype(np.int32)):
        with S.Context(0) as ctx:
            ctx.tune(group=group)
            mid = ctx.add_mesh_grid(g, aij, nij, perm=perm)
            for m in range(members):
                ctx.add_realization(mid, g.ryr_ele, g.ryr_jsr, g.ryr_nb, g.lcc_ele, p, seed=3, stream=m)
            ctx.finalize()
            for m in range(members):
                ctx.state_set(m, states[m])
            for m in range(members):
                assert np.array_equal(ctx.state_get(m), states[m])
            ctx.explicit_step(3)
            after.append([ctx.state_get(m) for m in range(members)])
    for a, b, x in zip(*after, states):
        assert np.array_equal(a, b) and not np.array_equal(a, x)
