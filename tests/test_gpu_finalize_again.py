"""srs_ctx_finalize called again after a call that failed part way: the second
call starts from nothing, so the context is that of a program that finalized
once."""
from __future__ import annotations

import numpy as np
import pytest

import srs_amd as S
from srs_amd import workloads as W
from tests.helpers import fast_gating

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("members,late", [(1, 0), (5, 0), (1, 2)])
def test_finalize_after_a_failed_finalize(members, late):
    """A record of 399 floats is refused with a record buffer and accepted
    without one.  `late` realizations are added between the two calls.  Gated
    steps, the loop body's included, and a transfer then equal those of a
    context finalized once, bit for bit."""
    g = S.box_grid(W.spark_box_spec(h=1.0 / 9, n_xy=9, ryr_rows=14, ryr_cols=14))
    aij, nij = S.assemble_operator(g)
    p = fast_gating(W.spark_params(dt=W.stable_dt(aij, 0.22)))
    p.seti(INIT_RYR=0, FLAG_RYR_OUT=1)
    X0, _ = S.equilibrium_state(g, p.reals)
    rng = np.random.default_rng(2)
    states = [X0 * rng.uniform(0.9, 1.0, X0.shape) for _ in range(members + late)]
    got = []
    for fail_first in (True, False):
        with S.Context(0) as ctx:
            ctx.record_layout(True)
            mid = ctx.add_mesh_grid(g, aij, nij)
            for m in range(members + late):
                if m == members and fail_first:
                    with pytest.raises(S.SrsError, match="record limit"):
                        ctx.finalize(16)
                ctx.add_realization(mid, g.ryr_ele, g.ryr_jsr, g.ryr_nb, g.lcc_ele, p, seed=5, stream=m)
            if fail_first and not late:
                for _ in range(2):
                    with pytest.raises(S.SrsError, match="record limit"):
                        ctx.finalize(16)
            ctx.finalize(0)
            for m, X in enumerate(states):
                ctx.state_set(m, X)
            ctx.explicit_step(40, S.STEP_GRAPH)
            ctx.explicit_step(7)
            got.append([(ctx.state_get(m), ctx.channels_get(m)) for m in range(members + late)])
    for (Xa, ca), (Xb, cb), X in zip(*got, states):
        assert np.array_equal(Xa, Xb) and not np.array_equal(Xa, X)
        assert all(np.array_equal(a, b) for a, b in zip(ca, cb))
