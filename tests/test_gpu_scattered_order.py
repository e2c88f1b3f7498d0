"""Element orders whose neighbours lie scattered: the context then keeps an
element's four diffusing species side by side and takes tiles of 128.  The same
elements in the default order, in blocks of 64, are the reference: an element's
step reads its neighbours in the order of its own row, so fields, channels and
records are the same bits in every order."""
from __future__ import annotations

import numpy as np
import pytest

import srs_amd as S
from srs_amd import workloads as W
from tests.helpers import fast_gating

pytestmark = pytest.mark.gpu


def _mesh(n_xy, dyad=False):
    g = S.box_grid(W.dyad_box_spec(h=2.0 / n_xy) if dyad else W.spark_box_spec(h=1.0 / n_xy, n_xy=n_xy))
    aij, nij = S.assemble_operator(g)
    p = fast_gating(W.spark_params(t_final=1e9, states_interval=0.001, dt=W.stable_dt(aij, 0.22)))
    p.seti(INIT_RYR=0)
    return g, aij, nij, p


def _context(g, aij, nij, p, perm, members, tune, cap=0):
    ctx = S.Context(0)
    late = {k: v for k, v in tune.items() if k in ("gated_sweep", "nt_state", "occupancy")}
    ctx.tune(**{k: v for k, v in tune.items() if k not in late})
    mid = ctx.add_mesh_grid(g, aij, nij, perm=perm)
    for m in range(members):
        ctx.add_realization(mid, g.ryr_ele, g.ryr_jsr, g.ryr_nb, g.lcc_ele, p, seed=9, stream=m)
    ctx.finalize(cap)
    ctx.tune(**late)
    rng = np.random.default_rng(4)
    X0 = S.equilibrium_state(g, p.reals)[0]
    for m in range(members):
        ctx.state_set(m, X0 * rng.uniform(0.9, 1.0, X0.shape))
    return ctx, mid


def _shuffled(g):
    return np.random.default_rng(11).permutation(g.n_ele).astype(np.int32)


@pytest.mark.parametrize("n_xy,dyad,members,tune", [
    (9, False, 1, {}), (22, False, 1, {}), (25, True, 1, {}), (22, False, 3, {}), (60, False, 1, {}),
    (22, False, 1, dict(compact=0, nt_state=1)), (22, False, 2, dict(compact=0, nt_state=1)),
    (22, False, 1, dict(tile=256, gated_sweep=0)), (22, False, 2, dict(tile=512, nt_state=1)),
    (22, False, 1, dict(tile=512, occupancy=6)), (22, False, 1, dict(tile=256, plane_pad=64))])
def test_scattered_order_steps_the_same_bits(n_xy, dyad, members, tune):
    """Gated steps, the loop body with its records, a recorded and a replayed
    run, Ca at the channels."""
    g, aij, nij, p = _mesh(n_xy, dyad)
    out = []
    for perm in (None, _shuffled(g)):
        ctx, _ = _context(g, aij, nij, p, perm, members, tune, cap=64)
        with ctx:
            ctx.explicit_step(23, S.STEP_GRAPH)
            ctx.explicit_step(40, S.STEP_PROTOCOL)
            o = [ctx.records(m) for m in range(members)]
            assert len(o[0]) > 0
            o += ctx.record_schedules(12)
            if members == 1:
                ctx.replay(0, o[-1])
            for m in range(members):
                o += [ctx.state_get(m), *ctx.channels_get(m), *ctx.channel_ca(m)]
            out.append(o)
    assert len(out[0]) == len(out[1])
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("members,gated", [(1, 1), (1, 0), (3, 1)])
def test_scattered_order_loss_and_gradient(members, gated):
    """Scan samples, losses and gradients.  Fields and adjoints are the same
    bits but for the loss coefficients, whose sums over cells run in another
    order (some 1e-15); a gradient component is a sum of at most a few hundred
    terms in a row (2e-14 of the terms' size), which may cancel to a few
    thousandths of it: 1e-10."""
    g, aij, nij, p = _mesh(22)
    rng = np.random.default_rng(6)
    steps = 12
    scheds = [(rng.random((steps, g.n_ryr)) < 0.3).astype(np.int32) for _ in range(members)]
    d = S.read_scan_parameters(None)
    c0 = np.array([0.5, 0.5, 0.3])
    rc = g.centroids()[g.ryr_ele].mean(axis=0) - c0
    d.axis, d.offset1, d.offset2 = 0, float(rc[1]), float(rc[2])
    d.x_min, d.x_max, d.res_x_f, d.res_x_ca = -0.45, 0.45, 0.9 / 21.5, 0.04
    for q, size in enumerate((1.0, 1.0, 0.6)):
        d.domain[q] = size
    d.pad_min, d.pad_max, d.pad_res = -1.5, 1.5, 0.5
    out = []
    for perm in (None, _shuffled(g)):
        ctx, mid = _context(g, aij, nij, p, perm, members, dict(gated_sweep=gated))
        with ctx:
            sid, nf, _ = ctx.add_scan(mid, g.centroids() - c0, d)
            tg = np.tile(np.linspace(0.0, 0.2, nf), (members, 3, 1))
            loss, grad = ctx.loss_grad_batch(range(members), sid, scheds, [4, 9, 12], tg, ckpt=4)
            out.append((ctx.scan_sample(0, sid), loss, grad))
    (sa, la, ga), (sb, lb, gb) = out
    assert np.array_equal(sa[0], sb[0]) and np.array_equal(sa[1], sb[1])
    np.testing.assert_allclose(sa[2], sb[2], rtol=1e-12, atol=0)
    np.testing.assert_allclose(la, lb, rtol=1e-10, atol=0)
    np.testing.assert_allclose(ga, gb, rtol=1e-10, atol=0)
    assert np.all(np.any(ga != 0, axis=0)[[0, 1, 4, 8, 11]])
