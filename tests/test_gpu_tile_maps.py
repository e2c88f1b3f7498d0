"""Where a tile's neighbours are staged: the maps that srs_ctx_finalize builds,
on one thread and on several, for every tile size and padding, and the fields'
way in and out in parts.  An element's step reads its neighbours in the order of
its own row, so fields are the same bits whatever the order, tile and padding."""
from __future__ import annotations

import numpy as np
import pytest

import srs_amd as S
from srs_amd import workloads as W

pytestmark = pytest.mark.gpu


def _mesh(n_xy):
    g = S.box_grid(W.spark_box_spec(h=1.0 / n_xy, n_xy=n_xy))
    aij, nij = S.assemble_operator(g)
    p = W.spark_params(dt=W.stable_dt(aij, 0.22))
    X = S.equilibrium_state(g, p.reals)[0]
    return g, aij, nij, p, X * np.random.default_rng(8).uniform(0.9, 1.0, X.shape)


def _stepped(m, members=1, tune=None, flags=0, **order):
    g, aij, nij, p, X = m
    with S.Context(0) as ctx:
        ctx.tune(**(tune or {}))
        mid = ctx.add_mesh_grid(g, aij, nij, **order)
        for k in range(members):
            ctx.add_realization(mid, g.ryr_ele, g.ryr_jsr, g.ryr_nb, g.lcc_ele, p, seed=3, stream=k)
        ctx.finalize()
        for k in range(members):
            ctx.state_set(k, X)
        ctx.explicit_step(16, flags)
        return ctx.state_get(members - 1)


# 124,146 and 138,720 elements: either side of 131,072, from where several
# threads build the map
@pytest.mark.parametrize("n_xy", [10, 33, 34])
def test_maps_of_every_tile_and_padding(n_xy):
    m = _mesh(n_xy)
    want = _stepped(m, order=S.ORDER_AS_GIVEN)
    assert not np.array_equal(want, m[4])
    for tile in (128, 256, 512):
        for pad in (0, 64):
            assert np.array_equal(_stepped(m, tune=dict(tile=tile, plane_pad=pad)), want), (tile, pad)


# one part (63,504 doubles), two (72,900), eight (514,692 doubles), two halves (550,800
# doubles); a small mesh's fields move through buffers that the large one's set
@pytest.mark.parametrize("n_xys", [(14,), (15,), (29,), (30,), (10, 37)])
def test_fields_in_parts(n_xys):
    meshes = [_mesh(n) for n in n_xys]
    with S.Context(0) as ctx:
        for g, aij, nij, p, _ in meshes:
            ctx.add_realization(ctx.add_mesh_grid(g, aij, nij), g.ryr_ele, g.ryr_jsr, g.ryr_nb, g.lcc_ele, p, seed=1, stream=0)
        ctx.finalize()
        for _ in range(2):
            for r, m in enumerate(meshes):
                ctx.state_set(r, m[4])
            for r, m in enumerate(meshes):
                assert np.array_equal(ctx.state_get(r), m[4])


# Runs of 64 elements of the block order, shuffled: a 512-element tile stages 2,500
# quads, of which two workgroups, not three, fit a CU's LDS, so 256 are taken
@pytest.mark.parametrize("members", [1, 3])
def test_tile_of_an_order_with_large_halos(members):
    m = _mesh(22)
    n = m[0].n_ele
    block = W.kuhn_block_order(m[0])
    runs = [block[i:i + 64] for i in range(0, n, 64)]
    perm = np.concatenate([runs[i] for i in np.random.default_rng(0).permutation(len(runs))])
    want = _stepped(m, members, order=S.ORDER_AS_GIVEN)
    for tune in ({}, dict(tile=512), dict(tile=256), dict(gated_sweep=0)):
        assert np.array_equal(_stepped(m, members, tune, perm=perm), want), tune


# 658,080 and 703,452 elements: the gated step's register budget changes at 700,000
@pytest.mark.parametrize("n_xy", [60, 61])
def test_register_budgets_either_side_of_their_line(n_xy):
    g = S.box_grid(W.dyad_box_spec(h=2.0 / n_xy))
    assert (g.n_ele < 700_000) == (n_xy == 60) and abs(g.n_ele - 700_000) < 50_000
    aij, nij = S.assemble_operator(g)
    p = W.spark_params(dt=W.stable_dt(aij, 0.22))
    m = g, aij, nij, p, S.equilibrium_state(g, p.reals)[0]
    got = _stepped(m)
    assert np.array_equal(got, _stepped(m, tune=dict(occupancy=6)))
    assert np.array_equal(got, _stepped(m, tune=dict(gated_sweep=0)))


# 253 and 276 tiles of 128 elements; 256 and 288 of 256
@pytest.mark.parametrize("n_xy,members", [(9, 11), (9, 12), (13, 8), (13, 9)])
def test_tiles_of_small_ensembles(n_xy, members):
    m = _mesh(n_xy)
    want = _stepped(m, order=S.ORDER_AS_GIVEN)
    for tune in ({}, dict(tile=512)):
        for flags in (0, S.STEP_GRAPH):
            assert np.array_equal(_stepped(m, members, tune, flags), want), (tune, flags)
