"""The adjoint where a mesh's channel elements are not all a realization's own:
the reverse step finds an element's record by counting the flags below it in
its wavefront, and by search where other clusters' elements lie between."""
import numpy as np
import pytest

from tests.test_gpu_adjoint import _batch_ctx, _batch_setup, _targets

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("members", [[0, 1, 2], [2, 0], [1, 1]])
def test_shared_mesh_gradients_equal_those_of_a_mesh_of_their_own(members):
    """Each member's loss and gradient, stepped with members of other RyR
    subsets on the same mesh, against a context of its own: the same
    operations in the same order, so the same bits."""
    pr, all_members, samples = _batch_setup()
    mem = [all_members[m] for m in members]
    tg, _ = _targets(pr, mem, samples)
    ctx, sid, _, _ = _batch_ctx(pr, mem)
    loss, grad = ctx.loss_grad_batch(range(len(mem)), sid, [m[2] for m in mem], samples, tg, ckpt=32)
    ctx.close()
    for k, m in enumerate(mem):
        one, s1, _, _ = _batch_ctx(pr, [m])
        l1, g1 = one.loss_grad_batch([0], s1, [m[2]], samples, tg[k:k + 1], ckpt=32)
        for levels in (2, 3):  # recomputed in blocks from checkpoints of checkpoints
            one.tune(adj_levels=levels)
            l2, g2 = one.loss_grad_batch([0], s1, [m[2]], samples, tg[k:k + 1])
            assert l2[0] == l1[0] and np.array_equal(g2, g1)
        one.close()
        assert l1[0] == loss[k] and np.array_equal(g1[0], grad[k]) and np.any(g1[0] != 0)
