"""A tree kick whose build overflows its node arrays first (they are grown and the tree redone)
adds the kick and nothing else."""
import numpy as np
import pytest

from lageunha_amd import lagpm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [lagpm.PREC_FP32, lagpm.PREC_FP64])
def test_kick_after_regrown_nodes_is_the_kick(ctx, prec):
    n, count = 32, 24000  # leaves of 4: more than count / 3 + 4096 nodes
    pos = np.random.default_rng(count).random((count, 3)) * n
    with lagpm.Box(ctx, lagpm.make_params(n, precision=prec), count) as b:
        b.set_tuning(4, 8)
        b.upload_pos(pos)
        b.treecorrection(lagpm.evolfact(1.0))
        first = b.velocities()
        assert b.tree_stats().n_nodes > count // 3 + 4096 + 64
        b.treecorrection(lagpm.evolfact(1.0))
        assert np.array_equal(b.velocities(), 2 * first)
