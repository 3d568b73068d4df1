"""A box whose particles were last sorted for a shallow tree, then given smaller leaves: the next tree
reaches below the levels that were sorted, and equals that of a fresh box with the same leaves."""
import numpy as np
import pytest

from lageunha_amd import lagpm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [lagpm.PREC_FP32, lagpm.PREC_FP64])
@pytest.mark.parametrize("clump", [40, 300])
def test_smaller_leaves_after_a_shallow_sort(ctx, prec, clump):
    n = 32
    g = np.random.default_rng(clump)
    # a clump inside one cell of level 10 (0.031 wide), its particles in finest cells of their own
    q = g.permutation(40 ** 3)[:clump]
    tight = np.array([9.0, 20.0, 14.0]) + (np.stack([q % 40, q // 40 % 40, q // 1600], -1) + 0.5) * (n / 65536.0)
    pos = np.concatenate([tight, g.random((600, 3)) * n])[g.permutation(clump + 600)]
    p = lagpm.make_params(n, precision=prec)
    with lagpm.Box(ctx, p, len(pos)) as b, lagpm.Box(ctx, p, len(pos)) as fresh:
        b.set_tuning(256, 64)
        b.upload_pos(pos)
        b.treecorrection(lagpm.evolfact(0.0))
        limit = b.tree_stats().depth_limit
        b.drift(0.0)
        b.tsc()  # sorts for that limit
        b.set_tuning(4, 8)
        b.treecorrection(lagpm.evolfact(1.0))
        fresh.set_tuning(4, 8)
        fresh.upload_pos(pos)
        fresh.treecorrection(lagpm.evolfact(1.0))
        print(f"limit {limit}, then deepest {b.tree_stats().deepest}", flush=True)
        assert b.tree_stats().deepest >= 13
        assert clump > 256 or limit <= 10  # 32 sorted key bits or fewer
        got, want = b.tree_nodes(), fresh.tree_nodes()
        assert np.array_equal(got["info"], want["info"]) and np.array_equal(got["com"], want["com"])
        assert np.array_equal(b.velocities(), fresh.velocities())
