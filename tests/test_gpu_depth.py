"""A tree that gets deeper from one step to the next than the box expected: where the sort has put all
key bits in order the build goes on below the expected depth, elsewhere it is redone. Either way the
step equals that of a fresh box (first tree at full depth) on the same particles, bit for bit."""
import numpy as np
import pytest

from lageunha_amd import ics, lagpm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [lagpm.PREC_FP32, lagpm.PREC_FP64])
@pytest.mark.parametrize("spacing,edge,below", [(0.25, 4, False), (0.03, 4, True), (0.02, 18, True), (0.013, 7, True)])
def test_a_tightening_clump_equals_a_fresh_box(ctx, spacing, edge, below, prec):
    n, a, da = 32, 1.0, 0.001
    g = np.random.default_rng(edge)
    # a small lattice, drawn 12 times tighter by one drift (da n v): its particles stay further apart than
    # the finest key cell (n / 65536), so the order of the keys has no ties
    centre = np.array([9.3, 20.1, 14.7])
    grid = np.stack(np.meshgrid(*[np.arange(edge)] * 3), -1).reshape(-1, 3) - (edge - 1) / 2
    clump = centre + spacing * (grid + 0.02 * g.uniform(-1, 1, grid.shape))
    lat = ics.perturbed_lattice(n, rms=0.3, seed=2)[len(clump):]
    pos = np.concatenate([lat, clump])
    vel = np.zeros_like(pos)
    vel[len(lat):] = (centre - clump) * (11.0 / 12.0) / (da * n)
    p = lagpm.make_params(n, precision=prec)
    with lagpm.Box(ctx, p, len(pos)) as b, lagpm.Box(ctx, p, len(pos)) as fresh:
        b.upload_pos(pos, vel)
        b.kdk_step(a, da)
        st = b.tree_stats()
        x, v = b.download()
        b.kdk_step(a + da, da)
        st2 = b.tree_stats()
        fresh.upload_pos(x, v)
        fresh.kdk_step(a + da, da)
        stf = fresh.tree_stats()
        got, want = b.download(), fresh.download()
    print(f"deepest {st.deepest} limit {st.depth_limit}, then deepest {st2.deepest} limit {st2.depth_limit}", flush=True)
    assert (st.depth_limit >= 11) == below and st2.deepest > st.depth_limit  # 11 levels and more: six sort passes
    assert st2.deepest == stf.deepest and st2.n_nodes == stf.n_nodes and st2.depth_limit == min(16, st2.deepest + 2)
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
