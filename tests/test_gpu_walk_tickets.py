"""Every target group is walked exactly once, whatever the number of groups against the walk's
waves: groups are handed out by rank first and by per-range tickets after."""
import numpy as np
import pytest

from lageunha_amd import lagpm

pytestmark = pytest.mark.gpu


def relerr(a, b):
    return float(np.sqrt(np.sum((a - b) ** 2) / np.sum(b ** 2)))


# 4096 waves on 256 CUs: from one group to fewer, about as many and many more groups than waves
@pytest.mark.parametrize("count", [1, 9, 700, 9000, 24000, 26000, 33000, 70000])
@pytest.mark.parametrize("reference_law", [False, True])
def test_every_group_is_walked(ctx, count, reference_law):
    n = 32
    pos = np.random.default_rng(count).random((count, 3)) * n
    kick = {}
    for prec in (lagpm.PREC_FP32, lagpm.PREC_FP64):
        p = lagpm.reference_params(n, precision=prec, theta=1e-6) if reference_law else lagpm.make_params(n, precision=prec, theta=1e-6)
        with lagpm.Box(ctx, p, count) as b:
            b.set_tuning(4, 8)
            b.upload_pos(pos)
            b.treecorrection(lagpm.evolfact(1.0))
            kick[prec] = b.velocities()
            st = b.tree_stats()
            print(f"count={count} prec={prec} groups={st.n_groups}", flush=True)
            # a second kick of the same tree adds the same, so no group was walked twice or left out
            b.treecorrection(lagpm.evolfact(1.0))
            assert np.array_equal(b.velocities(), 2 * kick[prec])
    a, r = kick[lagpm.PREC_FP32], kick[lagpm.PREC_FP64]
    if count == 1:
        assert not a.any() and not r.any()
        return
    # theta -> 0: both are within 3e-5 (rms) of the exact pair sums
    assert relerr(a, r) < 6e-5
    # an unwalked group of 8 would miss its whole kick
    worst = np.abs(a - r).max(axis=1) / np.abs(r).max(axis=1).mean()
    assert worst.max() < 1e-2
