"""The FP64 walk where a team of four waves takes several groups one after the other: about 1024 teams
and many more groups, of few targets and of up to 128, some boxes with heavy groups beside light ones.
Every particle gets the kick of its own group once: the accelerations are the FP32 walk's, the same bits
in every run."""
import numpy as np
import pytest

from lageunha_amd import ics, lagpm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("group,mode", [(8, 1), (16, 0), (64, 2)])
@pytest.mark.parametrize("n", [24, 48])
def test_teams_take_many_groups_each(ctx, n, group, mode):
    pos = ics.clustered_box(n, halo_fraction=0.3, nhalo=n, seed=group)
    acc = {}
    for prec in (lagpm.PREC_FP32, lagpm.PREC_FP64, lagpm.PREC_FP64):
        print(f"N={len(pos)} group {group} mode {mode} prec {prec}", flush=True)
        with lagpm.Box(ctx, lagpm.make_params(n, precision=prec, theta=0.5), len(pos)) as b:
            b.set_tuning(8, group, mode)
            b.upload_pos(pos)
            b.treecorrection(lagpm.evolfact(1.0))
            acc.setdefault(prec, []).append(b.velocities())
            groups = b.tree_stats().n_groups
    first, again = acc[lagpm.PREC_FP64]
    assert np.array_equal(first, again)
    d = acc[lagpm.PREC_FP32][0] - first
    assert groups > 100 and np.sqrt((d ** 2).sum() / (first ** 2).sum()) < 1e-4  # the FP32 walk's own bound
    # a particle without its kick, or with another's, is off by its whole acceleration: 1e-2 of the rms
    # is a hundred times the bound above
    rms = np.sqrt((first ** 2).sum(axis=1).mean())
    worst = np.sqrt((d ** 2).sum(axis=1)) / (rms + np.sqrt((first ** 2).sum(axis=1)))
    assert worst.max() < 1e-2
