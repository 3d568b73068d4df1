"""The FP32 walk's pair loops for every replication of a target (runs of up to 96 targets, the last of a cell of any size: 64, 32, 16, 8,
4, 2 or 1 lanes a target, one target or three a lane) against the FP64 walk of the same box and groups.

Tolerance: a target adds up to some 2000 terms of either sign in FP32, each rounded to 2^-24, and the table
is within 2.4e-6 of the law: 2000 x 2^-24 = 1.2e-4 of the largest sums at worst, taken relative to
the rms acceleration."""
import numpy as np
import pytest

from lageunha_amd import ics, lagpm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("group", [8, 11, 16, 20, 32, 40, 64, 96])
def test_pair_loops_of_every_group_size(ctx, group):
    n = 32
    pos = ics.clustered_box(n, halo_fraction=0.1, nhalo=30, seed=group)[:12000]
    out = []
    for prec in (lagpm.PREC_FP32, lagpm.PREC_FP64):
        with lagpm.Box(ctx, lagpm.make_params(n, precision=prec, theta=1e-6), len(pos)) as b:
            b.set_tuning(8, group, lagpm.GROUPS_RUNS)
            b.upload_pos(pos)
            b.treecorrection(lagpm.evolfact(1.0))
            out.append(b.velocities())
    rms = np.sqrt((out[1] ** 2).sum(axis=1).mean())
    assert rms > 0 and np.abs(out[0] - out[1]).max() <= 1.2e-4 * max(rms, np.abs(out[1]).max())
