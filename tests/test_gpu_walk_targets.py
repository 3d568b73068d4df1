"""The FP32 walk's pair loops for every replication of a target, target by target: a lost or doubled source
shows at its own target, however small that one's acceleration is beside a halo's.

Bound for target i, against the FP64 walk of the same box and groups at theta -> 0 (all pairs), with
s = sqrt(r^2 + eps^2) and N = r / s^3, which a pair's force stays below: the sum over its n_i sources of
  N ((n_i + 40) 2^-24 + 2 x 2.4e-6)   the sum's roundings and the operations of a term; the table's lines
                                      are within 2.4e-6 of the law, and a rounded r^2 may take the next line
  4 sqrt(3) d / s^3                   the positions' rounding, d = 4 x 2^-24 n an axis (both ends and the image
                                      shift; |dN/dr| <= 4 / s^3)
  N if |r - rcut| < 1e-4              a pair on the other side of the cutoff
"""
import numpy as np
import pytest
from scipy.spatial import cKDTree

from lageunha_amd import ics, lagpm
from oracle import pyoracle as orc

pytestmark = pytest.mark.gpu


def bound(pos, p):
    n, eps = p.n, p.epsilon
    tree = cKDTree(pos, boxsize=n)
    pairs = tree.query_pairs(p.rsphere + 1e-3, output_type="ndarray")
    d = pos[pairs[:, 0]] - pos[pairs[:, 1]]
    d -= n * np.round(d / n)
    r = np.sqrt((d ** 2).sum(axis=1))
    s = np.sqrt(r ** 2 + eps ** 2)
    count = np.bincount(pairs.ravel(), minlength=len(pos))
    out = np.zeros(len(pos))
    for side in (0, 1):
        i = pairs[:, side]
        e = r / s ** 3 * ((count[i] + 40) * 2.0 ** -24 + 4.8e-6 + (np.abs(r - p.rsphere) < 1e-4))
        e += 4 * np.sqrt(3) * (4 * 2.0 ** -24 * n) / s ** 3
        out += np.bincount(i, weights=e, minlength=len(pos))
    return out


@pytest.mark.parametrize("group", [8, 11, 16, 20, 32, 40, 64, 96])
def test_every_target_has_all_its_sources(ctx, group):
    n = 32
    pos = ics.clustered_box(n, halo_fraction=0.1, nhalo=30, seed=group)
    pos = pos[np.random.default_rng(group).permutation(len(pos))[:12000]]
    p = lagpm.make_params(n, theta=1e-6)
    # the force of a pair well inside the split: N times this
    two = np.array([[5.0, 5.0, 5.0], [5.05, 5.0, 5.0]])
    unit = np.abs(orc.pp_direct_analytic(1, n, p.epsilon, p.efold / 2, two, p.rsphere)[0, 0]) * (0.05 ** 2 + 0.1 ** 2) ** 1.5 / 0.05
    acc = []
    for prec in (lagpm.PREC_FP32, lagpm.PREC_FP64):
        with lagpm.Box(ctx, lagpm.make_params(n, precision=prec, theta=1e-6), len(pos)) as b:
            b.set_tuning(8, group, lagpm.GROUPS_RUNS)
            b.upload_pos(pos)
            b.treecorrection(lagpm.evolfact(1.0))
            acc.append(b.velocities())
    err, tol = np.sqrt(((acc[0] - acc[1]) ** 2).sum(axis=1)), unit * bound(pos, p)
    print(f"group {group}: worst error / bound {np.max(err / tol):.3f}, bound / |a| median {np.median(tol / np.sqrt((acc[1] ** 2).sum(axis=1))):.1e}", flush=True)
    assert np.all(err <= tol)
