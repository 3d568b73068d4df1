"""The FP64 walk's paths: teams of four waves and single ones, leaves of more particles than one
expansion takes, groups of one to 128 targets, and deep trees."""
import numpy as np
import pytest

from lageunha_amd import lagpm
from oracle import pyoracle as orc

pytestmark = pytest.mark.gpu


def kick(ctx, p, pos, tuning=None):
    with lagpm.Box(ctx, p, len(pos)) as b:
        if tuning:
            b.set_tuning(*tuning)
        b.upload_pos(pos)
        b.treecorrection(lagpm.evolfact(1.0))
        return b.velocities()


def relerr(a, b):
    return float(np.sqrt(np.sum((a - b) ** 2) / np.sum(b ** 2)))


# 2049 and 5000 coincident particles: a leaf beyond the 2048 of one expansion, several groups of it
@pytest.mark.parametrize("coincident", [1, 40, 2048, 2049, 5000])
@pytest.mark.parametrize("tuning", [(16, 64, 0), (32, 128, 0), (4, 8, 0), (16, 96, 2)])
def test_theta_zero_is_the_direct_sum(ctx, coincident, tuning):
    n = 24
    g = np.random.default_rng(coincident)
    pos = np.concatenate([np.full((coincident, 3), 7.25), (g.random((3000, 3)) * n)])
    tight = 11.0 + g.standard_normal((300, 3)) * 1e-3  # full key depth below it
    pos = np.concatenate([pos, tight]) % n
    p = lagpm.make_params(n, precision=lagpm.PREC_FP64, theta=1e-6)
    ref = orc.pp_direct_analytic(1, n, p.epsilon, p.efold / 2, pos, p.rsphere)
    assert relerr(kick(ctx, p, pos, tuning), ref) < 1e-5  # the force table's interpolation


@pytest.mark.parametrize("count", [300000, 300001])  # teams of four up to 300000 targets
@pytest.mark.parametrize("theta", [1e-6, 0.5])
def test_teams_agree_with_the_fp32_walk(ctx, count, theta):
    n = 64
    pos = np.random.default_rng(5).random((count, 3)) * n
    a = kick(ctx, lagpm.make_params(n, precision=lagpm.PREC_FP64, theta=theta), pos)
    b = kick(ctx, lagpm.make_params(n, theta=theta), pos)
    assert relerr(b, a) < 1e-4  # the bound of the FP32 walk against the FP64 one
