"""PreFoF's sub-cells (lagpm_prefof): links just at, above and below the values where the number of
sub-cells per cell changes, and below the smallest one whose sub-cells are single sets; coincident
particles, lattices spaced by the link, pairs in opposite corners of a sub-cell; a particle without a
position. The flags are whole numbers: they equal the oracle's."""
import numpy as np
import pytest

from lageunha_amd import lagpm
from oracle import pyoracle as orc

pytestmark = pytest.mark.gpu

SQ3 = 3.0 ** 0.5


def _flags(ctx, n, pos, link, minnum):
    with lagpm.Box(ctx, lagpm.make_params(n), len(pos)) as b:
        b.upload_pos(pos)
        return b.prefof(link, minnum)


@pytest.mark.parametrize("link", [0.004, 4 * SQ3 / 1024, 0.0069, 0.05, 4 * SQ3 / 35, 0.25, 0.5, 1.0, 2.0, 4 * SQ3 / 3, 4 * SQ3, 30.0])
@pytest.mark.parametrize("scale", [1.0 - 2e-7, 1.0, 1.0 + 2e-7])
def test_flags_where_the_sub_cells_change(ctx, link, scale):
    n = 18
    link = float(np.float32(link * scale))
    g = np.random.default_rng(int(1000 * link) + 1)
    step = min(link, 1.0)
    lattice = np.stack(np.meshgrid(*[np.arange(4) * step] * 3), -1).reshape(-1, 3) + [4.0, 4.0, 4.0]
    blob = 6.0 + step * g.normal(size=(400, 3))  # a dense knot: several links wide
    side = 4.0 / np.ceil(4 * SQ3 / link)
    corners = np.concatenate([[[8.0, 8.0, 0.0]], [[8.0, 8.0, 0.0] + np.full(3, side * (1 - 1e-12))]])
    same = np.tile([[1.0, 1.0, 1.0]], (30, 1))
    pos = np.concatenate([lattice, blob, corners, same, g.random((300, 3)) * n]) % n
    pos = pos[g.permutation(len(pos))]
    got, cnt = _flags(ctx, n, pos, link, 5)
    want, wcnt = orc.prefof(n, pos, link, 5)
    assert cnt == wcnt and np.array_equal(got, want)


def test_a_particle_without_position_is_linked_to_none(ctx):
    g = np.random.default_rng(3)
    pos = 2.0 + 0.02 * g.random((40, 3))
    bad = pos.copy()
    bad[::7, 1] = np.nan
    got, cnt = _flags(ctx, 16, bad, 0.2, 35)
    rest = np.isfinite(bad).all(axis=1)
    want, _ = orc.prefof(16, bad[rest], 0.2, 35)
    assert np.array_equal(got[rest], want) and cnt == int(got.sum())


@pytest.mark.parametrize("n,np_", [(128, 1), (128, 12), (64, 700)])
def test_few_particles_in_a_large_box_and_the_box_afterwards(ctx, n, np_):
    """The table of cells is larger than the box's own scratch; the box's particles are as they were."""
    g = np.random.default_rng(np_)
    pos = (8.0 + 0.3 * g.random((np_, 3))) % n
    vel = g.normal(size=(np_, 3))
    want, wcnt = orc.prefof(n, pos, 0.2, 5)
    with lagpm.Box(ctx, lagpm.make_params(n), np_) as b:
        b.upload_pos(pos, vel)
        got, cnt = b.prefof(0.2, 5)
        pos2, vel2 = b.download()
    assert cnt == wcnt and np.array_equal(got, want)
    assert np.array_equal(pos2, pos) and np.array_equal(vel2, vel)
