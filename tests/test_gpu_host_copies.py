"""Host copies around the size where they go through the pinned slots (2 MB in all) and around a
slot's 2 MB: what goes up comes back, in the caller's order."""
import numpy as np
import pytest

from lageunha_amd import lagpm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1000, 43690, 43691, 65536, 65537, 262143, 262144, 262145, 1500007])
def test_particles_up_and_down(ctx, count):
    n = 64
    g = np.random.default_rng(count)
    pos, vel = g.random((count, 3)) * n, g.normal(size=(count, 3))
    with lagpm.Box(ctx, lagpm.make_params(n), count) as b:
        for sort in (False, True):
            b.upload_pos(pos, vel)
            if sort:
                b.pmmain(lagpm.evolfact(0.0), lagpm.KICK)
            p, v = b.download()
            assert np.array_equal(p, pos) and np.array_equal(v, vel)
        b.upload_pos(pos)  # no velocities: zero
        assert not b.velocities().any()


@pytest.mark.parametrize("n", [62, 64, 80, 82])  # 64^3 int64 = 2 MB, 80^3 floats just below 2 MB
def test_meshes_down(ctx, n):
    g = np.random.default_rng(n)
    pos = g.random((n ** 3 // 4, 3)) * n
    with lagpm.Box(ctx, lagpm.make_params(n), len(pos)) as b:
        b.upload_pos(pos)
        den = b.tsc()
        acc, bits = b.tsc_fixed()
        assert np.array_equal(den.ravel(), (acc * 2.0 ** -bits - 1.0).astype(np.float32))
        b.set_potential(den)
        b.fda4(lagpm.evolfact(0.0), lagpm.KICK)
        assert np.array_equal(b.get_gradient()[:, 3], den.ravel())
