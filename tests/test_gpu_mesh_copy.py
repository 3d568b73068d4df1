"""Host copies of the padded mesh: the density against the raw fixed-point accumulator, and a
potential set from the host against numpy's FDA4 gradient of it."""
import numpy as np
import pytest

from lageunha_amd import lagpm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [8, 9, 27, 32, 50, 65])  # rows padded to n + 2 (even n) and n + 1 (odd n)
@pytest.mark.parametrize("precision", [lagpm.PREC_FP32, lagpm.PREC_FP64])
def test_density_and_potential_copies(ctx, n, precision):
    g = np.random.default_rng(n)
    pos = g.random((n ** 3 // 2, 3)) * n
    phi = g.normal(size=(n, n, n)).astype(np.float32)  # [z][y][x]
    with lagpm.Box(ctx, lagpm.make_params(n, precision=precision, rsphere=min(5.0, n / 4)), len(pos)) as b:
        b.upload_pos(pos)
        den = b.tsc()
        acc, bits = b.tsc_fixed()
        want = acc.astype(np.float64) * 2.0 ** -bits - 1.0  # exact, then one subtraction
        assert np.array_equal(den.ravel(), want.astype(np.float32))
        b.set_potential(phi)
        b.fda4(lagpm.evolfact(0.0), lagpm.KICK)
        grad = b.get_gradient()
    assert np.array_equal(grad[:, 3], phi.ravel())
    p = phi.astype(np.float64)
    for c, ax in enumerate((2, 1, 0)):
        d = (2 / 3) * (np.roll(p, 1, ax) - np.roll(p, -1, ax)) - (np.roll(p, 2, ax) - np.roll(p, -2, ax)) / 12
        # five roundings of terms of at most 2 max|phi|, in FP32
        assert np.abs(grad[:, c] - d.ravel()).max() <= 5 * 2.0 ** -23 * 2 * np.abs(p).max()
