"""The deposit's runs of particles in one mesh cell (added up node by node instead of by atomics):
run lengths around the shortest one taken, half a wave, a wave and a chunk, each followed by
particles of other cells, at shifted places in the wave. The sums are integers: exact, FP32 weights
against the oracle, FP64 against the same products in numpy."""
import numpy as np
import pytest

from lageunha_amd import lagpm
from oracle import pyoracle as orc

pytestmark = pytest.mark.gpu


def _axis64(x):
    r = np.rint(x)
    d = x - r
    s = np.where(np.signbit(d), -1, 1)
    d = np.abs(d)
    w0 = 0.75 - d * d
    w2 = 0.5 * (0.25 + d * (d - 1.0))
    return r.astype(np.int64), s, (w0, w2 + d, w2)


def _fixed64(n, pos, bits):
    acc = np.zeros(n ** 3, dtype=np.int64)
    ax = [_axis64(pos[:, a]) for a in range(3)]
    off = lambda a, k: (ax[a][0] + (0, ax[a][1], -ax[a][1])[k]) % n
    for c in range(3):
        for b in range(3):
            for a in range(3):
                w = 1.0 * ax[0][2][a] * ax[1][2][b] * ax[2][2][c]
                np.add.at(acc, off(0, a) + n * (off(1, b) + n * off(2, c)), np.rint(w * 2.0 ** bits).astype(np.int64))
    return acc


@pytest.mark.parametrize("prec", [lagpm.PREC_FP32, lagpm.PREC_FP64])
@pytest.mark.parametrize("run", [1, 7, 8, 9, 10, 31, 33, 63, 64, 65, 129, 1025])
def test_runs_of_one_cell(ctx, run, prec):
    n = 24
    g = np.random.default_rng(run)
    pos = [g.random((g.integers(1, 5), 3)) * n]
    for cell in [(0, 0, 0), (3, 3, 3), (3, 3, 4), (11, 12, 13), (23, 23, 23), (24, 7, 24)]:
        pos.append((np.array(cell) + g.uniform(-0.5, 0.5, (run, 3))) % n)  # every octant around the node
        pos.append((np.array(cell) + 0.25 + 0.1 * g.random((run, 3))) % n)  # one octant
        pos.append(g.random((5, 3)) * n)
    pos = np.concatenate(pos)
    with lagpm.Box(ctx, lagpm.make_params(n, precision=prec), len(pos)) as b:
        b.upload_pos(pos)
        acc, bits = b.tsc_fixed()
    if prec == lagpm.PREC_FP32:
        want, obits = orc.tsc_fixed(n, pos, mass=1.0)
        assert bits == obits
    else:
        want = _fixed64(n, pos, bits)
    assert np.array_equal(acc, want)
