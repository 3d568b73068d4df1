"""The octree's nodes (first particle, count, children, level, in pre-order) against one built level by
level from the Morton keys in numpy: every node exactly, at the edges of the build's particle blocks
and of its leaf sizes."""
import numpy as np
import pytest

from lageunha_amd import lagpm

pytestmark = pytest.mark.gpu

BITS = 16


def morton(pos, n):
    q = np.minimum(np.floor(pos * (65536.0 / n)), 65535).astype(np.uint64)
    key = np.zeros(len(pos), dtype=np.uint64)
    for b in range(BITS):
        for a in range(3):
            key |= ((q[:, a] >> np.uint64(b)) & np.uint64(1)) << np.uint64(3 * b + a)
    return np.sort(key)


def octree(key, level, nleaf):
    nodes = []

    def visit(lo, hi, l):
        at = len(nodes)
        nodes.append([lo, hi - lo, 0, l])
        if hi - lo > nleaf and l < BITS:
            sub = key[lo:hi] >> np.uint64(3 * (BITS - l - 1))
            cut = np.flatnonzero(np.concatenate([[True], sub[1:] != sub[:-1]])) + lo
            nodes[at][2] = len(cut)
            for a, b in zip(cut, np.append(cut[1:], hi)):
                visit(int(a), int(b), l + 1)

    top = key >> np.uint64(3 * (BITS - level))
    cut = np.flatnonzero(np.concatenate([[True], top[1:] != top[:-1]]))
    for a, b in zip(cut, np.append(cut[1:], len(key))):
        visit(int(a), int(b), level)
    return np.array(nodes)


def points(kind, count, n, g):
    if kind == "uniform":
        return g.random((count, 3)) * n
    centre = g.random((max(1, count // 60), 3)) * n  # clumps down to the finest cells, some coincident
    p = centre[g.integers(0, len(centre), count)] + g.standard_normal((count, 3)) * 10.0 ** g.uniform(-5, 0, (count, 1))
    p[:: 7] = p[0]
    return np.mod(p, n)


# 1024 particles make a block of the build; a leaf of 256 reaches over a quarter of one
@pytest.mark.parametrize("count", [1, 2, 5, 1023, 1024, 1025, 4097, 20000])
@pytest.mark.parametrize("kind", ["uniform", "clumps"])
@pytest.mark.parametrize("nleaf", [4, 16, 256])
@pytest.mark.parametrize("prec", [lagpm.PREC_FP32, lagpm.PREC_FP64])
def test_nodes_are_the_octree(ctx, count, kind, nleaf, prec):
    n = 24
    pos = points(kind, count, n, np.random.default_rng(count))
    with lagpm.Box(ctx, lagpm.make_params(n, precision=prec), count) as b:
        b.set_tuning(nleaf, 64)
        b.upload_pos(pos)
        for _ in range(2):  # the second build is limited to two levels below the first one's deepest
            b.treecorrection(lagpm.evolfact(0.0))
            got = b.tree_nodes()
            want = octree(morton(pos, n), 2, nleaf)
            assert np.array_equal(got["info"], want)
            assert np.array_equal(got["com"][:, 3], want[:, 1].astype(np.float64))
            st = b.tree_stats()
            assert st.n_nodes == len(want) and st.deepest == want[:, 3].max()
