"""GOTPM records decoded and encoded on the device against the host functions of the C ABI
(lagpm_eunha_decode / lagpm_eunha_encode: XofP, eunha.h:1212, 1228-1232)."""
import numpy as np
import pytest

from lageunha_amd import lagpm

pytestmark = pytest.mark.gpu


def make_records(n, count, seed):
    """Sites anywhere in the index word (beyond the lattice and above 32 bits too), a flag byte on
    top, displacements beyond the box either way, exact zeros and box lengths among them."""
    g = np.random.default_rng(seed)
    rec = np.zeros(count, dtype=lagpm.DM_RECORD)
    idx = g.integers(0, n ** 3, count, dtype=np.uint64)
    far = g.random(count) < 0.2
    idx[far] = g.integers(0, 1 << 56, int(far.sum()), dtype=np.uint64)
    rec["u4if"] = idx | (g.integers(0, 256, count, dtype=np.uint64) << np.uint64(56))
    for a in "xyz":
        rec[a] = g.normal(0, 3, count)
        rec["v" + a] = g.normal(0, 1, count)
    edge = g.random(count) < 0.2
    rec["x"][edge] = g.choice([0.0, -0.0, -1e-8, n, -n, -2.5 * n, 3.0 * n], int(edge.sum()))
    return rec


# a quarter of the records passes through one scratch array: counts around multiples of four
@pytest.mark.parametrize("count", [1, 2, 3, 4, 5, 255, 257, 4097, 70001])
@pytest.mark.parametrize("precision", [lagpm.PREC_FP32, lagpm.PREC_FP64])
def test_upload_decodes_as_the_host_does(ctx, count, precision):
    n = 24
    rec = make_records(n, count, count)
    pos, vel = lagpm.eunha_decode(rec, n)
    pos = np.where(pos < 0, pos + n, pos)  # every upload wraps into [0, n)
    pos[pos >= n] = 0.0
    with lagpm.Box(ctx, lagpm.make_params(n, precision=precision), count) as b:
        b.upload_eunha(rec)
        got, gv = b.download()
    assert np.array_equal(got, pos) and np.array_equal(gv, vel)


@pytest.mark.parametrize("count", [1, 2, 3, 5, 255, 257, 70001])
@pytest.mark.parametrize("precision", [lagpm.PREC_FP32, lagpm.PREC_FP64])
def test_download_encodes_as_the_host_does(ctx, count, precision):
    """After a sort (the box's order is not the caller's), into records with other sites than the
    uploaded ones; every byte of the records, kept fields included."""
    n = 24
    rec = make_records(n, count, count + 1)
    into = make_records(n, count, count + 2)
    into["x"][::3] = np.float32(np.nan)  # overwritten by a full download, kept by a velocity one
    with lagpm.Box(ctx, lagpm.make_params(n, precision=precision), count) as b:
        b.upload_eunha(rec)
        b.pmmain(lagpm.evolfact(1.0), lagpm.KICK)
        b.drift(0.7)
        pos, vel = b.download()
        for full in (True, False):
            want, got = into.copy(), into.copy()
            if full:
                lagpm.eunha_encode(want, n, pos, vel)
                b.download_eunha(got)
            else:
                for c, a in enumerate("xyz"):
                    want["v" + a] = vel[:, c].astype(np.float32)
                b.download_eunha_vel(got)
            assert got.tobytes() == want.tobytes()
