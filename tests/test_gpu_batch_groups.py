"""The default grouping of a batch step (lagpm_set_batch_pipeline not called): one box, too few boxes
for two groups, the smallest counts of two and three groups. Every box gets the bits that one
group of all boxes gives it."""
import numpy as np
import pytest

from lageunha_amd import ics, lagpm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nbox", [1, 5, 6, 9, 10])
def test_default_groups_equal_one_group(nbox):
    sizes = [24, 32, 28, 36, 24, 32, 28, 24, 32, 36][:nbox]
    pos = [ics.clustered_box(n, halo_fraction=0.3, nhalo=3, seed=i) for i, n in enumerate(sizes)]
    out = []
    for stages in (0, 1):
        ctx = lagpm.Context(0)
        if stages:
            ctx.set_batch_pipeline(stages)
        boxes = [lagpm.Box(ctx, lagpm.make_params(n), len(p)) for n, p in zip(sizes, pos)]
        for b, p in zip(boxes, pos):
            b.upload_pos(p)
        for s in range(2):
            lagpm.batch_step(ctx, boxes, 1.0 + 0.01 * s, 0.01)
        out.append([b.download() for b in boxes])
        for b in boxes:
            b.close()
        ctx.close()
    for (xa, va), (xb, vb) in zip(*out):
        assert np.array_equal(xa, xb) and np.array_equal(va, vb)
