"""Copies through the pinned slices: results equal those of small shapes, whose
copies go by the runtime, on both sides of the sizes where the slices start
(4 MB to the host, 16 MB to the device) and over several slices."""
import numpy as np
import pytest
import torch

from binarytpm_amd import thermal as th

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nf", [1613, 1614, 6452, 6453, 25811, 60013])
def test_sizes(ctx, nf):
    ntau = 650
    p = th.params(ntau, 20000.0)
    illum = np.random.default_rng(nf).random((nf, ntau), dtype=np.float32) * 1300.0
    shape = th.Shape(ctx, p, illum, 0.1)
    got = shape.facet_illum()
    shape.close()
    for f0 in list(range(0, nf, 9001)) + [nf - 7]:
        part = th.Shape(ctx, p, illum[f0:f0 + 7], 0.1)
        assert np.array_equal(got[f0:f0 + 7], part.facet_illum())
        part.close()


def test_pinned(ctx):
    ntau, nf = 650, 6500
    p = th.params(ntau, 20000.0)
    pinned = torch.empty((nf, ntau), pin_memory=True)
    pinned.uniform_(0.0, 1300.0)
    a = th.Shape(ctx, p, pinned.numpy(), 0.1)
    b = th.Shape(ctx, p, pinned.numpy().copy(), 0.1)
    assert np.array_equal(a.facet_illum(), b.facet_illum())
    a.close()
    b.close()
