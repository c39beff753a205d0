"""Results into pinned buffers, which go by DMA alone, equal those into pageable
ones, which go through the pinned slices."""
import numpy as np
import pytest
import torch

from binarytpm_amd import thermal as th

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nf", [1000, 6500])    # 2.6 MB: no slices; 16.9 MB
def test_results_into_pinned(ctx, nf):
    ntau = 650
    illum = np.random.default_rng(nf).random((nf, ntau), dtype=np.float32) * 1300.0
    shape = th.Shape(ctx, th.params(ntau, 20000.0, max_rev=2), illum, 0.1)
    s = th.Solve(ctx, shape, 200.0).run()
    want = s.surface_temps()
    whole = torch.full((nf * ntau + 24,), -1.0, pin_memory=True).numpy()
    for first in (0, 8, 17):                    # the buffer's start, and inside it
        whole[:] = -1.0
        s.surface_temps(out=whole[first:first + nf * ntau].reshape(nf, ntau))
        assert np.array_equal(whole[first:first + nf * ntau].reshape(nf, ntau), want)
        assert (whole[:first] == -1.0).all() and (whole[first + nf * ntau:] == -1.0).all()
    s.close()
    shape.close()
