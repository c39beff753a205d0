"""Initialisation of smooth sets of more columns than its launch has room for at
a time (16384 workgroups of 8 columns)."""
import numpy as np
import pytest

from binarytpm_amd import thermal as th

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nf", [131072, 131073, 300001])
def test_initial_temperatures(ctx, nf):
    """A column whose flux does not change over the cycle starts at its
    equilibrium and stays there; TI 0 would not show the start."""
    ntau = 20
    # 17 levels, so that neighbours and the columns a pass apart differ
    flux = (100.0 + 50.0 * (np.arange(nf) % 17)).astype(np.float32)
    p = th.params(ntau, 20000.0, max_rev=1)
    shape = th.Shape(ctx, p, np.repeat(flux[:, None], ntau, 1), 0.1,
                     numrevs=np.full(nf, 0.03, np.float32))
    s = th.Solve(ctx, shape, 200.0).run()
    want = (0.9 * flux.astype(np.float64) / (0.95 * 5.67e-8)) ** 0.25
    # FP32 temperatures up to 400 K: an ulp is 3.1e-5 K; the start, the balance
    # of each of 20 steps and the FP32 flux and emissivity (1.2e-7 of T / 4) add
    # at most a few
    assert np.abs(s.surface_temps() - want[:, None]).max() <= 3e-4
    assert np.abs(s.profile() - want[:, None]).max() <= 3e-4
    s.close()
    shape.close()
