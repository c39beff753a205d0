"""The 8-step conduction operator is no less accurate than per-node FP32 steps."""
import numpy as np
import pytest

from binarytpm_amd import inputs
from binarytpm_amd import thermal as th
from oracle import oracle as O

pytestmark = pytest.mark.gpu

NROT, NF = 30, 72
TIS = (20.0, 70.0, 200.0, 500.0, 1000.0)
# 360 columns whose errors are independent of each other give an rms good to
# 1 / sqrt(2 x 360) = 3.7 %, the ratio of two to 5.3 %: three of those and the
# half a percent that rounding the results to FP32 can add
RATIO = 1.17


@pytest.mark.parametrize("n", [1.0, 0.266, 0.0634, 0.0317, 0.0099])
def test_error_against_fp64(ctx, n):
    """FTCS numbers 0.47 to 0.005.  A shape of one spin rate runs on the
    operator; the same facets beside eight of other rates run step by step
    (facets without exchange do not see each other)."""
    case = inputs.config0(subdiv=1, ntau=650)
    kw = dict(max_rev=NROT, check_after=NROT)
    p, po = th.params(650, case.rot_period, **kw), O.params(650, case.rot_period, **kw)
    one = np.full(80, n, np.float32)
    many = one.copy()
    many[NF:] = n * np.linspace(0.5, 0.9, 80 - NF)
    errs = []
    for ti in TIS:
        ref = O.smooth_solve(po, case.illum[:NF], 0.1, ti, numrevs=one[:NF])
        row = []
        for nr in (one, many):
            shape = th.Shape(ctx, p, case.illum, 0.1, numrevs=nr)
            s = th.Solve(ctx, shape, ti).run()
            row += [s.surface_temps()[:NF] - ref.stemp, s.profile()[:NF] - ref.temp]
            s.close()
            shape.close()
        errs.append(row)
    rms = [np.sqrt(np.mean(np.concatenate([e[k].ravel() for e in errs]) ** 2)) for k in range(4)]
    print("[parity] r %.4f: rms error surface %.2e (steps %.2e), profile %.2e (steps %.2e)"
          % (0.47366 * n, rms[0], rms[2], rms[1], rms[3]), flush=True)
    assert rms[0] <= RATIO * rms[2]
    assert rms[1] <= RATIO * rms[3]
