"""The operator's smooth kernels at 16, 32 and 64 columns per wave: results bit for
bit alike where tiles are partly filled, and what the tuner keeps a width for."""
import numpy as np
import pytest

from binarytpm_amd import inputs
from binarytpm_amd import thermal as th

pytestmark = pytest.mark.gpu


def _run(c, shape, tis, tune):
    s = [th.Solve(c, shape, t) for t in tis]
    st = th.batch_run(c, s, th.batch_opts(autotune=tune))
    out = [(x.surface_temps(), x.profile()) for x in s]
    for x in s:
        x.close()
    return st, out


@pytest.mark.parametrize("nf", [1, 17, 33, 63, 65])
@pytest.mark.parametrize("ntau", [617, 650, 624])
@pytest.mark.parametrize("rates", [1, 3])
def test_widths_bitwise(nf, ntau, rates):
    """A trial runs each width twice (rotations at 16, 32, 64, 64, 32, 16
    columns per wave), untuned rotations are all 16 wide."""
    case = inputs.config0(subdiv=1, ntau=ntau)
    p = th.params(ntau, case.rot_period, max_rev=10, check_after=10)
    nr = (1.0 - 0.2 * (np.arange(nf) * 7 % 5 % rates)).astype(np.float32)
    out = []
    for tune in (False, True):
        with th.Context(0) as c:
            shape = th.Shape(c, p, case.illum[:nf], 0.1, numrevs=nr)
            st, o = _run(c, shape, [150.0], tune)
            assert st.tune_rotations == (6 if tune else 0)
            out.append(o[0])
            shape.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def test_wide_default_bitwise(ctx):
    """More columns than the 16-wide form is used for, in sets of 65 + ragged."""
    case = inputs.config0(subdiv=1, ntau=617)
    p = th.params(617, case.rot_period, max_rev=4, check_after=4)
    shape = th.Shape(ctx, p, case.illum[:65], 0.1)
    tis = np.linspace(20.0, 900.0, 330)
    many = _run(ctx, shape, tis, False)[1]
    for k in (0, 164, 329):
        one = _run(ctx, shape, tis[k:k + 1], False)[1][0]
        assert np.array_equal(one[0], many[k][0]) and np.array_equal(one[1], many[k][1])
    shape.close()


def test_tuned_by_load():
    """A width kept for some load is not taken for four times as much, and sets
    of different sizes that share a launch share a trial."""
    ntau, nf = 650, 5120
    rng = np.random.default_rng(3)
    illum = rng.random((nf, ntau), dtype=np.float32) * 1300.0
    # a chunk of 4 rotations before the trial, 6 in it
    p = th.params(ntau, 20000.0, max_rev=12, check_after=12)
    with th.Context(0) as c:
        big, small = th.Shape(c, p, illum, 0.1), th.Shape(c, p, illum[:640], 0.1)
        trials = []
        for shapes in ([big] * 5, [big] * 5, [big] * 20, [small, small], [small, big]):
            s = [th.Solve(c, sh, 100.0 + 10.0 * k) for k, sh in enumerate(shapes)]
            st = th.batch_run(c, s, th.batch_opts(autotune=True))
            trials.append((st.tune_decisions, st.tune_rotations))
            for x in s:
                x.close()
        assert trials == [(1, 6), (0, 0), (1, 6), (1, 6), (0, 0)]
        big.close()
        small.close()
