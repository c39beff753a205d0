"""The conduction kernels on the 8-step operator (linear_block.h) at the sizes
where their tiles and blocks end: columns per wave and craters per workgroup,
and cycles whose last time block has 1 to 8 steps."""
import numpy as np
import pytest

from binarytpm_amd import inputs
from binarytpm_amd import thermal as th
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# Nine rotations without freezing are a continuous function of the inputs.  A
# block rounds an offset of at most 200 K to FP32 (half an ulp: 7.6e-6 K) and
# the temperature itself to half an ulp of 300 K (1.5e-5 K); 9 x 82 blocks
# whose roundings add like a random walk give 7.6e-6 x sqrt(738) + 1.5e-5.
TOL = 2.3e-4


@pytest.fixture(scope="module")
def rough80():
    return inputs.rough_primary(subdiv=1)          # 80 facets x 100 sub-facets


def _fixed(ntau, period, nrot):
    kw = dict(max_rev=nrot, check_after=nrot)
    return th.params(ntau, period, **kw), O.params(ntau, period, **kw)


@pytest.mark.parametrize("nf", [1, 15, 17, 33, 64, 80])
@pytest.mark.parametrize("ntau", [617, 650, 655, 624])
def test_smooth_edges(ctx, nf, ntau):
    case = inputs.config0(subdiv=1, ntau=ntau)
    illum = case.illum[:nf]
    p, po = _fixed(ntau, case.rot_period, 9)
    with th.Context(0) as c:
        shape = th.Shape(c, p, illum, 0.1)
        s = th.Solve(c, shape, 150.0)
        th.batch_run(c, [s], th.batch_opts(autotune=False))
        ref = O.smooth_solve(po, illum, 0.1, 150.0)
        assert np.abs(s.surface_temps() - ref.stemp).max() <= TOL
        assert np.abs(s.profile() - ref.temp).max() <= TOL
        s.close()
        shape.close()


@pytest.mark.parametrize("ntau", [8, 5])
def test_slow_spin_rates(ctx, ntau):
    """Cycles of a block or less (numrevs small enough for a stable step)."""
    case = inputs.config0(subdiv=1, ntau=ntau)
    nr = np.full(80, 0.005, np.float32)
    p, po = _fixed(ntau, case.rot_period, 9)
    shape = th.Shape(ctx, p, case.illum, 0.1, numrevs=nr)
    s = th.Solve(ctx, shape, 150.0).run()
    ref = O.smooth_solve(po, case.illum, 0.1, 150.0, numrevs=nr)
    assert np.abs(s.surface_temps() - ref.stemp).max() <= TOL
    assert np.abs(s.profile() - ref.temp).max() <= TOL
    s.close()
    shape.close()


@pytest.mark.parametrize("ntau", [650, 617])
def test_widths_bitwise(ctx, rough80, ntau):
    """A column's arithmetic does not depend on what shares its wave or
    workgroup: solves alone (two craters per workgroup) equal the same solves
    in a batch with more craters than the wide form starts at (five), with
    remainders in both."""
    case, crater = rough80
    nf = 77
    p, _ = _fixed(ntau, case.rot_period, 8)
    illum = np.ascontiguousarray(case.illum[:nf, :ntau])
    cm = th.CraterModel(vf=crater["vf"], solar=crater["solar"],
                        shadow=np.ascontiguousarray(crater["shadow"][:nf, :ntau]),
                        cosang=np.ascontiguousarray(crater["cosang"][:nf, :ntau]))
    shape = th.Shape(ctx, p, illum, 0.1, crater=cm)
    tis = np.linspace(40.0, 700.0, 7)
    many = [th.Solve(ctx, shape, t, with_craters=True) for t in tis]
    th.batch_run(ctx, many, th.batch_opts(autotune=False))
    for t, m in list(zip(tis, many))[::3]:
        one = th.Solve(ctx, shape, t, with_craters=True).run()
        assert np.array_equal(one.surface_temps(), m.surface_temps())
        assert np.array_equal(one.crater_temps(), m.crater_temps())
        assert np.array_equal(one.crater_profile(), m.crater_profile())
        one.close()
    for m in many:
        m.close()
    shape.close()


@pytest.mark.parametrize("rates", [(0.5, 1.0), (1.0, 0.5, 0.25), tuple(np.linspace(0.25, 1.0, 8))])
@pytest.mark.parametrize("nf", [9, 77])
def test_spin_rate_classes_bitwise(ctx, rough80, rates, nf):
    """Without exchange between facets, facets of several spin rates in one
    shape equal the same facets in shapes of one rate each."""
    case, crater = rough80
    rng = np.random.default_rng(nf + len(rates))
    pick = rng.integers(0, len(rates), nf)
    p, _ = _fixed(650, case.rot_period, 8)
    cm = th.CraterModel(vf=crater["vf"], solar=crater["solar"],
                        shadow=crater["shadow"][:nf], cosang=crater["cosang"][:nf])
    illum = case.illum[:nf]

    def run(numrevs):
        shape = th.Shape(ctx, p, illum, 0.1, numrevs=numrevs.astype(np.float32), crater=cm)
        s = th.Solve(ctx, shape, 150.0, with_craters=True).run()
        out = (s.surface_temps(), s.profile(), s.crater_temps(), s.crater_profile())
        s.close()
        shape.close()
        return out

    mixed = run(np.asarray(rates)[pick])
    for k, r in enumerate(rates):
        for m, u in zip(mixed, run(np.full(nf, r))):
            assert np.array_equal(m[pick == k], u[pick == k])


def test_many_spin_rates(ctx):
    """More rates than operators are kept for."""
    case = inputs.config0(subdiv=1, ntau=650)
    nr = np.linspace(0.3, 1.0, 80).astype(np.float32)
    p, po = _fixed(650, case.rot_period, 9)
    shape = th.Shape(ctx, p, case.illum, 0.1, numrevs=nr)
    s = th.Solve(ctx, shape, 150.0).run()
    ref = O.smooth_solve(po, case.illum, 0.1, 150.0, numrevs=nr)
    assert np.abs(s.surface_temps() - ref.stemp).max() <= TOL
    assert np.abs(s.profile() - ref.temp).max() <= TOL
    s.close()
    shape.close()
