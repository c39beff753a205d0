"""Shapes of more spin rates than conduction operators are kept for: the
kernels that integrate node by node, through the scheduler, against the FP64
oracle.  37 facets fill crater workgroups of 10 + 10 + 10 + 7, each with
several rates in it."""
import numpy as np
import pytest

from binarytpm_amd import inputs
from binarytpm_amd import thermal as th
from oracle import oracle as O

pytestmark = pytest.mark.gpu
TOL_K = 0.05       # the stage's stated tolerance
NF = 37


def _rates(nf, top=1.0):
    return np.random.default_rng(nf).permutation(np.linspace(0.4, top, 11)[np.arange(nf) % 11])


def _case(ctx, ntau, nf=NF):
    case, crater = inputs.rough_primary(subdiv=1, ntau=ntau)
    sh, co = (np.ascontiguousarray(crater[k][:nf]) for k in ("shadow", "cosang"))
    nr = _rates(nf).astype(np.float32)
    cm = th.CraterModel(vf=crater["vf"], shadow=sh, cosang=co, solar=crater["solar"],
                        multiple=True, scatter_acc=1e-4)
    shape = th.Shape(ctx, th.params(ntau, case.rot_period, tacc=0.01), case.illum[:nf], 0.1,
                     numrevs=nr, crater=cm)
    po = O.params(ntau, case.rot_period, tacc=0.01)
    zero = np.zeros((nf, ntau, 100))
    il = O.crater_scatter(crater["vf"], 0.1, sh, co, zero, crater["solar"], multiple=True, acc=1e-4)
    return case, crater, nr, shape, po, il, zero


# r of the fastest facet: 0.49980 (the scale is folded back every block),
# 0.48870 (every second) and 0.47366 (every third)
@pytest.mark.parametrize("ntau", [616, 630, 650])
def test_parity(ctx, ntau):
    case, crater, nr, shape, po, il, zero = _case(ctx, ntau)
    s = th.Solve(ctx, shape, 200.0, with_craters=True).run()
    sm = O.smooth_solve(po, case.illum[:NF], 0.1, 200.0, numrevs=nr)
    cr = O.crater_solve(po, crater["vf"], 0.1, 200.0, il, zero, numrevs=nr)
    info = s.info()
    assert info.converged and info.crater_converged
    d = [np.abs(s.surface_temps() - sm.stemp).max(), np.abs(s.crater_temps() - cr.stemp).max()]
    print(f"[parity] 11 rates, ntau {ntau}: smooth {d[0]:.5f} K, craters {d[1]:.5f} K", flush=True)
    assert max(d) <= TOL_K
    assert abs(info.rotations - sm.rotations) <= 1
    assert abs(info.crater_rotations - cr.rotations) <= 1
    s.close()
    shape.close()


def test_ti0(ctx):
    case, crater, nr, shape, po, il, zero = _case(ctx, 650)
    s = th.Solve(ctx, shape, 0.0, with_craters=True).run()
    sm = O.smooth_solve(po, case.illum[:NF], 0.1, 0.0, numrevs=nr)
    cr = O.crater_solve(po, crater["vf"], 0.1, 0.0, il, zero, numrevs=nr,
                        temp=np.zeros((NF, 57, 100)), stemp=np.zeros(il.shape))
    assert np.abs(s.surface_temps() - sm.stemp).max() <= TOL_K
    assert np.abs(s.crater_temps() - cr.stemp).max() <= TOL_K
    s.close()
    shape.close()


@pytest.mark.parametrize("nf", [63, 65, 80])
def test_tuned_equals_untuned(nf):
    """256, 128 and 64 columns per workgroup, each twice in the trial."""
    out = []
    for tune in (True, False):
        with th.Context(0) as c:  # a fresh context: nothing tuned yet
            case, _, _, shape, _, _, _ = _case(c, 650, nf)
            s = th.Solve(c, shape, 200.0, with_craters=True)
            st = th.batch_run(c, [s], th.batch_opts(autotune=tune))
            assert st.tune_rotations == (6 if tune else 0)
            out.append((s.surface_temps(), s.profile(), s.crater_temps(), s.crater_profile()))
            s.close()
            shape.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
