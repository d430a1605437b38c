"""GDsteady's kernels with more work-groups than compute units (half the threads for each then),
and runs of adhesion that pass the ends of the wavefronts which measure them.

Tolerances: a patch's sums keep their order whichever patches share its launches: equal bits.
Against the oracle as both stop at eps 1e-11 of the traction's rms with a mean rate of convergence
of about 0.9 a sweep: 1e-8 of the largest pressure.
"""
import numpy as np
import pytest

from contact_amd import workloads as W

pytestmark = pytest.mark.gpu


def case(mx, my, eps=1e-11):
    c = dict(fn=9e4, cksi=-4e-4, ceta=3e-4, cphi=1e-4) if mx < 50 else dict(fn=2e4, cksi=-1e-4, ceta=6e-5, cphi=0.0)
    return W.base_case(tang=3, norm=1, eps=eps, ipotcn=-3, mx=mx, my=my, aa=6.0, bb=6.0 * min(1.0, 1.5 * my / mx),
                       scale=max(1.3, min(mx, my) / (min(mx, my) - 3.0)), **c)


def test_more_groups_than_compute_units(cntc):
    c = case(10, 9, 1e-8)
    n, one = 300, 600
    for k in range(n + 1):
        W.apply_case(cntc, one + k, 1, c)
    assert cntc.calculate(one, 1) == 0
    err = cntc.calculatebatch(list(range(one + 1, one + n + 1)), [1] * n)
    want = [a.tobytes() for a in cntc.gettractions(one, 1)]
    its = cntc.getiterations(one, 1)
    got = [([a.tobytes() for a in cntc.gettractions(one + k, 1)], cntc.getiterations(one + k, 1)) for k in range(1, n + 1)]
    for k in range(n + 1):
        cntc.finalize(one + k)
    print("iterations", its)
    assert its[3] > 5 and not np.any(err)
    assert all(g[0] == want and g[1][:4] == its[:4] for g in got)


@pytest.mark.parametrize("mx,my", [(90, 12), (150, 9), (210, 8)])
def test_long_adhesion(cntc, oracle, mx, my):
    c = case(mx, my)
    ire = 943
    W.apply_case(cntc, ire, 1, c)
    assert cntc.calculate(ire, 1) == 0
    p = [a.ravel() for a in cntc.gettractions(ire, 1)]
    its = cntc.getiterations(ire, 1)
    el = cntc.getelementdivision(ire, 1).reshape(my, mx)
    cntc.finalize(ire)
    rc, of, P = oracle.solve_case(c)
    assert rc == 0
    print(mx, my, "longest adhesion", (el == 1).sum(1).max(), "iterations", its, P.iters())
    assert (el == 1).sum(1).max() > 64
    for a, b in zip(p, P.tractions()):
        assert np.abs(a - b).max() <= 1e-8 * np.abs(P.tractions()[0]).max()


def test_long_adhesion_in_many_groups(cntc):
    """Runs of adhesion over several wavefronts where the scaling takes four elements a thread in turn."""
    c = case(150, 9, 1e-6)
    n, one = 140, 600    # two groups each
    for k in range(n + 1):
        W.apply_case(cntc, one + k, 1, c)
    assert cntc.calculate(one, 1) == 0
    err = cntc.calculatebatch(list(range(one + 1, one + n + 1)), [1] * n)
    want = [a.tobytes() for a in cntc.gettractions(one, 1)]
    its = cntc.getiterations(one, 1)
    el = cntc.getelementdivision(one, 1).reshape(9, 150)
    got = [([a.tobytes() for a in cntc.gettractions(one + k, 1)], cntc.getiterations(one + k, 1)) for k in range(1, n + 1)]
    for k in range(n + 1):
        cntc.finalize(one + k)
    assert its[3] > 5 and not np.any(err) and (el == 1).sum(1).max() > 64
    assert all(g[0] == want and g[1][:4] == its[:4] for g in got)
