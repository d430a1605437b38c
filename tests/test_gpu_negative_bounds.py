"""A negative coefficient of friction, which the calls accept: every |p| exceeds the traction bound,
and what is put on it changes sign, in the GD and in the SteadyGS kernels.

No such case converges, so a few sweeps are compared, at which the iteration is not yet sensitive: the
oracle's own tractions change by 3e-12 of the largest pressure where Fn does by 5e-13, and the two
differ in the rounding of their sums alone, 1e-14: compared to 1e-8.
"""
import numpy as np
import pytest

from contact_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gausei,maxgs", [(5, 6), (0, 12)])
def test_negative_friction(cntc, oracle, gausei, maxgs):
    c = W.base_case(tang=3, norm=1, fn=9e4, cksi=-4e-4, ceta=3e-4, cphi=1e-4, eps=1e-8, ipotcn=-3, mx=18, my=15, aa=6.0,
                    bb=6.0, scale=1.3, gausei=gausei, fstat=-0.3, maxgs=maxgs, maxin=1)
    rc, of, P = oracle.solve_case(c)
    ire = 945
    W.apply_case(cntc, ire, 1, c)
    assert cntc.calculate(ire, 1) == rc
    p = [a.ravel() for a in cntc.gettractions(ire, 1)]
    its = cntc.getiterations(ire, 1)
    el = cntc.getelementdivision(ire, 1).ravel()
    cntc.finalize(ire)
    print(gausei, rc, its, P.iters(), "adhesion", (el == 1).sum(), "slip", (el == 2).sum())
    assert its[3] == P.iters()[3]
    for a, b in zip(p, P.tractions()):
        assert np.abs(a - b).max() <= 1e-8 * np.abs(P.tractions()[0]).max()
