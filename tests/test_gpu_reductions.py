"""The fused reductions at the edges of their work-group counts (1024 elements a group): one group,
just over one, one and just over one wavefront of groups.  The frictionless problem runs every
masked sum, dot, maximum and count of NormCG through them.

Tolerances: at eps 1e-12 both solvers stop within about 1e-11 of the solution, so the pressures
are compared to 1e-9 of the largest, the approach to 1e-9 of itself; the force is prescribed.
"""
import numpy as np
import pytest

from contact_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mx,my", [(12, 9), (32, 32), (41, 25), (256, 256), (257, 256)])
def test_normal_problem_at_group_edges(cntc, oracle, mx, my):
    c = W.base_case(tang=0, norm=1, fn=9e4, eps=1e-12, ipotcn=-3, mx=mx, my=my, aa=6.0, bb=4.5, scale=1.4)
    ire = 940
    W.apply_case(cntc, ire, 1, c)
    assert cntc.calculate(ire, 1) == 0
    pn = cntc.gettractions(ire, 1)[0].ravel()
    pen, fn = cntc.getpenetration(ire, 1), cntc.getcontactforces(ire, 1)[0]
    cntc.finalize(ire)
    rc, of, P = oracle.solve_case(c)
    opn = P.tractions()[0]
    assert rc == 0
    assert abs(fn - 9e4) <= 1e-9 * 9e4 and abs(of[0] - 9e4) <= 1e-9 * 9e4
    assert np.abs(pn - opn).max() <= 1e-9 * opn.max()
    assert abs(pen - P.pen()) <= 1e-9 * abs(P.pen())
