"""The column stage of the products with one to nine groups of columns and a last one of few (they
are dealt to the eight XCDs in contiguous shares), in a coupled solve with three components.

Tolerances: at eps 1e-12 both solvers stop within about 1e-11 of the solution: tractions to 1e-9 of
the largest pressure.
"""
import numpy as np
import pytest

from contact_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mx", [4, 15, 16, 33, 79, 81, 112, 127, 128, 144])
def test_column_groups(cntc, oracle, mx):
    my = 9
    c = W.base_case(tang=1, norm=1, fn=3e4, cksi=2e-4, ceta=-1e-4, cphi=0.0, eps=1e-12, maxgs=300, ipotcn=-3, mx=mx, my=my,
                    aa=6.0, bb=6.0 * min(1.0, my / mx), scale=1.5, gausei=0)
    ire = 944
    W.apply_case(cntc, ire, 1, c)
    assert cntc.calculate(ire, 1) == 0
    p = [a.ravel() for a in cntc.gettractions(ire, 1)]
    its = cntc.getiterations(ire, 1)
    cntc.finalize(ire)
    rc, of, P = oracle.solve_case(c)
    assert rc == 0
    print(mx, "iterations", its, P.iters())
    for a, b in zip(p, P.tractions()):
        assert np.abs(a - b).max() <= 1e-9 * np.abs(P.tractions()[0]).max()
