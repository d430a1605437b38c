"""GDsteady's row recurrences at row lengths around the read-ahead of their LDS cells (blocks of
four and eight), at tiles of one row (rows longer than half a tile, and than a tile) and of many.

Tolerances: both solvers stop at eps 1e-11 of the traction's rms, with a mean rate of convergence
of about 0.9 a sweep: within about 1e-9 of the solution, compared to 1e-8 of the largest pressure;
forces to 1e-8 of mu Fn.
"""
import numpy as np
import pytest

from contact_amd import workloads as W

pytestmark = pytest.mark.gpu

GRIDS = [(9, 10), (10, 9), (13, 12), (16, 21), (17, 13), (18, 30), (40, 33), (600, 7), (1030, 6)]
WIDE = 500     # gross sliding there: GDsteady needs about a thousand sweeps for partial slip


@pytest.mark.parametrize("mx,my", GRIDS)
def test_row_lengths(cntc, oracle, mx, my):
    # element sides within a factor of two, partial slip
    aa, bb = (6.0, 6.0 * min(1.0, 1.5 * my / mx))
    fn = 9e4 if bb > 3 else 3e3
    cksi, ceta, cphi = (-4e-4, 3e-4, 1e-4) if mx < WIDE else (-2e-2, 1e-2, 0.0)
    c = W.base_case(tang=3, norm=1, fn=fn, cksi=cksi, ceta=ceta, cphi=cphi, eps=1e-11, ipotcn=-3,
                    mx=mx, my=my, aa=aa, bb=bb, scale=max(1.3, min(mx, my) / (min(mx, my) - 3.0)))
    ire = 941
    W.apply_case(cntc, ire, 1, c)
    assert cntc.calculate(ire, 1) == 0
    p = [a.ravel() for a in cntc.gettractions(ire, 1)]
    f, its = cntc.getcontactforces(ire, 1), cntc.getiterations(ire, 1)
    cntc.finalize(ire)
    rc, of, P = oracle.solve_case(c)
    assert rc == 0
    print(mx, my, "iterations", its, P.iters())
    for a, b in zip(p, P.tractions()):
        assert np.abs(a - b).max() <= 1e-8 * np.abs(P.tractions()[0]).max()
    for a, b in zip(f[:3], of[:3]):
        assert abs(a - b) <= 1e-8 * c["fstat"] * fn
