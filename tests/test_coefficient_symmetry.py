"""The SteadyGS row walk uses no xy coefficients within a row (offsets along x only): they vanish in
the half space's closed form, for equal and for dissimilar materials, whatever the elements' shape."""
import numpy as np
import pytest


@pytest.mark.parametrize("mx,my,dx,dy", [(9, 11, 1.0, 1.0), (40, 37, 0.18, 0.13), (300, 4, 0.02, 1.5), (16, 16, 1.0, 0.01)])
@pytest.mark.parametrize("akv", [0.0, 0.1])
def test_no_xy_influence_within_a_row(oracle, mx, my, dx, dy, akv):
    cf = oracle.elascf_pcwcns(akv, 0.28, mx, my, dx, dy)
    for block in (cf[0, 1], cf[1, 0]):
        # rows of offsets -my .. my - 1 along y: offset 0 is row my
        assert np.abs(block[my]).max() <= 1e-15 * cf[0, 0, my, mx]
        assert np.abs(block).max() > 0.0
