"""The integral terms of the pair-product propagator at grid sizes around the 64 x
64 tiles of the contraction kernel, against the oracle's sums over the same
nodes."""
import numpy as np
import pytest

import oracle as O
from pimc import prop_int_terms

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 63, 64, 65, 129])
@pytest.mark.parametrize("tau", [0.5, 0.01])
def test_prop_terms_at_tile_edges(n, tau):
    """A term is a sum of up to 6 000 products whose absolute values add up to at
    most three times the largest diagonal entry (Cauchy-Schwarz), each product
    good to a few roundings: 6 000 x 4 x 1.1e-16 x 3 = 8e-12 of that entry.  The
    matrix is symmetric to the bit."""
    r1, g0 = 9.0, 2.0
    got, ref = prop_int_terms(n, 1e-20, r1, g0, tau), O.prop_int_terms(n, 1e-20, r1, g0, tau)
    assert np.max(np.abs(got - ref)) < 8e-12 * np.max(np.abs(np.diag(ref)))
    assert np.array_equal(got, got.T)
