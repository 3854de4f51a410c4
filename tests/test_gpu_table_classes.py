"""Tables by images take modes as equal in absolute value only where they are to rounding: modes of a caller's grid that are
symmetric to 9e-13 only get entries of their own.  Bound: the Landau rule sums 2048 terms of size up to max|W| with FP64
roundings of 1.1e-16 each, 5e-15 if all fell one way for the root of their number; 1e-13 leaves 20 times that.  Entries
computed at the other mode's value would be 1e-12 off."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,Lv", [(5, 6.0), (6, 4.0)])
@pytest.mark.parametrize("shift", [9e-13])
def test_modes_of_nearly_equal_size(spb, orc, N, Lv, shift):
    v, eta = orc.grid_0d(N, Lv)
    eta = eta.copy()
    eta[N - 2] *= 1 + shift
    op = spb.Operator(N, Lv, v, eta)
    op.generate_weights_landau(0.5)
    ref = orc.weights_landau(N, eta, Lv, 0.5)
    assert np.abs(op.get_weights() - ref).max() <= 1e-13 * np.abs(ref).max()
    op.close()
