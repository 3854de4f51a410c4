"""Tables whose quadratures run over the distinct entries only (k_weights.hip, with_entries): every entry against the
oracle's on grids whose modes have mirror images (even N: all but one; odd N: all, or the 1D grid's half-integer modes),
and on one whose modes have none.  Bounds as for the same tables elsewhere: 1e-12 of max|W| for the Landau rule, 1e-10
for the glance table's, 1e-8 of max|W| for an isotropic exponent without a closed form."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,grid", [(2, "0d"), (3, "0d"), (5, "0d"), (5, "1d"), (6, "0d"), (6, "shifted"), (7, "1d")])
def test_tables_by_images_against_oracle(spb, orc, N, grid):
    Lv, lam = 4.0, 0.5
    v, eta = (orc.grid_1d if grid == "1d" else orc.grid_0d)(N, Lv)
    if grid == "shifted":
        eta = eta + 0.3 * (eta[1] - eta[0])
    op = spb.Operator(N, Lv, v, eta)
    op.generate_weights_iso(lam, 1.0, 2.0, 1.0, 2.0)
    ref = orc.weights_iso(N, eta, Lv, lam, 1.0, 2.0, 1.0, 2.0)
    assert np.abs(op.get_weights() - ref).max() <= 1e-8 * np.abs(ref).max()
    op.generate_weights_landau(lam)
    ref = orc.weights_landau(N, eta, Lv, lam)
    assert np.abs(op.get_weights() - ref).max() <= 1e-12 * np.abs(ref).max()
    op.generate_weights_glance(lam, 0.1)
    rng = np.random.default_rng(N)
    rows, cols = rng.integers(0, N ** 3, 30), rng.integers(0, N ** 3, 30)
    ref = orc.weights_glance_entries(N, eta, Lv, lam, 0.1, rows, cols, (6, 6, 4, 4))
    assert np.abs(op.get_weights()[rows, cols] - ref).max() <= 1e-10 * np.abs(ref).max()
    op.close()
