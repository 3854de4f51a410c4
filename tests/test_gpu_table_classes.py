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


def _uneven(orc, N, Lv):
    """A grid whose positive modes are 4 roundings of the largest above their mirror images: one class each, still."""
    v, eta = orc.grid_0d(N, Lv)
    eta = eta + np.where(eta > 0, 4 * np.finfo(float).eps * np.abs(eta).max(), 0.0)
    return v, eta


@pytest.mark.parametrize("N,Lv,r0", [(6, 4.0, 0), (10, 6.1, 555)])
def test_landau_entries_are_those_of_their_own_modes(spb, orc, N, Lv, r0):
    """The phases of an entry reach 14 (N = 6) and 24 (N = 10), so modes 4 roundings off would move it by 1e-14; its own
    roundings and the oracle's, each 1e-15 of the largest at most, leave 3e-15."""
    v, eta = _uneven(orc, N, Lv)
    op = spb.Operator(N, Lv, v, eta)
    op.generate_weights_landau(1.0)
    nr = 40
    W, ref = op.get_weights()[r0:r0 + nr], orc.weights_landau(N, eta, Lv, 1.0, rows=(r0, nr))
    op.close()
    assert np.linalg.norm(W - ref) <= 3e-15 * np.linalg.norm(ref)


@pytest.mark.parametrize("N,Lv,m_j", [(8, 5.0, 1.0), (10, 6.1, 3.0), (15, 6.3, 1.0)])
def test_isotropic_entries_are_those_of_their_own_modes(spb, orc, N, Lv, m_j):
    """The same for an exponent without a closed form, against the same 64 panels of 20 points in long double; bound 1e-15:
    1280 terms each with its own roundings average to less than one."""
    L, lam = np.longdouble, 0.5
    v, eta = _uneven(orc, N, Lv)
    op = spb.Operator(N, Lv, v, eta)
    op.generate_weights_iso(lam, 2.0, 2.0, 1.0, m_j)
    W = op.get_weights()
    op.close()
    rng = np.random.default_rng(N)
    r, c = rng.integers(0, N ** 3, 400), rng.integers(0, N ** 3, 400)
    e, mu = eta.astype(L), L(m_j) / (1 + L(m_j))
    z, k = (np.stack([e[q // N ** 2], e[q // N % N], e[q % N]], 1) for q in (r, c))
    a0, a1, a2 = mu * np.sqrt((z * z).sum(1)), np.sqrt((k * k).sum(1)), np.sqrt(((k - mu * z) ** 2).sum(1))
    x, w = (q.astype(L) for q in np.polynomial.legendre.leggauss(20))
    for _ in range(2):   # the rule to long double
        p = [np.ones_like(x), x]
        for j in range(2, 21):
            p.append(((2 * j - 1) * x * p[-1] - (j - 1) * p[-2]) / j)
        d = 20 * (x * p[20] - p[19]) / (x * x - 1)
        x = x - p[20] / d
    w = 2 / ((1 - x * x) * d * d)
    h = L(Lv) / 64
    rho = (np.arange(64)[:, None] * h + h * (x[None] + 1) / 2).ravel()
    wr = np.tile(w, 64) * h / 2 * rho ** (L(lam) + 2)

    def sinc(a):
        y = a[:, None] * rho[None]
        return np.where(y == 0, 1, np.sin(y) / np.where(y == 0, 1, y))
    ref = ((sinc(a0) * sinc(a2) - sinc(a1)) * wr).sum(1)
    tw = np.where((np.arange(N) == 0) | (np.arange(N) == N - 1), 0.5, 1.0)
    pi, he = L("3.141592653589793238462643383279502884"), L(eta[1] - eta[0])
    ref = ref * (tw[c // N ** 2] * tw[c // N % N] * tw[c % N]) * 16 * pi ** 2 * he ** 3 / (2 * pi) ** L(1.5) / (4 * pi)
    assert np.linalg.norm(W[r, c] - ref) <= 1e-15 * np.linalg.norm(ref)
