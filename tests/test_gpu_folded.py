"""The folded weighted sum (half the output modes, and half the summed ones for
Q(f, f)) against the oracle's whole sum, on tables without any symmetry of their
own, so that a wrong partner, mirror image or sign shows.

Bounds: FP64 sums of at most N^3 terms of random sign round to about 1e-15 of
their result; 1e-12 as for every FP64 form.  FP32 weights and products round
each term by 2^-24, independently: 1e-6 of the result, as for every FP32 form."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

TILES = {16: [None, (4, 1, 1, 1), (4, 1, 2, 16), (2, 1, 1, 8), (1, 1, 1, 64), (1, 2, 1, 32), (1, 4, 1, 256),
           (4, 4, 2, 16), (4, 4, 1, 8)],
         24: [None, (3, 3, 1, 1), (3, 3, 2, 24), (4, 2, 1, 1)],   # the last one straddles planes: whole table
         32: [None, (8, 2, 1, 4), (4, 4, 4, 1), (4, 2, 1, 64), (4, 1, 1, 2)]}


def _cells(N, n, seed):
    return np.random.default_rng(seed).uniform(0.0, 1.0, (n, N ** 3))


def _op(spb, orc, N, grid, seed):
    Lv = 6.0
    v, eta = (orc.grid_1d if grid == "1d" else orc.grid_0d)(N, Lv)
    if grid == "shifted":   # modes not symmetric about zero: no row fold
        eta = eta + 0.3 * (eta[1] - eta[0])
    W = np.random.default_rng(seed).standard_normal((N ** 3, N ** 3))
    op = spb.Operator(N, Lv, v, eta)
    op.set_weights(W)
    return op, v, eta, W


@pytest.mark.parametrize("grid", ["0d", "1d", "shifted"])
@pytest.mark.parametrize("mp", [False, True])
@pytest.mark.parametrize("pair", [False, True])
def test_folded_sum_n16_against_oracle(spb, orc, grid, mp, pair):
    N, n = 16, 3
    op, v, eta, W = _op(spb, orc, N, grid, 1)
    f = _cells(N, n, 2)
    g = _cells(N, n, 3) if pair else f
    q = orc.compute_q_maxpreserve if mp else orc.compute_q
    ref = np.stack([q(N, v, eta, W, f[b], g[b]).ravel() for b in range(n)])
    for form, tol in (("fp64", 1e-12), ("fp32", 1e-6), ("fp32a", 1e-6)):
        for t in TILES[N]:
            try:
                op.set_tile(form, mp, *((0, 0, 0) if t is None else t))
            except spb.SpbteError:
                continue   # not instantiated for this form
            e = rel_l2(op.compute_q(f, g if pair else None, form=form, maxpreserve=mp), ref)
            assert e < tol, (form, t, e)
        op.set_tile(form, mp, 0, 0, 0)
    op.close()


@pytest.mark.parametrize("N,mp,pair", [(24, False, True), (24, True, False), (32, False, False), (32, True, True)])
def test_folded_sum_against_whole_sum(spb, orc, N, mp, pair):
    """N = 24 and 32: the folded tiles against the tiled kernel, which sums the whole table."""
    n = 5
    op, v, eta, W = _op(spb, orc, N, "0d", 4)
    f, g = _cells(N, n, 5), _cells(N, n, 6) if pair else None
    op.set_tile("fp64", mp, *{24: (6, 8, 1, 0), 32: (4, 2, 1, 0)}[N])
    ref = op.compute_q(f, g, maxpreserve=mp)
    for form, tol in (("fp64", 1e-12), ("fp32a", 1e-6)):
        for t in TILES[N]:
            try:
                op.set_tile(form, mp, *((0, 0, 0) if t is None else t))
            except spb.SpbteError:
                continue
            e = rel_l2(op.compute_q(f, g, form=form, maxpreserve=mp), ref)
            assert e < tol, (form, t, e)
    op.close()


@pytest.mark.parametrize("N,grid,n", [(2, "0d", 3), (3, "0d", 2), (6, "0d", 5), (8, "1d", 64), (9, "0d", 3), (9, "1d", 3),
                                      (10, "0d", 7), (10, "shifted", 2), (12, "0d", 1), (14, "0d", 33), (15, "0d", 2),
                                      (15, "1d", 2), (18, "0d", 2), (20, "1d", 1), (23, "0d", 2)])
def test_folded_sum_other_grids_against_oracle(spb, orc, N, grid, n):
    """Grids without streaming tiles: even and odd, with the mirror symmetry and without (the 1D grid of
    odd N), one and two cells a workgroup, planes of one to nine waves."""
    op, v, eta, W = _op(spb, orc, N, grid, 10)
    f, g = _cells(N, n, 11), _cells(N, n, 12)
    some = sorted({0, n // 2, n - 1})
    for mp in (False, True):
        q = orc.compute_q_maxpreserve if mp else orc.compute_q
        for h in (f, g):
            got = op.compute_q(f, None if h is f else g, maxpreserve=mp)
            ref = np.stack([q(N, v, eta, W, f[b], h[b]).ravel() for b in some])
            assert rel_l2(got[some], ref) < 1e-12, (mp, h is g)
    op.close()


def test_noalloc_before_the_folded_table(spb, orc):
    """An allocation-free call on a grid without streaming tiles needs nothing resident: it sums the whole table then."""
    N = 10
    op, v, eta, W = _op(spb, orc, N, "0d", 13)
    f = _cells(N, 3, 14)
    d_f, d_Q = spb.DeviceArray.from_host(f), spb.DeviceArray(f.shape)
    ref = np.stack([orc.compute_q(N, v, eta, W, x, x).ravel() for x in f])
    for _ in range(2):   # before and after the table is there
        assert spb.lib().spbte_compute_q_noalloc(op.h, d_f.ptr, None, d_Q.ptr, 3, 0, spb.SELF) == 0
        op.sync()
        assert rel_l2(d_Q.download(), ref) < 1e-12
        assert rel_l2(op.compute_q(f), ref) < 1e-12
    op.close()


def test_qhat_of_complex_operands_is_whole(spb, orc):
    """spbte_qhat takes any operands and returns every mode: it never folds, whatever compute_q built before."""
    N = 16
    op, v, eta, W = _op(spb, orc, N, "0d", 7)
    op.compute_q(_cells(N, 1, 8))
    rng = np.random.default_rng(9)
    F, G = (rng.standard_normal((2, N ** 3)) + 1j * rng.standard_normal((2, N ** 3)) for _ in range(2))
    ref = np.stack([orc.qhat(N, W, F[b], G[b]).ravel() for b in range(2)])
    assert rel_l2(op.qhat(F, G, "fp64"), ref) < 1e-12
    op.close()
