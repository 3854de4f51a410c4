"""Tiles: what is pinned is what runs and what get_tile reports.

A cell's result depends on the tile's slices and on nothing else of the batch, so the same slices give the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _op(spb, N, n):
    from spectralbte_amd import workloads
    v, eta = workloads.grid_0d(N, 6.0)
    op = spb.Operator(N, 6.0, v, eta)
    op.generate_weights_iso(1.0)
    return op, workloads.two_maxwellian_ensemble(N, 6.0, n, seed=N)


@pytest.mark.parametrize("N,tile", [(24, (3, 3, 1, 24)), (32, (4, 4, 2, 16)), (32, (4, 4, 1, 32))])
def test_pinned_slices_run_as_given(spb, N, tile):
    """One cell group takes the pinned slices like several groups do: the same bits for the same cell."""
    op, f = _op(spb, N, 2 * tile[2] + 1)
    op.set_tile("fp64", True, *tile[:3], kind=tile[3])
    assert op.get_tile(1, "fp64", True) == (tile[3],) + tile[:3]
    assert np.array_equal(op.compute_q(f[:1], maxpreserve=True)[0], op.compute_q(f, maxpreserve=True)[0])
    op.close()


@pytest.mark.parametrize("N,form,mp", [(16, "fp64", True), (24, "fp64", False), (24, "fp32a", True), (32, "fp64", True),
                                       (32, "fp64", False), (32, "fp32a", True)])
def test_reported_tile_can_be_pinned(spb, N, form, mp):
    """The default tile of one cell, pinned, accepted and with the same bits."""
    op, f = _op(spb, N, 1)
    q = op.compute_q(f, form=form, maxpreserve=mp)
    kind, tr, lines, tb = op.get_tile(1, form, mp)
    op.set_tile(form, mp, tr, lines, tb, kind=kind)
    assert np.array_equal(op.compute_q(f, form=form, maxpreserve=mp), q)
    op.close()


def test_slice_counts_that_are_refused(spb):
    op, _ = _op(spb, 32, 1)
    for k in (3, 31, 33, 44, 46, 1025):
        with pytest.raises(spb.SpbteError):
            op.set_tile("fp64", True, 4, 4, 1, kind=k)
    op.close()


@pytest.mark.parametrize("N,n,tile", [(16, 1, (1, 4, 1, 32)), (16, 12, (4, 1, 2, 32)), (32, 1, (4, 4, 1, 16)), (32, 2, (4, 4, 2, 16))])
def test_sum_over_the_whole_table_has_its_own_slices(spb, N, n, tile):
    """spbte_qhat runs over all rows and columns: its slices are counted from those, not from a folded table's."""
    op, _ = _op(spb, N, 1)
    rng = np.random.default_rng(N)
    F, G = (rng.standard_normal((n, N ** 3)) + 1j * rng.standard_normal((n, N ** 3)) for _ in range(2))
    q = op.qhat(F, G)
    op.set_tile("fp64", False, *tile[:3], kind=tile[3])
    assert np.array_equal(op.qhat(F, G), q)
    op.close()


BOTH = [(form, mp) for form in ("fp64", "fp32", "fp16x2") for mp in (False, True)]
ALL = BOTH + [("fp32a", False), ("fp32a", True)]
ONE = [(form, False) for form in ("fp64", "fp32", "fp16x2")]


@pytest.mark.parametrize("N,tiles", [
    (16, {(4, 1, 1): BOTH, (4, 1, 2): ALL, (2, 1, 1): BOTH, (1, 1, 1): BOTH, (1, 2, 1): BOTH, (1, 4, 1): BOTH,
          (4, 4, 2): [("fp64", False)], (4, 4, 1): [("fp64", True)]}),
    (24, {(3, 3, 1): ALL, (3, 3, 2): ONE + [("fp32a", False), ("fp32a", True)], (4, 2, 1): ALL}),
    (32, {(8, 2, 1): BOTH, (4, 4, 4): ONE + [("fp32a", False)], (4, 2, 1): BOTH, (4, 1, 1): ONE})])
def test_streaming_tiles_that_are_there(spb, N, tiles):
    """The tiles that the folded sums are tested with, for each (form, two products): a test that passes over a refused
    tile must not do so for one of these."""
    op, _ = _op(spb, N, 1)
    for tile, pairs in tiles.items():
        for form, mp in pairs:
            op.set_tile(form, mp, *tile, kind=2)
            assert op.get_tile(1, form, mp) == (2,) + tile
            op.set_tile(form, mp, 0, 0, 0)
    op.close()
