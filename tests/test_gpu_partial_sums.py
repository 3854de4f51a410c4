"""Split sums whose partial sums do not fit their buffer go part of the batch by part, with the same slices: the results
are those of one launch, bit for bit."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FORMS = {"fp64": 0, "fp32": 1, "fp16x2": 2, "fp32a": 3}


def _op(spb, N):
    from spectralbte_amd import workloads
    v, eta = workloads.grid_0d(N, 6.0)
    op = spb.Operator(N, 6.0, v, eta)
    op.generate_weights_iso(1.0)
    return op, workloads


# how: "default", "tuned" on a larger batch of the same power of two, or a pinned tile (tr, lines, tb, slices)
@pytest.mark.parametrize("N,n,form,mp,how", [
    (32, 4, "fp64", True, "default"), (32, 10, "fp64", True, "default"), (32, 17, "fp64", False, "default"),
    (32, 10, "fp64", True, "tuned"), (32, 10, "fp32a", True, "default"), (32, 11, "fp32a", True, (4, 4, 1, 64)),
    (32, 7, "fp32", False, (4, 4, 4, 32)), (32, 5, "fp16x2", True, "default"), (24, 11, "fp32a", True, "default"),
    (24, 9, "fp64", False, "default"), (16, 100, "fp64", True, "default"), (16, 40, "fp64", False, (1, 4, 1, 256)),
    (20, 100, "fp64", False, "default"), (18, 70, "fp64", True, "default"), (10, 200, "fp64", True, "default")])
def test_noalloc_part_by_part(spb, N, n, form, mp, how):
    """The workspace of 64 MiB holds the partial sums of some of the cells only (or just of all)."""
    op, workloads = _op(spb, N)
    if how == "tuned":
        op.autotune(16, form, mp)
    elif how != "default":
        op.set_tile(form, mp, *how[:3], kind=how[3])
    f = workloads.two_maxwellian_ensemble(N, 6.0, n, seed=n)
    flags = spb.SELF | spb.CONSERVE | (spb.MAXPRESERVE if mp else 0)
    d_f, d_Q, d_R = spb.DeviceArray.from_host(f), spb.DeviceArray(f.shape), spb.DeviceArray(f.shape)
    L = spb.lib()
    assert L.spbte_compute_q(op.h, d_f.ptr, None, d_R.ptr, n, FORMS[form], flags) == 0
    op.sync()
    ref = d_R.download()
    d_Q.upload(np.full(f.shape, np.nan))
    assert L.spbte_compute_q_noalloc(op.h, d_f.ptr, None, d_Q.ptr, n, FORMS[form], flags) == 0, L.spbte_last_error()
    op.sync()
    assert np.array_equal(d_Q.download(), ref)
    op.close()


def _free(spb):
    a, b = ctypes.c_size_t(), ctypes.c_size_t()
    assert spb.lib().hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0   # from the runtime the library is linked to
    return a.value


def _growth(spb, op, d_f, d_Q, n, form, flags):
    free = _free(spb)
    assert spb.lib().spbte_compute_q(op.h, d_f.ptr, None, d_Q.ptr, n, FORMS[form], flags) == 0, spb.lib().spbte_last_error()
    op.sync()
    return free - _free(spb)


def _unsplit_first(spb, op, d_f, d_Q, n, form, flags):
    """Scratch and tables of a batch without partial sums; leaves the batch's own tile, which it returns, to be split."""
    tile = op.get_tile(n, form, True)
    op.set_tile(form, True, *tile[1:], kind=1)
    _growth(spb, op, d_f, d_Q, n, form, flags)
    op.set_tile(form, True, 0, 0, 0)
    return tile


def test_partial_sums_of_a_large_batch_are_bounded(spb):
    """1000 problems at N = 32 with FP32 products, 16 slices: 7.8 GiB of partial sums at once, 6 GiB at most are kept."""
    N, n, form, flags = 32, 1000, "fp32a", spb.SELF | spb.MAXPRESERVE
    op, workloads = _op(spb, N)
    f = np.resize(workloads.two_maxwellian_ensemble(N, 6.0, 50, seed=1), (n, N ** 3)) * (1 + np.arange(n)[:, None] / n)
    d_f, d_Q = spb.DeviceArray.from_host(f), spb.DeviceArray(f.shape)
    tile = _unsplit_first(spb, op, d_f, d_Q, n, form, flags)
    assert tile[0] == 16
    assert _growth(spb, op, d_f, d_Q, n, form, flags) <= (6 << 30) + (64 << 20)
    q = d_Q.download()
    op.set_tile(form, True, *tile[1:], kind=tile[0])
    some = [0, 1, 499, 500, 501, 998, 999]   # on both sides of the parts
    assert np.array_equal(op.compute_q(f[some], form=form, maxpreserve=True), q[some])
    op.close()


def test_partial_sums_without_room(spb):
    """Memory short of the partial sums (64 cells at N = 32: 256 MiB): the batch goes in smaller parts."""
    N, n, form, flags = 32, 64, "fp64", spb.SELF | spb.MAXPRESERVE
    op, workloads = _op(spb, N)
    f = workloads.two_maxwellian_ensemble(N, 6.0, n, seed=2)
    d_f, d_Q = spb.DeviceArray.from_host(f), spb.DeviceArray(f.shape)
    tile = _unsplit_first(spb, op, d_f, d_Q, n, form, flags)
    hold = []
    while _free(spb) > 180 << 20 and len(hold) < 100:
        hold.append(spb.DeviceArray((min(_free(spb) - (160 << 20), 8 << 30) // 8,)))
    grown = _growth(spb, op, d_f, d_Q, n, form, flags)
    q = d_Q.download()
    hold.clear()
    assert grown <= 160 << 20 < tile[0] * n * 16 * N ** 3
    op.set_tile(form, True, *tile[1:], kind=tile[0])
    assert np.array_equal(op.compute_q(f[:3], form=form, maxpreserve=True), q[:3])
    assert np.array_equal(op.compute_q(f[-3:], form=form, maxpreserve=True), q[-3:])
    op.close()
