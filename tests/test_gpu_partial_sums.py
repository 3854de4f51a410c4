"""Split sums whose partial sums do not fit their buffer go part of the batch by part, with the same slices: the results
are those of one launch, bit for bit."""
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
