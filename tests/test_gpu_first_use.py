"""What the first evaluation of a kind builds, and what later calls of the other kind do without it."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

from conftest import ROOT, rel_l2

pytestmark = pytest.mark.gpu

ERR_ARG = -1


def _setup(spb, N, n, seed=3):
    from spectralbte_amd import workloads
    v, eta = workloads.grid_0d(N, 6.0)
    op = spb.Operator(N, 6.0, v, eta)
    op.generate_weights_iso(1.0)
    f = workloads.two_maxwellian_ensemble(N, 6.0, 2 * n, seed=seed)
    return op, f[:n], f[n:]


def _free(spb):
    a, b = ctypes.c_size_t(), ctypes.c_size_t()
    assert spb.lib().hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0   # from the runtime the library is linked to
    return a.value


@pytest.mark.parametrize("N,pad", [(24, 1.0), (20, 1.28)])
def test_first_evaluation_builds_one_table(spb, N, pad):
    """Q(f, f) needs the table with rows and columns folded (N/2 + 1 planes of each; N = 20: rows padded from 400 to 512)
    and 60 MB of scratch and partial sums at most; the one for Q(f, g), all columns, is not built with it.  So the folded
    tables are what these calls sum: there is no room for the whole one's copy."""
    op, f, g = _setup(spb, N, 1)
    op.sync()
    whole, half = 8 * N ** 6 * pad, (N // 2 + 1) / N
    free0 = _free(spb)
    op.compute_q(f)
    free1 = _free(spb)
    op.compute_q(f, g)
    free2 = _free(spb)
    op.close()
    slack = 64 << 20
    assert free0 - free1 <= whole * half ** 2 + slack < whole
    assert free1 - free2 <= whole * half + slack < whole


@pytest.mark.parametrize("N,form", [(16, "fp64"), (16, "fp32"), (16, "fp32a"), (24, "fp64"), (24, "fp32a"), (32, "fp64"),
                                    (32, "fp32"), (32, "fp32a")])
@pytest.mark.parametrize("mp", [False, True])
def test_noalloc_after_the_other_kind_of_call(spb, N, form, mp):
    """Refused while no evaluation has built a table for the tile; then served for both kinds of call: by rounding as
    spbte_compute_q's (1e-12; FP32 weights and products 1e-6) before that kind's table is there, with its bits after."""
    op, f, g = _setup(spb, N, 1)
    F = {"fp64": 0, "fp32": 1, "fp32a": 3}[form]
    flags = spb.MAXPRESERVE if mp else 0
    d_f, d_g, d_Q = spb.DeviceArray.from_host(f), spb.DeviceArray.from_host(g), spb.DeviceArray(f.shape)
    L = spb.lib()

    def noalloc(second):
        rc = L.spbte_compute_q_noalloc(op.h, d_f.ptr, second, d_Q.ptr, 1, F, flags | (0 if second else spb.SELF))
        op.sync()
        return rc, d_Q.download()
    assert noalloc(None)[0] == ERR_ARG and noalloc(d_g.ptr)[0] == ERR_ARG
    tol = 1e-12 if form == "fp64" else 1e-6
    own = op.compute_q(f, form=form, maxpreserve=mp)
    rc, q = noalloc(None)
    assert rc == 0 and np.array_equal(q, own)
    rc, before = noalloc(d_g.ptr)
    assert rc == 0, L.spbte_last_error()
    pair = op.compute_q(f, g, form=form, maxpreserve=mp)
    assert rel_l2(before, pair) < tol
    rc, q = noalloc(d_g.ptr)
    assert rc == 0 and np.array_equal(q, pair)
    op.close()


SCRIPT = """
import ctypes
import numpy as np
import spectralbte_amd as spb
from spectralbte_amd import workloads
N = 24
v, eta = workloads.grid_0d(N, 6.0)
op = spb.Operator(N, 6.0, v, eta)
op.generate_weights_iso(1.0)
W = op.get_weights()
f, g = workloads.two_maxwellian_ensemble(N, 6.0, 2, seed=1)
ref = op.compute_q(f[None], g[None])[0]
op.close()
spb.initialize_coll(N, 6.0, v, eta)
a, b = spb.WeightRows(W), spb.WeightRows(W)
q = spb.ComputeQ(f, f, a)
spb.ComputeQ(f, f, b)
# leave less than Q(f, g)'s table (0.83 GB) free
free, total, hold = ctypes.c_size_t(), ctypes.c_size_t(), []
while True:
    assert spb.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    if free.value <= 640 << 20 or len(hold) == 100:
        break
    hold.append(spb.DeviceArray((min(free.value - (600 << 20), 8 << 30) // 8,)))
got = spb.ComputeQ(f, g, a)
assert np.linalg.norm(np.ravel(got) - np.ravel(ref)) < 1e-12 * np.linalg.norm(ref)
assert np.array_equal(np.ravel(spb.ComputeQ(f, f, a)), np.ravel(q))
print("evicted and served", flush=True)
"""


def test_reference_interface_makes_room_for_the_table_of_a_pair(spb):
    """Two tables cached, then memory short of the one a first Q(f, g) builds: the other operator goes, the call is served."""
    out = subprocess.run([sys.executable, "-c", SCRIPT], cwd=ROOT, capture_output=True, text=True, timeout=100,
                         env=dict(os.environ, PYTHONPATH=ROOT))
    assert out.returncode == 0 and "evicted and served" in out.stdout, out.stderr[-2000:]
    assert "evicting the least recently used" in out.stderr
