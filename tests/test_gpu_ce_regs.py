"""Cross-entropy rows held in registers (ce.hip ce_row_regs_kernel): vocabularies
at the edges of what a workgroup's registers hold, rows that start at every
offset from a 16-byte boundary, row counts that are and are not powers of two,
and rows with infinite or NaN logits, against float64.

Tolerance. dl = (exp(x - max) * inv - [v == t]) / M in fp32: x - max is rounded
once, at most 2^-24 |x - max| < 2^-24 * 32 in the exponent here (logits of
deviation 3 over 51201 entries), which is 2e-6 of p; the exponential, the sum
over at most 104 terms per thread, the reciprocal, product and quotient add a few
2^-24. So 4e-6 of the largest gradient, and 1e-5 of the loss.
"""
import numpy as np
import pytest

import pcl
from gpu_util import announce, rel, require_device
from test_gpu_ce import LOSS_RTOL, _ce, _ce64, _inputs

pytestmark = pytest.mark.gpu
TOL = 4e-6


@pytest.fixture(scope="module", autouse=True)
def _device():
    require_device()


@pytest.mark.parametrize("V", [1, 3, 4, 7, 2047, 2048, 2049, 8192, 8193, 16384, 16385, 32768, 32769, 51199, 51200,
                               51201])
@pytest.mark.parametrize("M,extra,inplace", [(8, 0, True), (5, 1, True), (6, 3, False)])
def test_ce_register_edges(V, M, extra, inplace):
    announce("ce_regs", M, V, extra, inplace)
    lg, t = _inputs(M, V, 2000 + V + M)
    loss, dl = _ce(lg, t, V + extra, inplace)
    loss64, dl64 = _ce64(lg, t)
    assert loss == pytest.approx(loss64, rel=LOSS_RTOL, abs=1e-7)
    assert np.abs(dl - dl64).max() <= TOL * max(np.abs(dl64).max(), 1.0 / M)


@pytest.mark.parametrize("V", [5, 2050, 9000, 50257])
def test_ce_register_rows_not_finite(V):
    """Alone in its row an infinite logit takes the sum to 1, leaves the other
    entries their p = 0 and is NaN itself; two of them, a NaN or a row of -inf
    leave the whole row NaN. The rows between are untouched."""
    announce("ce_regs_nonfinite", V)
    M = 8
    lg, t = _inputs(M, V, 2100 + V)
    t[:] = 2
    lg[1, V - 1] = np.inf
    lg[3, [0, V - 1]] = np.inf
    lg[5, 3] = np.nan
    lg[6, :] = -np.inf
    lg[7, 1] = -np.inf
    loss, dl = _ce(lg, t)
    assert np.isnan(loss)
    one = np.zeros(V)
    one[2], one[V - 1] = -1.0 / M, np.nan
    np.testing.assert_array_equal(dl[1], one)
    assert np.isnan(dl[[3, 5, 6]]).all()
    fine = [0, 2, 4, 7]
    _, dl64 = _ce64(lg[fine], t[fine])
    assert rel(dl[fine], dl64 * (len(fine) / M)) <= TOL


def test_ce_register_and_two_pass_rows_agree():
    """The same rows through both kernels: dlogits at another offset from a
    16-byte boundary than its logits takes the two-pass one."""
    M, V, ld = 6, 5000, 5004
    lg, t = _inputs(M, V, 2200)
    host = np.zeros((M, ld), np.float32)
    host[:, :V] = lg
    dlg, dt, got = pcl.dev(host), pcl.dev(t), []
    for ldd in (ld, ld + 1):
        dd, dloss = pcl.dev(np.full((M, ldd), np.nan, np.float32)), pcl.dev(np.zeros(1, np.float32))
        pcl.check(pcl.lib.pcl_cross_entropy(dlg.ptr, ld, dt.ptr, dd.ptr, ldd, M, V, dloss.ptr, None))
        pcl.sync()
        got.append((float(dloss.download((1,), np.float32)[0]), dd.download((M, ldd), np.float32)[:, :V]))
    assert got[0][0] == pytest.approx(got[1][0], rel=LOSS_RTOL)
    assert rel(got[0][1], got[1][1]) <= 2 * TOL
