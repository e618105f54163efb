"""The tied head's dlogits written as split rows by the cross-entropy itself (ce.hip
ce_row_regs_kernel, SPLIT), against float64: vocabularies that end at every kind of place
in a piece of eight and at the most a workgroup's registers hold, row counts that are
not multiples of eight, chunks, and rows that are not finite.

Tolerance: FP32_TOL of the largest value of each row of d_lnf (one row's split must not
hide behind another's scale) and of dwte as a whole, as everywhere for the head.
"""
import numpy as np
import pytest

import binding as ob
from gpu_util import FP32_TOL, announce, rel, require_device
from test_gpu_ce import LOSS_RTOL, _head, _head64

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    require_device()


def _case(M, D, V):
    x = ob.normal((M, D), 2300 + V, 0.0, 1.0)
    w = ob.normal((V, D), 2301 + V, 0.0, 0.1)
    t = (ob.u8((M,), 2302 + V).astype(np.int64) * 7919 % V).astype(np.int32)
    t[0], t[1], t[2] = V - 1, 0, V // 8 * 8 - 1
    return x, w, t


def _rows(dx, want):
    assert (np.abs(dx - want).max(1) <= FP32_TOL * np.abs(want).max(1)).all()


@pytest.mark.parametrize("M,D,V,chunk_rows", [(1030, 512, 2051, 0), (131, 256, 16390, 0), (150, 128, 33599, 0),
                                              (150, 128, 50257, 0), (200, 128, 53248, 0),
                                              (150, 128, 53249, 0),  # past the registers: split by its own pass
                                              (400, 256, 16390, 128)])  # three chunks and one of 16 rows
def test_head_split_rows(M, D, V, chunk_rows):
    announce("head_ce split", M, D, V, chunk_rows)
    x, w, t = _case(M, D, V)
    x[5] *= 40  # nearly one-hot
    dw0 = ob.normal((V, D), 2303, 0.0, 1e-3)
    loss, dx, dw = _head(x, w, t, dw0, chunk_rows * ((V + 63) // 64 * 64) * 4)
    loss64, dx64, dw64 = _head64(x, w, t, dw0)
    assert loss == pytest.approx(loss64, rel=LOSS_RTOL)
    _rows(dx, dx64)
    assert rel(dw - dw0, dw64 - dw0) <= FP32_TOL


def test_head_split_rows_not_finite():
    """A row of NaN logits gives a NaN row of d_lnf and no other; a target out of range
    a NaN loss and its row's plain probabilities."""
    M, D, V = 1030, 512, 2051
    announce("head_ce split nonfinite", M, D, V)
    x, w, t = _case(M, D, V)
    x[7, 3] = np.nan
    t[9] = V + 1  # inside the padding of the logits' rows
    loss, dx, _ = _head(x, w, t, np.zeros((V, D), np.float32), want_dw=False)
    assert np.isnan(loss) and np.isnan(dx[7]).all()
    lg = x[9].astype(np.float64) @ w.T.astype(np.float64)
    p = np.exp(lg - lg.max())
    _rows(dx[9:10], (p / p.sum() / M @ w.astype(np.float64))[None])
    fine = np.delete(np.arange(M), [7, 9])
    _, dx64, _ = _head64(x[fine], w, t[fine])
    _rows(dx[fine], dx64 * (len(fine) / M))
