"""Large FP32 products whose rows or columns past the whole rounds of tiles are a launch
of their own (csrc/sgemm_split.hip, the cut in plan_sgemm_f16), against float64 under the
bound of test_gpu_sgemm_f16: both directions of the cut, the rest with and without a K
split and down to one row or column, every layout, epilogue and operands off 16 bytes.
"""
import numpy as np
import pytest

import pcl
from gpu_util import announce, require_device
from test_gpu_sgemm_f16 import N_, T_, check, operands, run

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    require_device()


# (M, N, K): the rest beside it
SHAPES = [(4097, 4096, 700),   # one row, K split in three
          (4096, 4097, 700),   # one column, K split in three
          (4143, 4187, 155),   # 303 rows, not split
          (4187, 4143, 155),   # 347 rows, not split
          (2339, 3369, 2149)]  # 35 rows, K split in nine


@pytest.mark.parametrize("opA,opB", [(N_, N_), (N_, T_), (T_, N_), (T_, T_)])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_cut_layouts(M, N, K, opA, opB):
    announce("sgemm f16 cut", M, N, K, opA, opB)
    a, b = operands(M, N, K, opA, opB, 21)
    check(run(a, b, opA, opB, 3, 1, 1), a, b)


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_cut_epilogues(M, N, K):
    """Bias, old values, residual and both GELU operands at the rest's rows and columns."""
    announce("sgemm f16 cut epilogues", M, N, K)
    a, b = operands(M, N, K, N_, N_, 22)
    r = np.random.default_rng(23)
    bias, old = r.standard_normal(N, np.float32), r.standard_normal((M, N), np.float32)
    shift = bias[None, :].astype(np.float64)
    check(run(a, b, N_, N_, bias=bias, C0=old), a, b, shift + old)
    check(run(a, b, N_, N_, bias=bias, epi=pcl.EPI_RESID, aux=old), a, b, shift + old)
    out, pre = run(a, b, N_, N_, bias=bias, epi=pcl.EPI_GELU, want_pre=True)
    check(pre, a, b, shift)
    gelu = lambda x: 0.5 * x * (1 + np.tanh(np.sqrt(2 / np.pi) * (x + 0.044715 * x**3)))  # noqa: E731
    v = pre.astype(np.float64)
    assert (np.abs(out - gelu(v)) <= 1e-6 * (np.abs(v) + 1)).all()  # the activation's own fp32 error
    t = np.tanh(np.sqrt(2 / np.pi) * (old + 0.044715 * old.astype(np.float64)**3))
    grad = 0.5 * (1 + t) + 0.5 * old * (1 - t * t) * np.sqrt(2 / np.pi) * (1 + 3 * 0.044715 * old.astype(np.float64)**2)
    v = v - shift
    got = run(a, b, N_, N_, epi=pcl.EPI_GELU_BWD, aux=old)
    # pre's own distance from v: a few 2^-22 of the sum's scale (|a| ~ 1, |b| ~ 0.05)
    assert (np.abs(got - v * grad) <= 2e-6 * (np.abs(v) + 0.05 * np.sqrt(K) + 3)).all()


def test_cut_rows_not_finite():
    """An infinity in a kept row and a NaN in the rest's: only their rows change."""
    announce("sgemm f16 cut nonfinite")
    M, N, K = SHAPES[0]
    a, b = operands(M, N, K, N_, N_, 24)
    a[17, 3], a[M - 1, K - 1] = np.inf, np.nan
    C = run(a, b, N_, N_)
    assert np.array_equal(C[17], np.sign(b[3]) * np.float32(np.inf)) and np.isnan(C[M - 1]).all()
    fine = np.isfinite(a).all(1)
    check(C[fine], a[fine], b)
