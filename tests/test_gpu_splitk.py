"""The second pass of K-split FP32 products (csrc/sgemm.hip sgemm_splitk_reduce_kernel):
one to sixteen partials, groups of eight and remainders, one and four outputs per thread,
result rows on and off 16 bytes, old C, bias and epilogues, against float64.

Bound per output: K fused products, the partials' sum and the bias, each rounded to 2^-24
of a partial sum no larger than sum |a b| + |bias| + |old C|:
  |C - R| <= (K + 32) 2^-24 (sum|a b| + |bias| + |C0|);
GELU's slope is below 1.13 and its own error below 2^-21 of |value| plus 2^-22 of |x|.
"""
import numpy as np
import pytest

import pcl
from gpu_util import announce, require_device

pytestmark = pytest.mark.gpu
N_, T_ = pcl.OP_N, pcl.OP_T


@pytest.fixture(scope="module", autouse=True)
def _device():
    require_device()


def gelu(x):
    return 0.5 * x * (1 + np.tanh(np.sqrt(2 / np.pi) * (x + 0.044715 * x ** 3)))


# M x N below 16 tiles of 64 x 64 split K into chunks of 64 or 128: K / 64 partials; the
# last three have a million outputs, which go four to a thread where N % 4 == 0, in two and
# three partials made from f16 parts (errors within the same bound for these inputs)
SHAPES = [(M, N, K) for M, N in [(100, 256), (63, 333), (1, 68), (130, 130)] for K in [128, 512, 576, 1024]]


@pytest.mark.parametrize("M,N,K", SHAPES + [(1024, 1024, 2048), (1030, 1028, 4096), (1030, 1026, 4096)])
@pytest.mark.parametrize("form", ["plain", "accumulate", "gelu", "resid", "odd rows"])
def test_splitk(M, N, K, form):
    announce("splitk", M, N, K, form)
    r = np.random.default_rng(M * 7 + N * 3 + K)
    a, b = r.standard_normal((M, K), np.float32), r.standard_normal((K, N), np.float32) * np.float32(K ** -0.5)
    bias, extra = r.standard_normal(N, np.float32), r.standard_normal((M, N), np.float32)
    ldc, shift = (N + 5, 1) if form == "odd rows" else (N, 0)
    c0 = np.full(shift + M * ldc, 7.5, np.float32)
    c0[shift:].reshape(M, ldc)[:, :N] = extra
    dA, dB, dbias, dC, dx = pcl.dev(a), pcl.dev(b), pcl.dev(bias), pcl.dev(c0), pcl.dev(extra)
    pre = pcl.empty((M, N), np.float32)
    if form in ("gelu", "resid"):
        epi, aux = (pcl.EPI_GELU, None) if form == "gelu" else (pcl.EPI_RESID, dx.ptr)
        pcl.check(pcl.lib.pcl_sgemm_ex(N_, N_, M, N, K, dA.ptr, K, dB.ptr, N, dbias.ptr, epi, aux,
                                       pre.ptr if form == "gelu" else None, N, dC.ptr, N, None))
    else:
        pcl.check(pcl.lib.pcl_sgemm(N_, N_, M, N, K, dA.ptr, K, dB.ptr, N, dbias.ptr,
                                    int(form == "accumulate"), dC.ptr + 4 * shift, ldc, None))
    pcl.sync()
    out = dC.download((shift + M * ldc,), np.float32)
    C = out[shift:].reshape(M, ldc)
    v = a.astype(np.float64) @ b + bias
    mag = np.abs(a).astype(np.float64) @ np.abs(b) + np.abs(bias)
    bound = (K + 32) * 2.0 ** -24
    if form == "gelu":
        assert np.all(np.abs(pre.download((M, N), np.float32) - v) <= bound * mag)
        R, tol = gelu(v), 1.13 * bound * mag + 2.0 ** -21 * np.abs(gelu(v)) + 2.0 ** -22 * np.abs(v)
    elif form in ("accumulate", "resid"):
        R, tol = v + extra, bound * (mag + np.abs(extra))
    else:
        R, tol = v, bound * mag
    assert np.all(np.abs(C[:, :N] - R) <= tol)
    assert np.all(out[:shift] == 7.5) and np.all(C[:, N:] == 7.5)  # nothing beside the result
