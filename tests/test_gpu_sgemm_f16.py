"""Large FP32 products on the f16 matrix cores (csrc/sgemm_split.hip): tile edges and
K tails of every tile shape and split, layouts and strides, epilogues, rows of any scale,
infinities and NaN, and graph replays, against float64.

Bound per output. Each operand element is hi + lo (11 bits each) of the element scaled so
that its row's maximum is below 2^15: off by at most 2^-22 of itself, or 2^-39 of the row's
maximum where that is more. lo*lo, left out, is below 2^-22 |a b|. One accumulator takes
3 K/32 additions, each rounded to 2^-24 of a partial sum no larger than sum |a b|:
  |C - R| <= (3*2^-22 + (3 K/32 + 32) 2^-24) sum|a b| + 2^-38 (max|a| sum|b| + max|b| sum|a|)
plus 2^-22 of what bias, old C or residual add.
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


def operands(M, N, K, opA, opB, seed, padA=0, padB=0):
    """op(A) (M x K), op(B) (K x N) and their stored forms with padded rows."""
    r = np.random.default_rng(seed)
    a = r.standard_normal((M, K), np.float32)
    b = (r.standard_normal((K, N), np.float32) * np.float32(0.05))
    return a, b


def stored(x, transpose, pad):
    s = x.T if transpose else x
    out = np.full((s.shape[0], s.shape[1] + pad), np.nan, np.float32)  # padding is never read
    out[:, :s.shape[1]] = s
    return out


def run(a, b, opA, opB, padA=0, padB=0, shift=0, bias=None, C0=None, epi=None, aux=None, want_pre=False):
    """op(A).op(B) on the GPU; shift: floats that the operands' bases are off 16 bytes."""
    M, K = a.shape
    N = b.shape[1]
    sa, sb = stored(a, opA == T_, padA), stored(b, opB == T_, padB)
    off = np.zeros(shift, np.float32)
    dA, dB = pcl.dev(np.concatenate([off, sa.ravel()])), pcl.dev(np.concatenate([off, sb.ravel()]))
    dC = pcl.dev(C0) if C0 is not None else pcl.empty((M, N), np.float32)
    dbias = pcl.dev(bias) if bias is not None else None
    pa, pb, pbias = dA.ptr + 4 * shift, dB.ptr + 4 * shift, dbias.ptr if dbias else None
    if epi is None:
        pcl.check(pcl.lib.pcl_sgemm(opA, opB, M, N, K, pa, sa.shape[1], pb, sb.shape[1], pbias,
                                    0 if C0 is None else 1, dC.ptr, N, None))
        pcl.sync()
        return dC.download((M, N), np.float32)
    daux = pcl.dev(aux) if aux is not None else None
    dpre = pcl.empty((M, N), np.float32)
    pcl.check(pcl.lib.pcl_sgemm_ex(opA, opB, M, N, K, pa, sa.shape[1], pb, sb.shape[1], pbias, epi,
                                   daux.ptr if daux else None, dpre.ptr if want_pre else None, N, dC.ptr, N, None))
    pcl.sync()
    out = dC.download((M, N), np.float32)
    return (out, dpre.download((M, N), np.float32)) if want_pre else out


def bound(a, b):
    A, B, K = np.abs(a.astype(np.float64)), np.abs(b.astype(np.float64)), a.shape[1]
    small = A.max(1)[:, None] * B.sum(0)[None, :] + A.sum(1)[:, None] * B.max(0)[None, :]
    return (3 * 2.0**-22 + (3 * K / 32 + 32) * 2.0**-24) * (A @ B) + 2.0**-38 * small


def check(C, a, b, extra=None):
    R = a.astype(np.float64) @ b.astype(np.float64)
    lim = bound(a, b)
    if extra is not None:
        R = R + extra
        lim = lim + 2.0**-22 * (np.abs(R) + np.abs(extra))
    assert (np.abs(C - R) <= lim).all(), float((np.abs(C - R) / lim).max())


# (M, N, K): the tile that the plan takes for each is beside it
SHAPES = [(4097, 3073, 97),     # 256x256, one row and one column over
          (3000, 3000, 100),    # 256x192
          (2050, 2055, 200),    # 256x128
          (1300, 5000, 130),    # 128x128, two per CU
          (1030, 2100, 300),    # 128x128, two K groups
          (300, 4100, 470),     # 64x128, two K groups
          (128, 2049, 2560),    # the narrowest output; K split
          (1000, 1200, 2305),   # K split, a tail in the last chunk
          (130, 140, 30001),    # rows held by 1024 threads; K split
          (129, 131, 66001)]    # rows read twice; K split


@pytest.mark.parametrize("opA,opB", [(N_, N_), (N_, T_), (T_, N_), (T_, T_)])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_tiles_and_layouts(M, N, K, opA, opB):
    announce("sgemm f16", M, N, K, opA, opB)
    a, b = operands(M, N, K, opA, opB, 1)
    check(run(a, b, opA, opB), a, b)


@pytest.mark.parametrize("opA,opB", [(N_, N_), (N_, T_), (T_, N_)])
@pytest.mark.parametrize("padA,padB,shift", [(4, 8, 0), (1, 3, 0), (0, 0, 1), (5, 2, 3)])
def test_strides_and_alignment(opA, opB, padA, padB, shift):
    announce("sgemm f16 strides", opA, opB, padA, padB, shift)
    a, b = operands(1024, 1280, 1088, opA, opB, 2)
    check(run(a, b, opA, opB, padA, padB, shift), a, b)


@pytest.mark.parametrize("M,N,K", [(2050, 2055, 200), (1030, 2100, 300), (1000, 1200, 2305)])
def test_bias_accumulate_and_epilogues(M, N, K):
    announce("sgemm f16 epilogues", M, N, K)
    a, b = operands(M, N, K, N_, N_, 3)
    r = np.random.default_rng(4)
    bias, old = r.standard_normal(N, np.float32), r.standard_normal((M, N), np.float32)
    check(run(a, b, N_, N_, bias=bias), a, b, bias[None, :].astype(np.float64))
    check(run(a, b, T_, N_, C0=old), a, b, old.astype(np.float64))
    check(run(a, b, N_, N_, bias=bias, epi=pcl.EPI_RESID, aux=old), a, b, bias[None, :].astype(np.float64) + old)
    # the activations' own fp32 error stays below 1e-6 of |v| + 1
    v = a.astype(np.float64) @ b.astype(np.float64) + bias
    lim = bound(a, b) + 2.0**-22 * np.abs(v)
    gelu = lambda x: 0.5 * x * (1 + np.tanh(np.sqrt(2 / np.pi) * (x + 0.044715 * x**3)))  # noqa: E731
    out, pre = run(a, b, N_, N_, bias=bias, epi=pcl.EPI_GELU, want_pre=True)
    assert (np.abs(pre - v) <= lim).all()
    assert (np.abs(out - gelu(v)) <= 1.2 * lim + 1e-6 * (np.abs(v) + 1)).all()
    u = old.astype(np.float64)
    t = np.tanh(np.sqrt(2 / np.pi) * (u + 0.044715 * u**3))
    grad = 0.5 * (1 + t) + 0.5 * u * (1 - t * t) * np.sqrt(2 / np.pi) * (1 + 3 * 0.044715 * u * u)
    out = run(a, b, N_, T_, epi=pcl.EPI_GELU_BWD, aux=old)
    v = v - bias
    assert (np.abs(out - v * grad) <= 1.2 * bound(a, b) + 2e-6 * (np.abs(v) + 1e-3)).all()


@pytest.mark.parametrize("opA,opB", [(N_, N_), (T_, T_)])
def test_rows_of_any_scale(opA, opB):
    """Rows of A and columns of B from denormals to 2^120, zero rows, single entries."""
    announce("sgemm f16 scales", opA, opB)
    a, b = operands(1030, 1100, 1000, opA, opB, 5)
    ea = np.linspace(-135, 100, 1030).astype(np.int32)
    eb = np.linspace(20, -120, 1100).astype(np.int32)
    a, b = np.ldexp(a, ea[:, None]).astype(np.float32), np.ldexp(b, eb[None, :]).astype(np.float32)
    a[7], b[:, 9] = 0, 0
    a[8] = 0
    a[8, 999] = 3
    C = run(a, b, opA, opB).astype(np.float64)
    R = a.astype(np.float64) @ b.astype(np.float64)
    tiny = 2.0**-149  # a result below the normal range is rounded to its grid
    assert (np.abs(C - R) <= bound(a, b) + tiny).all()
    assert (C[7] == 0).all() and (C[:, 9] == 0).all()
    assert np.array_equal(C[8][eb > -100], (np.float32(3) * b[999]).astype(np.float64)[eb > -100]) or \
        (np.abs(C[8] - R[8]) <= 2.0**-22 * np.abs(R[8]) + tiny).all()


@pytest.mark.parametrize("opA,opB", [(N_, N_), (N_, T_), (T_, N_)])
@pytest.mark.parametrize("M,N,K", [(1030, 1100, 1000), (300, 1100, 4500)])
def test_infinities_and_nan(M, N, K, opA, opB):
    announce("sgemm f16 nonfinite", M, N, K, opA, opB)
    a, b = operands(M, N, K, opA, opB, 6)
    a[3, 5], a[200, K - 1], a[299, 0] = np.inf, np.nan, -np.inf
    b[5, 7], b[:, 11], b[9, N - 1] = 1.0, 0.0, np.inf
    with np.errstate(invalid="ignore"):
        R = a.astype(np.float64) @ b.astype(np.float64)
    C = run(a, b, opA, opB)
    assert np.array_equal(np.isnan(C), np.isnan(R))
    inf = np.isinf(R)
    assert np.array_equal(np.isinf(C), inf) and np.array_equal(C[inf], R[inf].astype(np.float32))
    rows, cols = np.isfinite(a).all(1), np.isfinite(b).all(0)
    check(C[np.ix_(rows, cols)], a[rows], b[:, cols])


def test_graph_replays():
    """A captured product reads its operands anew on every replay."""
    announce("sgemm f16 graph")
    M, N, K = 1030, 2100, 700
    st = pcl.lib.pcl_stream_create()
    try:
        pcl.check(pcl.lib.pcl_set_stream(st))
        a, b = operands(M, N, K, N_, N_, 7)
        dA, dB, dC = pcl.dev(a), pcl.dev(b), pcl.empty((M, N), np.float32)
        import ctypes as C
        g = C.c_void_p()
        pcl.check(pcl.lib.pcl_graph_begin())
        pcl.check(pcl.lib.pcl_sgemm(N_, N_, M, N, K, dA.ptr, K, dB.ptr, N, None, 0, dC.ptr, N, st))
        pcl.check(pcl.lib.pcl_graph_end(C.byref(g)))
        for seed in (7, 8, 9):
            a, b = operands(M, N, K, N_, N_, seed)
            if seed == 8:
                a[4, 4] = np.inf
            dA.upload(a), dB.upload(b)
            pcl.check(pcl.lib.pcl_graph_launch(g))
            pcl.sync()
            got = dC.download((M, N), np.float32)
            fin = np.isfinite(a).all(1)
            check(got[fin], a[fin], b)
            assert not np.isfinite(got[~fin]).any()
            pcl.check(pcl.lib.pcl_sgemm(N_, N_, M, N, K, dA.ptr, K, dB.ptr, N, None, 0, dC.ptr, N, st))
            pcl.sync()
            assert np.array_equal(got[fin], dC.download((M, N), np.float32)[fin])
        pcl.check(pcl.lib.pcl_graph_destroy(g))
    finally:
        pcl.lib.pcl_set_stream(None)
        pcl.check(pcl.lib.pcl_stream_destroy(st))
