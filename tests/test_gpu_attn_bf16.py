"""Attention on the bf16 matrix cores (csrc/attn.hip) against float64: every remainder of
its 32-key blocks and 128-query workgroups, both groups of waves empty or not, dS kept or
formed again, and rows that infinities and NaN send to the fp32 fma path.

Bounds (max |x - r| / max |r|): a score is a sum of 6 dh/16 <= 48 matrix-core additions of
three-way split operands, each rounded to 2^-24 of a partial sum: 48 2^-24 of sum |q||k|,
which for these inputs is below 8 in the exponent's units, so a probability is within 8 *
48 * 2^-24 = 2.3e-5; the sums over at most 300 keys add 6 * 300/16 * 2^-24 = 7e-6.
"""
import numpy as np
import pytest

import pcl
from gpu_util import announce, require_device

pytestmark = pytest.mark.gpu
TOL = 3e-5


@pytest.fixture(scope="module", autouse=True)
def _device():
    require_device()


def inputs(B, T, H, dh, seed):
    r = np.random.default_rng(seed)
    return [r.standard_normal((B, T, H, dh), np.float32) for _ in range(4)]


def reference(q, k, v, do):
    """Per (b, h) in float64; infinities and NaN follow from the formulas, key by key."""
    B, T, H, dh = q.shape
    o = {n: np.zeros((B, T, H, dh)) for n in ("att", "dq", "dk", "dv")}
    o["p"], o["lse"] = np.zeros((B, H, T, T)), np.zeros((B, H, T))
    with np.errstate(all="ignore"):
        for b in range(B):
            for h in range(H):
                Q, K, V, D = (x[b, :, h].astype(np.float64) for x in (q, k, v, do))
                S = Q @ K.T / np.sqrt(dh)
                for i in range(T):
                    s = S[i, :i + 1]
                    m = np.max(s) if not np.isnan(s).any() else np.nan
                    e = np.exp(s - m)
                    p = e / e.sum()
                    o["p"][b, h, i, :i + 1], o["lse"][b, h, i] = p, m + np.log(e.sum())
                    o["att"][b, i, h] = p @ V[:i + 1]
                    dp = V[:i + 1] @ D[i]
                    ds = p * (dp - D[i] @ o["att"][b, i, h]) / np.sqrt(dh)
                    o["dq"][b, i, h] = ds @ K[:i + 1]
                    o["dk"][b, :i + 1, h] += ds[:, None] * Q[i][None, :]
                    o["dv"][b, :i + 1, h] += p[:, None] * D[i][None, :]
    return o


def gpu(q, k, v, do, scratch, with_att):
    B, T, H, dh = q.shape
    D, n = H * dh, B * T * H * dh
    bufs = [pcl.dev(x.reshape(B * T, D)) for x in (q, k, v, do)]
    att, one, p, lse = pcl.empty((n,), np.float32), pcl.empty((n,), np.float32), pcl.empty((B * H * T * T,), np.float32), \
        pcl.empty((B * H * T,), np.float32)
    g = [pcl.empty((n,), np.float32) for _ in range(3)]
    ds = pcl.empty((B * H * T * T,), np.float32) if scratch else None
    Q, K, V, dO = (b.ptr for b in bufs)
    pcl.check(pcl.lib.pcl_attn_fwd(Q, K, V, D, att.ptr, D, p.ptr, B, T, H, dh, None))
    pcl.check(pcl.lib.pcl_attn_fwd_lse(Q, K, V, D, one.ptr, D, lse.ptr, B, T, H, dh, None))
    sc = ds.ptr if scratch else None
    if with_att:
        pcl.check(pcl.lib.pcl_attn_bwd_ex(g[0].ptr, g[1].ptr, g[2].ptr, D, sc, dO, D, Q, K, V, D, p.ptr, att.ptr, D,
                                          B, T, H, dh, 0, None))
    else:
        pcl.check(pcl.lib.pcl_attn_bwd(g[0].ptr, g[1].ptr, g[2].ptr, D, sc, dO, D, Q, K, V, D, p.ptr, B, T, H, dh, 0, None))
    pcl.sync()
    o = {n_: b.download((B, T, H, dh), np.float32) for n_, b in zip(("att", "one", "dq", "dk", "dv"), [att, one] + g)}
    o["p"], o["lse"] = p.download((B, H, T, T), np.float32), lse.download((B, H, T), np.float32)
    return o


def close(x, r):
    return np.abs(x - r).max() <= TOL * np.abs(r).max()


@pytest.mark.parametrize("dh", [32, 64, 128])
@pytest.mark.parametrize("T", [1, 31, 32, 33, 64, 65, 96, 127, 129, 161, 257, 300])
def test_edges(T, dh):
    announce("attn bf16", T, dh)
    x = inputs(2, T, 2, dh, T + dh)
    r = reference(*x)
    for scratch, with_att in ((False, True), (True, True), (False, False), (True, False)):
        o = gpu(*x, scratch, with_att)
        for n, m in (("att", "att"), ("one", "att"), ("p", "p"), ("lse", "lse"), ("dq", "dq"), ("dk", "dk"), ("dv", "dv")):
            assert close(o[n], r[m]) or T == 1 and n in ("dq", "dk"), (n, scratch, with_att)  # T = 1: dS is 0
        assert (np.triu(np.ones((T, T)), 1) * o["p"] == 0).all()


@pytest.mark.parametrize("dh", [32, 64, 128])
@pytest.mark.parametrize("scratch", [False, True])
def test_infinities_and_nan(dh, scratch):
    announce("attn bf16 nonfinite", dh, scratch)
    q, k, v, do = inputs(1, 200, 4, dh, dh)
    k[0, 50, 0, 3] = -np.inf   # head 0: rows >= 50 score -inf (weight 0) or +inf (NaN) at key 50
    v[0, 70, 1, 2] = np.inf    # head 1: rows >= 70 are infinite in one column
    q[0, 90, 2, 1] = np.nan    # head 2: one row
    do[0, 150, 3, 5] = np.inf  # head 3: the backward of rows and keys up to 150
    with np.errstate(all="ignore"):
        r = reference(q, k, v, do)
    o = gpu(q, k, v, do, scratch, True)
    fin = lambda x: np.isfinite(x)  # noqa: E731
    for n, m, head in (("att", "att", 0), ("one", "att", 0), ("att", "att", 1), ("one", "att", 1), ("att", "att", 2),
                       ("one", "att", 2), ("dv", "dv", 3)):
        X, R = o[n][:, :, head], r[m][:, :, head]
        assert np.array_equal(np.isnan(X), np.isnan(R)) and np.array_equal(np.isinf(X), np.isinf(R)), (n, head)
        assert close(np.where(fin(R), X, 0), np.where(fin(R), R, 0)), (n, head)
    seen = np.tril(np.ones((200, 200), bool))
    assert np.array_equal(np.isnan(o["p"])[:, :, seen], np.isnan(r["p"])[:, :, seen])
    # what no infinity reaches is as ever
    for n in ("dq", "dk", "dv"):
        X, R = o[n][:, :, 3], r[n][:, :, 3]
        assert fin(X[:, 151:]).all() and close(X[:, 151:], R[:, 151:]), n
    assert close(o["dq"][:, :150, 3], r["dq"][:, :150, 3])
