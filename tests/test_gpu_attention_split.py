"""The fp16-part attention kernel at the edges of its dispatch.

Query fragments per block (1 to 4) and waves (2, 4, 8) follow from the sizes;
the sizes here lie on both sides of each of those lines, of the 16-query and
32-key tiles and of the head widths. Against double-precision softmax: the
parts keep every operand to 2^-22 of itself or 2^-40 of the largest that shares
its scale, so the outputs are held to what fp32 sums give (2e-6 of the result's
2-norm; about 2e-7 is seen).
"""

import math

import numpy as np
import pytest

from test_gpu_attention import LOWEST, naive

pytestmark = pytest.mark.gpu


def rel(got, want):
    return float(np.linalg.norm(got - want) / np.linalg.norm(want))


def qkv(seed, sq, sk, nq, nkv, hd):
    r = np.random.default_rng(seed)
    return tuple(r.standard_normal((n, h * hd), dtype=np.float32) for n, h in ((sq, nq), (sk, nkv), (sk, nkv)))


@pytest.mark.parametrize("sq,sk,nq,nkv,hd", [
    (1, 1, 1, 1, 64), (15, 31, 2, 1, 64), (17, 33, 15, 5, 64), (16, 64, 4, 4, 64), (17, 65, 4, 2, 64),  # W 2, 4
    (33, 256, 8, 8, 64), (33, 257, 8, 8, 64),                                                          # W 4, 8
    (336, 290, 12, 12, 64), (352, 290, 12, 12, 64),   # 21 and 22 fragments x 12: one and two per block
    (672, 290, 12, 12, 64), (688, 290, 12, 12, 64),   # two and three
    (1008, 290, 12, 4, 64), (1040, 290, 12, 4, 64),   # three and four
    (1400, 70, 12, 12, 64),                           # past one round, 4 waves
    (40, 300, 3, 1, 4), (40, 300, 3, 1, 60), (700, 300, 12, 12, 32), (1100, 300, 12, 12, 32),
    (40, 300, 3, 1, 68), (40, 300, 3, 1, 128), (600, 90, 8, 8, 128), (600, 90, 8, 8, 100),
])
@pytest.mark.parametrize("kind", ["none", "dense", "causal", "groups"])
def test_sizes(vla, sq, sk, nq, nkv, hd, kind):
    Q, K, V = qkv(sq * 7 + sk, sq, sk, nq, nkv, hd)
    scale = np.float32(1 / math.sqrt(hd))
    r = np.random.default_rng(5)
    kw, mask = {}, None
    if kind == "dense":
        mask = np.where(r.random((sq, sk)) < 0.3, LOWEST, r.standard_normal((sq, sk))).astype(np.float32)
        mask[sq // 2] = -np.inf  # a row with nothing to see
        kw = dict(kind=vla.MASK_DENSE, dense=mask)
    elif kind == "causal":
        mask = np.where(np.arange(sk)[None] > np.arange(sq)[:, None] + 3, -np.inf, 0).astype(np.float32)
        kw = dict(kind=vla.MASK_CAUSAL, causal_offset=3)
    elif kind == "groups":
        G = 70 if sk > 256 else 40  # past and within the two-word rows of the table
        qg, kg = r.integers(0, G, sq).astype(np.uint8), np.sort(r.integers(0, G, sk)).astype(np.uint8)
        allow = (r.random((G, G)) < 0.4).astype(np.uint8)
        allow[3] = 0
        mask = np.where(allow[qg][:, kg], 0, -np.inf).astype(np.float32)
        kw = dict(kind=vla.MASK_GROUPS, q_group=qg, k_group=kg, allow=allow.reshape(-1))
    got = vla.attention(Q, K, V, nq, nkv, hd, scale, **kw)
    assert rel(got, naive(Q, K, V, sq, sk, nq, nkv, hd, float(scale), mask)) < 2e-6


@pytest.mark.parametrize("what", ["k", "v", "q"])
@pytest.mark.parametrize("size", [1e-30, 1e-12, 1e12, 1e30])
def test_magnitudes(vla, what, size):
    """Operands far from 1 (the scales are theirs), some rows of V far from the others."""
    Q, K, V = qkv(3, 60, 200, 4, 2, 64)
    x = {"q": Q, "k": K, "v": V}
    x[what] = (x[what] * np.float32(size)).astype(np.float32)
    if what != "v":
        other = "k" if what == "q" else "q"
        x[other] = (x[other] / np.float32(size)).astype(np.float32)
    x["v"] = (x["v"] * np.exp2(np.random.default_rng(1).integers(-6, 7, (200, 1)))).astype(np.float32)
    got = vla.attention(x["q"], x["k"], x["v"], 4, 2, 64, 0.125)
    assert rel(got, naive(x["q"], x["k"], x["v"], 60, 200, 4, 2, 64, 0.125)) < 2e-6


def test_growing_tiles(vla):
    """Each 32-key tile of K and V larger than the last: every scale changes on the way."""
    Q, K, V = qkv(4, 40, 1024, 2, 2, 64)
    K = (K * np.exp2(np.arange(1024) // 32 / 8 - 3)[:, None]).astype(np.float32)
    V = (V * np.exp2(np.arange(1024) // 32 - 16)[:, None]).astype(np.float32)
    got = vla.attention(Q, K, V, 2, 2, 64, 0.125)
    assert rel(got, naive(Q, K, V, 40, 1024, 2, 2, 64, 0.125)) < 2e-6


@pytest.mark.parametrize("scale", [-0.125, 0.0])
def test_scale_sign(vla, scale):
    Q, K, V = qkv(6, 40, 300, 2, 2, 64)
    mask = np.where(np.arange(300)[None] > np.arange(40)[:, None], -np.inf, 0).astype(np.float32)
    got = vla.attention(Q, K, V, 2, 2, 64, scale, kind=vla.MASK_CAUSAL, causal_offset=0)
    assert rel(got, naive(Q, K, V, 40, 300, 2, 2, 64, scale, mask)) < 2e-6


def test_infinities(vla):
    """-inf scores (a key of infinities against queries of one sign) weigh nothing; an
    infinite value reaches only the outputs of its own column; NaN stays NaN."""
    Q, K, V = qkv(8, 50, 300, 2, 2, 64)
    Q = np.abs(Q) + np.float32(0.01)
    Ki = K.copy()
    Ki[37, :64] = -np.inf  # head 0
    keep = np.zeros((50, 300), np.float32)
    keep[:, 37] = -np.inf
    want = naive(Q, K, V, 50, 300, 2, 2, 64, 0.125)
    want[:, :64] = naive(Q, K, V, 50, 300, 2, 2, 64, 0.125, keep)[:, :64]
    assert rel(vla.attention(Q, Ki, V, 2, 2, 64, 0.125), want) < 2e-6
    for bad in (np.inf, np.nan):
        Vi = V.copy()
        Vi[200, 70] = bad  # head 1, dim 6
        got = vla.attention(Q, K, Vi, 2, 2, 64, 0.125)
        cols = np.arange(128) != 70
        assert not np.isfinite(got[:, 70]).any()
        assert rel(got[:, cols], naive(Q, K, V, 50, 300, 2, 2, 64, 0.125)[:, cols]) < 2e-6
