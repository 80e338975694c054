"""Masked attention where its numbers leave the ordinary range: additive masks of
large finite values, scores past the point where floats are whole numbers apart,
queries and keys of zeros or nearly so, blocked keys that hold anything.

Against double-precision softmax. A mask value m leaves a score s + m its fp32
rounding, half an ulp of m: where that matters the expectation is taken from the
rounded scores. Tolerance: fp32 sums, 2e-6 of the result's 2-norm (2e-7 is seen).
"""

import math

import numpy as np
import pytest

from test_gpu_attention import LOWEST, naive

pytestmark = pytest.mark.gpu

HD = 64


def rel(got, want):
    return float(np.linalg.norm(got - want) / np.linalg.norm(want))


def qkv(seed, sq, sk, nq=2, nkv=2, hd=HD):
    r = np.random.default_rng(seed)
    return tuple(r.standard_normal((n, h * hd), dtype=np.float32) for n, h in ((sq, nq), (sk, nkv), (sk, nkv)))


def rounded(Q, K, V, nq, nkv, hd, scale, mask):
    """naive() with the scores rounded to fp32 where the mask is added."""
    sq, sk = len(Q), len(K)
    q, k, v = (x.astype(np.float64).reshape(len(x), -1, hd) for x in (Q, K, V))
    out = np.zeros((sq, nq, hd))
    for h in range(nq):
        s = (q[:, h] @ k[:, h // (nq // nkv)].T * scale).astype(np.float32)
        with np.errstate(over="ignore"):
            s = np.where(mask == LOWEST, np.float32(-np.inf), s + mask).astype(np.float64)
        mx = s.max(axis=1, keepdims=True)
        with np.errstate(invalid="ignore"):
            e = np.where(np.isneginf(s), 0.0, np.exp(s - mx))
        z = e.sum(axis=1, keepdims=True)
        out[:, h] = np.where(z == 0, v[:, h // (nq // nkv)].mean(axis=0), (e @ v[:, h // (nq // nkv)]) / np.where(z == 0, 1, z))
    return out.reshape(sq, nq * hd)


@pytest.mark.parametrize("sq,sk", [(1, 33), (20, 70), (50, 300), (700, 300)])
@pytest.mark.parametrize("m", [-1e4, -3e6, -1e7, -3e7, -1e8, -1e9, -1e30])
def test_large_finite_masks(vla, m, sq, sk):
    """Padding written as an additive value: trailing and leading key ranges (whole
    32-key tiles of a wave among them), single keys, and rows with nothing else."""
    Q, K, V = qkv(sq + sk, sq, sk)
    r = np.random.default_rng(2)
    mask = np.zeros((sq, sk), np.float32)
    mask[0::4, sk // 3:] = m
    mask[1::4, :sk // 2 + 3] = m
    mask[2::4][r.random((len(mask[2::4]), sk)) < 0.3] = m
    mask[3::8] = m
    mask[7::8] = m
    mask[7::8, sk // 2] = LOWEST
    got = vla.attention(Q, K, V, 2, 2, HD, 0.125, kind=vla.MASK_DENSE, dense=mask)
    want = rounded(Q, K, V, 2, 2, HD, 0.125, mask)
    mine = np.abs(got - want).max(axis=1)
    # where every key carries the mask the weights hang on the last bit of s + m,
    # whose product and sum may round once or twice: one step either way
    whole = (mask != 0).all(axis=1)
    assert np.isfinite(got).all()
    assert rel(got[~whole], want[~whole]) < 2e-6, mine.max()
    ulp = float(np.spacing(np.float32(-m)))
    if whole.any():
        if ulp > 64:  # every score is absorbed: the weights are equal
            assert rel(got[whole], want[whole]) < 2e-6
        else:
            bound = 2 * np.expm1(min(2.0, ulp)) * np.abs(V).max() + 1e-5
            assert mine[whole].max() < bound


@pytest.mark.parametrize("low", [-2.4e38, -3.3e38, -3.3895314e38])
def test_masks_next_to_lowest(vla, low):
    """Values between lowest() and its quotient by log2 e are additive like any
    other (bf16's lowest is one): only lowest() and -inf block."""
    sq, sk = 40, 200
    Q, K, V = qkv(3, sq, sk)
    low = np.float32(low)
    mask = np.full((sq, sk), LOWEST, np.float32)
    mask[:, 20:90] = low
    mask[::2, 150] = 0
    mask[1::4, 40:60] = low * np.float32(0.9)
    got = vla.attention(Q, K, V, 2, 2, HD, 0.125, kind=vla.MASK_DENSE, dense=mask)
    assert rel(got, rounded(Q, K, V, 2, 2, HD, 0.125, mask)) < 2e-6


@pytest.mark.parametrize("kind", ["none", "causal", "groups", "dense"])
@pytest.mark.parametrize("size", [1e7, 1e8, 1e10, 1e20])
def test_scores_past_whole_numbers(vla, size, kind):
    """Scores whose floats lie more than one apart: the largest takes all."""
    sq, sk = 40, 300
    Q, K, V = qkv(9, sq, sk)
    Q = (Q * np.float32(size)).astype(np.float32)
    kw, keep = {}, np.ones((sq, sk), bool)
    if kind == "causal":
        keep = np.arange(sk)[None] <= np.arange(sq)[:, None] + 5
        kw = dict(kind=vla.MASK_CAUSAL, causal_offset=5)
    elif kind == "groups":
        r = np.random.default_rng(1)
        qg, kg = r.integers(0, 9, sq).astype(np.uint8), r.integers(0, 9, sk).astype(np.uint8)
        allow = (r.random((9, 9)) < 0.5).astype(np.uint8)
        allow[np.arange(9), np.arange(9)] = 1
        keep = allow[qg][:, kg].astype(bool)
        kw = dict(kind=vla.MASK_GROUPS, q_group=qg, k_group=kg, allow=allow.reshape(-1))
    elif kind == "dense":
        kw = dict(kind=vla.MASK_DENSE, dense=np.zeros((sq, sk), np.float32))
    got = vla.attention(Q, K, V, 2, 2, HD, 0.125, **kw)
    assert np.isfinite(got).all()
    want = naive(Q, K, V, sq, sk, 2, 2, HD, 0.125, np.where(keep, 0, -np.inf).astype(np.float32))
    # rows whose two largest scores lie apart by more than the scores' fp32 error
    q, k = (x.astype(np.float64).reshape(-1, 2, HD) for x in (Q, K))
    for h in range(2):
        s = np.where(keep, q[:, h] @ k[:, h].T * 0.125, -np.inf)
        top = np.sort(s, axis=1)[:, -2:]
        clear = top[:, 1] - top[:, 0] > 40 + 4e-6 * np.linalg.norm(q[:, h], axis=1) * np.linalg.norm(k[:, h], axis=1).max() * 0.125
        assert clear.sum() > sq // 2
        assert rel(got[clear, h * HD:(h + 1) * HD], want[clear, h * HD:(h + 1) * HD]) < 2e-6


def masks_of(vla, kind, sq, sk):
    if kind == "causal":
        return dict(kind=vla.MASK_CAUSAL, causal_offset=2), np.arange(sk)[None] <= np.arange(sq)[:, None] + 2
    if kind == "groups":
        qg, kg = (np.arange(sq) % 5).astype(np.uint8), (np.arange(sk) // 7 % 5).astype(np.uint8)
        allow = np.tril(np.ones((5, 5), np.uint8))
        return dict(kind=vla.MASK_GROUPS, q_group=qg, k_group=kg, allow=allow.reshape(-1)), allow[qg][:, kg].astype(bool)
    if kind == "dense":
        keep = np.random.default_rng(5).random((sq, sk)) < 0.6
        return dict(kind=vla.MASK_DENSE, dense=np.where(keep, 0, LOWEST).astype(np.float32)), keep
    return {}, np.ones((sq, sk), bool)


@pytest.mark.parametrize("kind", ["none", "causal", "groups", "dense"])
@pytest.mark.parametrize("q,k", [(0, 0), (0, 1), (1, 0), (0, 2.0 ** -9), (1e-20, 1e-20), (1e-30, 1e-15), (1e-38, 1e-38)])
@pytest.mark.parametrize("sq,sk", [(5, 33), (40, 300)])
def test_zero_and_tiny_scores(vla, kind, q, k, sq, sk):
    """Queries and keys of zeros or whose products underflow: equal weights."""
    Q, K, V = qkv(11, sq, sk)
    Q, K = (Q * np.float32(q)).astype(np.float32), (K * np.float32(k)).astype(np.float32)
    kw, keep = masks_of(vla, kind, sq, sk)
    got = vla.attention(Q, K, V, 2, 2, HD, 0.125, **kw)
    assert rel(got, naive(Q, K, V, sq, sk, 2, 2, HD, 0.125, np.where(keep, 0, -np.inf).astype(np.float32))) < 2e-6


@pytest.mark.parametrize("kind", ["causal", "groups", "dense"])
def test_some_zero_rows(vla, kind):
    """Zero query rows and zero 32-key tiles among ordinary ones."""
    sq, sk = 70, 300
    Q, K, V = qkv(12, sq, sk)
    Q[3::5] = 0
    K[64:128] = 0
    K *= np.float32(2.0 ** -10)
    kw, keep = masks_of(vla, kind, sq, sk)
    got = vla.attention(Q, K, V, 2, 2, HD, 0.125, **kw)
    assert rel(got, naive(Q, K, V, sq, sk, 2, 2, HD, 0.125, np.where(keep, 0, -np.inf).astype(np.float32))) < 2e-6


@pytest.mark.parametrize("kind", ["causal", "groups", "dense"])
@pytest.mark.parametrize("which", ["k", "v", "kv"])
@pytest.mark.parametrize("size", [1e3, 1e5, 1e6, 1e12, 1e30, 3e38])
def test_blocked_keys_of_any_size(vla, kind, which, size):
    """Rows that the mask blocks for every query (padding, the stale end of a cache)
    may hold any finite value: they weigh exactly nothing, and the others keep
    their full precision."""
    sq, sk = 40, 200
    Q, K, V = qkv(13, sq, sk)
    if kind == "causal":
        keep = np.arange(sk)[None] <= np.arange(sq)[:, None] + 20
        kw = dict(kind=vla.MASK_CAUSAL, causal_offset=20)
    else:
        pad = np.zeros(sk, bool)
        pad[[0, 1, 17, 40, 95]] = True
        pad[130:150] = True
        keep = np.broadcast_to(~pad, (sq, sk))
        if kind == "groups":
            kw = dict(kind=vla.MASK_GROUPS, q_group=np.zeros(sq, np.uint8), k_group=pad.astype(np.uint8),
                      allow=np.array([1, 0, 0, 0], np.uint8))
        else:
            kw = dict(kind=vla.MASK_DENSE, dense=np.where(keep, 0, LOWEST).astype(np.float32))
    out = ~keep.any(axis=0)
    mask = np.where(keep, 0, -np.inf).astype(np.float32)
    want = naive(Q, K, V, sq, sk, 2, 2, HD, 0.125, mask)
    for x, name in ((K, "k"), (V, "v")):
        if name in which:
            x[out] = np.sign(x[out]) * np.float32(size)
    assert rel(vla.attention(Q, K, V, 2, 2, HD, 0.125, **kw), want) < 2e-6


@pytest.mark.parametrize("what", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("kind", ["causal", "groups", "dense", "dense-inf"])
def test_not_finite_behind_a_mask(vla, kind, what):
    """Infinities and NaN in a key or value reach only the queries that see it."""
    sq, sk = 140, 300
    Q, K, V = qkv(14, sq, sk)
    at = 100
    if kind == "causal":
        keep = np.arange(sk)[None] <= np.arange(sq)[:, None]
        kw = dict(kind=vla.MASK_CAUSAL, causal_offset=0)
    else:
        qg = (np.arange(sq) >= 60).astype(np.uint8)
        keep = np.ones((sq, sk), bool)
        keep[:60, at - 5:at + 9] = False
        if kind == "groups":
            kg = np.zeros(sk, np.uint8)
            kg[at - 5:at + 9] = 1
            kw = dict(kind=vla.MASK_GROUPS, q_group=qg, k_group=kg, allow=np.array([1, 0, 1, 1], np.uint8))
        else:
            kw = dict(kind=vla.MASK_DENSE, dense=np.where(keep, 0, LOWEST if kind == "dense" else -np.inf).astype(np.float32))
    want = naive(Q, K, V, sq, sk, 2, 2, HD, 0.125, np.where(keep, 0, -np.inf).astype(np.float32))
    blind = ~keep[:, at]
    assert blind.sum() >= 60
    for x in (K, V):
        y = x.copy()
        y[at, 3] = what
        got = vla.attention(Q, y if x is K else K, y if x is V else V, 2, 2, HD, 0.125, **kw)
        assert rel(got[blind], want[blind]) < 2e-6
        assert rel(got[:, HD:], want[:, HD:]) < 2e-6  # the other head
        if x is V:
            assert rel(got[:, 4:], want[:, 4:]) < 2e-6 and not np.isfinite(got[~blind, 3]).any()


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("size", [1e-36, 1e-33, 1e33, 1e36])
def test_values_near_the_range_ends(vla, hd, size):
    sq, sk = 40, 200
    Q, K, V = qkv(15, sq, sk, hd=hd)
    V = (V * np.float32(size)).astype(np.float32)
    got = vla.attention(Q, K, V, 2, 2, hd, 1 / math.sqrt(hd))
    want = naive(Q, K, V, sq, sk, 2, 2, hd, 1 / math.sqrt(hd))
    assert rel(got / size, want / size) < 2e-6
    one = V.copy()
    one[:, 5] /= np.float32(size)  # a column of its own size keeps its own precision
    got = vla.attention(Q, K, one, 2, 2, hd, 1 / math.sqrt(hd))
    want = naive(Q, K, one, sq, sk, 2, 2, hd, 1 / math.sqrt(hd))
    for cols, unit in ((np.arange(2 * hd) == 5, 1.0), (np.arange(2 * hd) != 5, size)):
        assert rel(got[:, cols] / unit, want[:, cols] / unit) < 2e-6


@pytest.mark.parametrize("what", ["q", "k"])
@pytest.mark.parametrize("size", [1e-36, 1e36])
def test_scores_of_far_operands(vla, what, size):
    """Queries and keys near opposite ends of the range, their scores ordinary."""
    sq, sk = 40, 200
    Q, K, V = qkv(16, sq, sk)
    f = np.float32(size)
    Q, K = (Q * f, K / f) if what == "q" else (Q / f, K * f)
    got = vla.attention(Q, K, V, 2, 2, HD, 0.125)
    assert rel(got, naive(Q, K, V, sq, sk, 2, 2, HD, 0.125)) < 2e-6


def test_operands_of_mixed_sizes(vla):
    """Keys, values and their columns over 2^-30 .. 2^30 in one tile: each key's score
    and each column's sum keep fp32's precision of their own size."""
    sq, sk = 40, 300
    Q, K, V = qkv(17, sq, sk)
    r = np.random.default_rng(3)
    cols = np.exp2(r.integers(-30, 31, V.shape[1])).astype(np.float32)
    dims = np.exp2(r.integers(-30, 31, K.shape[1])).astype(np.float32)
    got = vla.attention(Q / dims, K * dims, V * cols, 2, 2, HD, 0.125)
    want = naive(Q / dims, K * dims, V * cols, sq, sk, 2, 2, HD, 0.125)
    err = np.linalg.norm(got - want, axis=0) / np.linalg.norm(want, axis=0)
    assert err.max() < 4e-6, err.max()


@pytest.mark.parametrize("sq,sk,nq,hd", [(40, 60, 2, 64), (40, 100, 2, 64), (1400, 70, 12, 64), (40, 300, 2, 64), (400, 290, 12, 64),
                                         (700, 290, 12, 64), (1040, 290, 12, 64), (1100, 300, 12, 32), (40, 90, 3, 128),
                                         (600, 90, 8, 100)])
@pytest.mark.parametrize("kind", ["none", "causal", "groups", "dense"])
def test_plain_form_of_every_block_shape(vla, sq, sk, nq, hd, kind):
    """One infinite value of V sends every block of its head to the plain form, at each
    count of queries and waves per block; the other columns are what they are without."""
    Q, K, V = qkv(sq + hd, sq, sk, nq, nq, hd)
    kw, keep = masks_of(vla, kind, sq, sk)
    scale = 1 / math.sqrt(hd)
    want = naive(Q, K, V, sq, sk, nq, nq, hd, scale, np.where(keep, 0, -np.inf).astype(np.float32))
    V[0, hd + 3] = np.inf  # head 1
    got = vla.attention(Q, K, V, nq, nq, hd, scale, **kw)
    rest = np.arange(nq * hd) != hd + 3
    assert rel(got[:, rest], want[:, rest]) < 2e-6
    sees = keep[:, 0] | ~keep.any(axis=1)
    assert not np.isfinite(got[sees, hd + 3]).any()
    assert np.isfinite(got[~sees, hd + 3]).all()
