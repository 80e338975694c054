"""Attention over the layouts that the models use it in: q, k and v as column ranges of
one row (strides of three heads' widths and of odd paddings), outputs into a range of
a wider row whose other columns stay, and group masks over more keys than the key
groups' place in LDS (4096), with tables of up to 64 groups and of more.
"""

import math

import numpy as np
import pytest

from test_gpu_attention import naive
from test_gpu_attention_split import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sq,nq,nkv,hd,pad", [(302, 8, 8, 64, 0), (700, 12, 12, 64, 0), (177, 15, 5, 64, 20), (60, 4, 2, 128, 4),
                                              (90, 3, 3, 32, 12), (40, 2, 1, 200, 8)])
@pytest.mark.parametrize("kind", ["none", "causal"])
def test_interleaved(vla, torch_cuda, sq, nq, nkv, hd, pad, kind):
    torch = torch_cuda
    qw, kw = nq * hd, nkv * hd
    r = np.random.default_rng(sq)
    rows = r.standard_normal((sq, qw + 2 * kw + pad), dtype=np.float32)
    rows[:, qw + 2 * kw:] = np.nan  # the padding is nobody's
    x = torch.from_numpy(rows).cuda()
    out = torch.full((sq, qw + 8), 7.0, device="cuda")
    m = vla.VlaMask(kind=vla.MASK_CAUSAL, causal_offset=0) if kind == "causal" else None
    scale = 1 / math.sqrt(hd)
    vla.attention_dev(out[:, 4:4 + qw], x[:, :qw], x[:, qw:qw + kw], x[:, qw + kw:qw + 2 * kw], nq, nkv, hd, scale, m)
    mask = np.where(np.arange(sq)[None] > np.arange(sq)[:, None], -np.inf, 0).astype(np.float32) if m else None
    want = naive(rows[:, :qw].copy(), rows[:, qw:qw + kw].copy(), rows[:, qw + kw:qw + 2 * kw].copy(), sq, sq, nq, nkv, hd,
                 scale, mask)
    got = out.cpu().numpy()
    assert rel(got[:, 4:4 + qw], want) < 2e-6
    assert (got[:, :4] == 7).all() and (got[:, 4 + qw:] == 7).all()


@pytest.mark.parametrize("sk", [4096, 4097, 5003])
@pytest.mark.parametrize("groups", [40, 64, 65, 200])
def test_groups_over_many_keys(vla, sk, groups):
    sq, n, hd = 70, 2, 64
    r = np.random.default_rng(sk + groups)
    Q, K, V = (r.standard_normal((s, n * hd), dtype=np.float32) for s in (sq, sk, sk))
    qg, kg = r.integers(0, groups, sq).astype(np.uint8), np.sort(r.integers(0, groups, sk)).astype(np.uint8)
    allow = (r.random((groups, groups)) < 0.3).astype(np.uint8)
    allow[qg[5]] = 0  # a query with nothing to see
    mask = np.where(allow[qg][:, kg], 0, -np.inf).astype(np.float32)
    got = vla.attention(Q, K, V, n, n, hd, 0.125, kind=vla.MASK_GROUPS, q_group=qg, k_group=kg, allow=allow.reshape(-1))
    assert rel(got, naive(Q, K, V, sq, sk, n, n, hd, 0.125, mask)) < 2e-6
