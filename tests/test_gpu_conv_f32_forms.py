"""The fp32 convolutions' implicit form against im2col + GEMM, bit for bit, where
the scales that both take by guess differ from row to row: filters of mixed
sizes, images with flat and bright parts, and Octo's stems, whose second layer has
32 channels (half of the widest slab), over even maps and over odd ones whose last
pixel is a patch's centre.
"""

import os

import numpy as np
import pytest

from helpers import load_pkg

pytestmark = pytest.mark.gpu


def _ck():
    load_pkg()
    import vla_simd_amd.checkpoints as ck
    return ck


def both(monkeypatch, call):
    monkeypatch.setenv("VLA_CONV_F32_IMPLICIT", "0")
    want = call()
    monkeypatch.delenv("VLA_CONV_F32_IMPLICIT")
    return call(), want


@pytest.mark.parametrize("H,W", [(240, 320), (97, 130)])
def test_trunk(vla, monkeypatch, tmp_path, H, W):
    ck = _ck()
    d = ck.write_act_model(str(tmp_path / "act"), dict(ck.ACT_MODEL_BASE, img_h=H, img_w=W, n_cams=1, n_enc=1, ff=256))
    p = os.path.join(d, "backbone.bin")
    raw = np.fromfile(p, np.float32)
    r = np.random.default_rng(1)
    raw *= np.exp2(r.integers(-3, 2, raw.size)).astype(np.float32)
    raw.tofile(p)
    monkeypatch.setenv("ACT_INT8", "31")
    images = r.integers(0, 256, (1, H, W, 3), dtype=np.uint8)
    images[:, H // 3:H // 2] = 0
    images[:, :, W // 2:W // 2 + 9] = 255
    got, want = both(monkeypatch, lambda: vla.ActModel(d).encode(images))
    assert np.isfinite(want).all() and np.abs(want).max() > 0
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("stride,tokens", [(2, (256, 64)), (3, (16, 4))])
def test_octo_stems(vla, monkeypatch, tmp_path, stride, tokens):
    ck = _ck()
    c = dict(t5=dict(ck.T5_BASE, d_model=128, n_layers=1, n_heads=2, d_kv=64, d_ff=256, vocab=1024),
             stem=dict(ck.OCTO_STEM_BASE, features=(32, 96, 64, 64), embed_dim=64, gn_groups=8),
             tf=dict(ck.OCTO_BASE, d=128, n_layers=1, heads=2, head_dim=64, mlp=256, max_horizon=2, stem_dim=64, t5_dim=128,
                     repeat_task=1, tok_primary=tokens[0], tok_wrist=tokens[1]),
             head=dict(ck.OCTO_HEAD_BASE, hidden=64, num_blocks=1, steps=2))
    d = ck.write_octo_model(str(tmp_path / "octo"), c)
    for name in ("stem_primary", "stem_wrist"):
        with open(os.path.join(d, name + ".meta"), "a") as f:
            f.write(f"stride {stride}\n")
    monkeypatch.delenv("OCTO_INT8", raising=False)
    p, w, tm, n, z = ck.octo_model_inputs(c)
    got, want = both(monkeypatch, lambda: vla.OctoModel(d).predict(p, w, tm, "pick up the red block", noise=n, z=z))
    assert np.isfinite(want).all() and np.abs(want).max() > 0
    np.testing.assert_array_equal(got, want)
