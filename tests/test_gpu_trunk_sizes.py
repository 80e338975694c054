"""The fp32 image trunk against float64 at odd image sizes: stem pixel counts
and rows that are no multiple of the stem gather's four pixels, one camera and
two. Tolerance: every one of the 18 convolutions on a path adds a relative
error of at most 4e-7 (fp32 sums of up to 4608 products): 8e-6.
"""

import os

import numpy as np
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def trunk64(raw, images, eps):
    at = 0

    def conv(x, cin, cout, k, stride):
        nonlocal at
        n = cout * k * k * cin
        W = raw[at:at + n].reshape(cout, k, k, cin).permute(0, 3, 1, 2)
        b = raw[at + n:at + n + cout]
        at += n + cout
        return F.conv2d(x, W, b, stride, k // 2)

    mean = torch.tensor([0.485, 0.456, 0.406], dtype=torch.float64)
    std = torch.tensor([0.229, 0.224, 0.225], dtype=torch.float64) + eps
    x = ((torch.from_numpy(images).double() / 255 - mean) / std).permute(0, 3, 1, 2)
    x = F.max_pool2d(torch.relu(conv(x, 3, 64, 7, 2)), 3, 2, 1)
    for stage in range(4):
        for b in range(2):
            cin, cout, s = x.shape[1], 64 << stage, 2 if stage and not b else 1
            y = conv(torch.relu(conv(x, cin, cout, 3, s)), cout, cout, 3, 1)
            x = torch.relu(y + (conv(x, cin, cout, 1, s) if s == 2 else x))
    return x.permute(0, 2, 3, 1).reshape(-1, x.shape[1]).numpy()


@pytest.mark.parametrize("H,W,cams", [(33, 45, 1), (64, 64, 2), (97, 130, 2), (240, 318, 1)])
def test_trunk_against_float64(vla, monkeypatch, tmp_path, H, W, cams):
    import vla_simd_amd.checkpoints as ck
    c = dict(ck.ACT_MODEL_BASE, img_h=H, img_w=W, n_cams=cams, n_enc=1, ff=256)
    d = ck.write_act_model(str(tmp_path / "act"), c)
    monkeypatch.setenv("ACT_INT8", "31")
    images = np.random.default_rng(H).integers(0, 256, (cams, H, W, 3), dtype=np.uint8)
    got = np.asarray(vla.ActModel(d).encode(images))
    raw = torch.from_numpy(np.fromfile(os.path.join(d, "backbone.bin"), np.float32)).double()
    want = trunk64(raw, images, c["norm_eps"]).reshape(got.shape)
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert err < 8e-6, err
