"""The fp32 trunk's residual add + ReLU in the convolution's epilogue (unsplit
tiles and the split-K sum) against the pass of its own, bit for bit; with an
int8 stage after fp32 ones, which reads the maxima that only the pass writes.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W", [(480, 640), (224, 224), (136, 248)])
@pytest.mark.parametrize("bits,stages", [("31", None), ("63", ("2", "4"))])
def test_fused_add_is_the_pass(vla, monkeypatch, tmp_path, H, W, bits, stages):
    import vla_simd_amd.checkpoints as ck
    c = dict(ck.ACT_MODEL_BASE, img_h=H, img_w=W, n_enc=1, ff=256)
    d = ck.write_act_model(str(tmp_path / "act"), c)
    monkeypatch.setenv("ACT_INT8", bits)
    if stages:
        monkeypatch.setenv("ACT_I8_CONV_FROM", stages[0])
        monkeypatch.setenv("ACT_I8_CONV_TO", stages[1])
    images, _ = ck.act_model_inputs(c)
    m = vla.ActModel(d)
    got = m.encode(images)
    monkeypatch.setenv("VLA_HIP_CONV_FUSE", "0")
    want = vla.ActModel(d).encode(images)
    assert np.isfinite(want).all() and np.abs(want).max() > 0
    np.testing.assert_array_equal(got, want)
