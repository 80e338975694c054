"""The Python face launches on torch's current stream of the current device."""

import pytest

pytestmark = pytest.mark.gpu


def test_current_stream_is_torchs(vla, torch_cuda):
    torch = torch_cuda
    assert vla._stream(None) == torch.cuda.current_stream().cuda_stream
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        assert vla._stream(None) == s.cuda_stream
        x = torch.ones(1 << 20, device="cuda")
        vla._call("vla_add_dev", vla._dp(x), vla._dp(x), vla._dp(x), x.numel(), vla._stream(None))
    s.synchronize()
    assert float(x.sum()) == 2.0 * x.numel()
    assert vla._stream(None) == torch.cuda.current_stream().cuda_stream
    assert vla._stream(s.cuda_stream) == s.cuda_stream
