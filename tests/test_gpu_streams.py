"""The Python calls run on torch's current stream of the current device, or on the stream given."""
import numpy as np
import pytest
import torch

import cretif_amd as cri
from cretif_amd import quant

pytestmark = pytest.mark.gpu


def test_current_stream_address():
    assert cri._stream(None) == torch.cuda.current_stream().cuda_stream
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        assert cri._stream(None) == s.cuda_stream
        with torch.cuda.stream(torch.cuda.default_stream()):
            assert cri._stream(None) == torch.cuda.default_stream().cuda_stream
        assert cri._stream(None) == s.cuda_stream
    assert cri._stream(None) == torch.cuda.current_stream().cuda_stream
    assert cri._stream(s) == s.cuda_stream and cri._stream(7) == 7


def test_ordered_with_torch_on_a_side_stream():
    """A product between two torch operations on one side stream sees the first and is seen by the second."""
    M, N, K = 1, 4096, 2048
    B = torch.from_numpy(quant.synthetic_weights("q8_0", N, K, seed=3)).cuda()
    A = torch.from_numpy(quant.randn(K, seed=4).reshape(1, K)).cuda()
    ref = torch.empty(M, N, device="cuda")
    cri.matmul("q8_0", A, B, ref, M, N, K)
    x, C = torch.zeros_like(A), torch.zeros_like(ref)
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        big = torch.ones(1 << 26, device="cuda").cumsum(0)  # keeps the stream busy first
        x.copy_(A + 0 * big[:1])
        cri.matmul("q8_0", x, B, C, M, N, K)
        y = C * 2
    s.synchronize()
    assert np.array_equal(y.cpu().numpy(), (ref * 2).cpu().numpy())


def test_pointer_checks():
    C = torch.empty(1, 32, device="cuda")
    assert cri._ptr(None) is None and cri._ptr(16) == 16 and cri._ptr(C) == C.data_ptr()
    with pytest.raises(ValueError, match="device"):
        cri._ptr(torch.empty(4))
    with pytest.raises(ValueError, match="contiguous"):
        cri._ptr(torch.empty(4, 4, device="cuda").t())
    with pytest.raises(TypeError):
        cri._ptr("address")
    with pytest.raises(TypeError):
        cri._ptr(np.zeros(4, np.float32).tolist())
