"""What a call of bfly.ops reads from its tensors besides their memory: the
current stream of their device, and whether the memory holds the values."""
import pytest
import torch

from bfly import ops


def test_host_tensors_have_no_stream():
    with pytest.raises(ValueError):
        ops._stream(torch.empty(4))


@pytest.mark.gpu
def test_stream_is_the_current_one():
    x = torch.empty(4, device="cuda")
    assert ops._stream(x) == torch.cuda.current_stream(x.device).cuda_stream
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert ops._stream(x) == side.cuda_stream


@pytest.mark.gpu
@pytest.mark.parametrize("call", [ops.c2c, ops.fft2])
def test_lazy_conjugates_are_refused(call):
    x = torch.zeros(2, 64, 64, dtype=torch.complex64, device="cuda")
    with pytest.raises(RuntimeError):
        call(x.conj())
    assert torch.equal(call(x), x)
