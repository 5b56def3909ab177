"""The stream an operation runs on is torch's current one, on every way of
making a stream current, and the given one where one is given."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("how", ["default", "side", "external", "capture"])
def test_current_stream_handle(how):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from xinfer_amd import ops
    torch.cuda.init()
    want = lambda: torch.cuda.current_stream().cuda_stream  # noqa: E731
    if how == "default":
        assert ops._stream() == want()
    elif how == "capture":
        g = torch.cuda.CUDAGraph()
        x = torch.zeros(4, device="cuda")
        with torch.cuda.graph(g):
            assert ops._stream() == want()
            x.add_(1)
    else:
        side = torch.cuda.Stream()
        if how == "external":
            side = torch.cuda.ExternalStream(side.cuda_stream)
        with torch.cuda.stream(side):
            assert ops._stream() == want() == side.cuda_stream
        assert ops._stream(side) == side.cuda_stream
        assert ops._stream(side.cuda_stream) == side.cuda_stream
