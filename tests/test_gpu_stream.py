"""The binding's default stream is torch's current one: on the default stream, inside a stream
context, and while a graph is captured."""
import pytest

pytestmark = pytest.mark.gpu


def test_default_stream_is_the_current_one(dev):
    import torch
    from cuda_gpt2_inference_amd import kvattn

    def same():
        return kvattn._stream(None) == torch.cuda.current_stream().cuda_stream

    assert same()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert kvattn._stream(None) == side.cuda_stream and same()
    assert same()
    seen = []
    x = torch.zeros(8, device=dev)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        seen.append(same())
        x.add_(1)
    assert seen == [True]
    assert kvattn._stream(side) == side.cuda_stream and kvattn._stream(5) == 5
