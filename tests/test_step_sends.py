"""What a step of the sequence mixers sends to the device: from pinned memory, without waiting, in the order of the stream."""
import pytest
import torch

from umbrella_amd.attn.cache import send


def test_send_on_the_host():
    a = torch.arange(7)
    assert torch.equal(send(a, "cpu"), a)
    into = torch.zeros(7, dtype=torch.int64)
    assert send(a, "cpu", into=into) is into and torch.equal(into, a)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 3, 5000])
def test_send_in_order_behind_a_busy_stream(n):
    big = torch.ones(64 << 20, device="cuda")
    into = torch.zeros(n, dtype=torch.int32, device="cuda")
    got = []
    for i in range(40):                                   # more than the device has done by then: every copy needs a block of its own
        big.mul_(1.0)
        host = torch.arange(n, dtype=torch.int32) + i
        got.append((send(host, "cuda:0"), send(host, "cuda:0", into=into).clone()))
        host.fill_(-1)
    for i, pair in enumerate(got):
        for t in pair:
            assert torch.equal(t.cpu(), torch.arange(n, dtype=torch.int32) + i)


@pytest.mark.gpu
def test_send_is_refused_under_capture():
    a = torch.zeros(4, device="cuda")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, capture_error_mode="thread_local"):
        a += 1.0
        with pytest.raises(RuntimeError, match="capturing"):
            send(torch.arange(3), "cuda:0")
    graph.replay()
    assert a.tolist() == [1.0] * 4
