"""A capture outside inference mode while a graph that was captured inside it is alive."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_captures_inside_and_outside_inference_mode():
    import gc
    from umbrella_amd import _lib
    gc.collect()                                               # graphs of earlier tests: the first capture below is the process's only one
    x, graphs = torch.zeros(64, device="cuda"), []
    for mode in (True, False, True):
        with torch.inference_mode(mode):
            graphs.append(torch.cuda.CUDAGraph())
            with _lib.capturing(graphs[-1]):
                assert torch.is_inference_mode_enabled() == mode
                x.add_(1.0)
    for _ in range(3):
        for g in graphs:
            g.replay()
    assert bool((x == 9.0).all())


@pytest.mark.parametrize("first", ["own graph inside the mode", "own graph outside", "this library's"])
def test_captures_beside_a_callers_own_graph(first):
    """the generator's tensors belong to whichever graph came first: in either mode every capture may write them"""
    import gc
    from umbrella_amd import _lib
    gc.collect()
    x, graphs = torch.zeros(64, device="cuda"), []

    def capture(mode, own):
        with torch.inference_mode(mode):
            graphs.append(torch.cuda.CUDAGraph())
            with torch.cuda.graph(graphs[-1]) if own else _lib.capturing(graphs[-1]):
                assert torch.is_inference_mode_enabled() == mode
                x.add_(1.0)
    if first != "this library's":
        capture(first.endswith("inside the mode"), True)
    capture(True, False)
    capture(False, False)
    capture(True, True)
    if first != "own graph inside the mode":                   # (a plain capture outside the mode never took that one's tensors)
        capture(False, True)
    for _ in range(3):
        for g in graphs:
            g.replay()
    assert bool((x == 3.0 * len(graphs)).all())
    del graphs[:]
