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
