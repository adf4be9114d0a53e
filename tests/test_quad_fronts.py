"""Rows of 64 and 128 features that many (token, head) slots are prepared in by quads: against launches of few slots."""
import pytest
import test_prompt_kernels as prompt
import torch

pytestmark = pytest.mark.gpu


# both layouts of pairs; nothing, a part and all of a row turned; one and two maps; rows that end inside a wave's sixteen; queries alone; values of another size
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("H,G,D,E,maps,layout,rot,append,norm,mixed", [(8, 2, 64, 64, 1, 0, 64, 1, 1, True), (9, 3, 128, 64, 2, 1, 80, 1, 0, False),
                                                                       (17, 17, 64, 128, 1, 1, 36, 1, 1, True), (30, 2, 128, 128, 1, 0, 48, 0, 1, False),
                                                                       (15, 1, 128, 128, 1, 0, 128, 1, 0, True), (12, 4, 64, 64, 1, 1, 0, 1, 1, False)])
def test_attention_slots(dtype, H, G, D, E, maps, layout, rot, append, norm, mixed):
    prompt.test_many_slots_are_prepared_as_few_are(dtype, H, G, D, E, maps, layout, rot, append, norm, mixed)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("H,G,D,rot", [(15, 1, 64, 32), (16, 8, 128, 128), (20, 4, 64, 0), (17, 1, 128, 60)])
def test_pooled_slots(dtype, H, G, D, rot):
    prompt.test_many_pooled_slots_are_prepared_as_few_are(dtype, H, G, D, rot)
