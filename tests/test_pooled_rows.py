"""Prompt attention over pooled windows where token rows come by LDS-DMA (heads of 64, 128, 256), with more heads a group than a workgroup has waves: the
staging starts again for the heads that are left.  Against the 64-bit oracle of the other shapes."""
import pytest
import torch

import test_prompt_kernels as prompts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,G,D,window,pool", [(6, 1, 64, 2 ** 20, 16), (9, 1, 128, 33, 4), (5, 1, 256, 32, 16), (10, 2, 64, 1, 1), (3, 1, 128, 64, 5)])
def test_rows_that_fill_their_tile(dtype, H, G, D, window, pool):
    prompts.test_prompt_pooled_attention(dtype, H, G, D, window, pool)
