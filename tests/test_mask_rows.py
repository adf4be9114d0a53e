"""Boolean masks of any layout as the mask kernels walk them: row t at element t * ld, unit column stride (host side, no GPU)."""
import pytest
import torch

FORMS = {
    "plain": lambda T, C: torch.rand(T, C) < 0.5,
    "wide rows": lambda T, C: (torch.rand(T, C + 3) < 0.5)[:, :C],
    "more rows": lambda T, C: (torch.rand(T + 4, C) < 0.5),
    "transposed": lambda T, C: (torch.rand(C, T) < 0.5).T,
    "transposed part": lambda T, C: (torch.rand(C, T + 2) < 0.5)[:, 1:T + 1].T,
    "expanded rows": lambda T, C: (torch.rand(1, C) < 0.5).expand(T, C),
    "expanded columns": lambda T, C: (torch.rand(T, 1) < 0.5).expand(T, C),
    "every third column": lambda T, C: (torch.rand(T, 3 * C) < 0.5)[:, ::3],
    "floats": lambda T, C: (torch.rand(T, C) < 0.5).float().masked_fill(torch.rand(T, C) < 0.2, float("nan")),
}


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("T,C", [(1, 1), (1, 7), (1, 130), (2, 1), (5, 1), (3, 65)])
def test_rows_and_their_stride(form, T, C):
    from umbrella_amd.models.llama import mask_rows
    torch.manual_seed(T * 1000 + C)
    mask = FORMS[form](T, C)
    rows, ld = mask_rows(mask, T)
    want = torch.stack([torch.tensor([bool(mask[t, c]) for c in range(C)]) for t in range(T)])
    assert rows.dtype == torch.bool and rows.shape == (T, C) and ld >= C
    flat = torch.as_strided(rows, (rows.untyped_storage().nbytes() - rows.storage_offset(),), (1,), rows.storage_offset())
    got = torch.stack([flat[t * ld:t * ld + C] for t in range(T)])           # what a kernel reads from the data pointer
    assert torch.equal(got, want)
