"""What stands between a prompt's projection and its mixer, walked in quads: against the kernels of single channels, which take the same numbers from
columns that are not 16-byte aligned."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _steps(lens, first, dev="cuda"):
    """positions and slots of stretches of `lens` tokens that start at `first`, in slots of their own in mixed order"""
    slots = [(3 * i + 1) % len(lens) if len(lens) % 3 else i for i in range(len(lens))]
    pos = [p for n, f in zip(lens, first) for p in range(f, f + n)]
    slot = [s for n, s in zip(lens, slots) for _ in range(n)]
    return torch.tensor(pos, dtype=torch.int32, device=dev), torch.tensor(slot, dtype=torch.int32, device=dev)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("taps", [3, 4])
@pytest.mark.parametrize("Hk,H,D,E", [(2, 4, 24, 40), (1, 1, 128, 128), (3, 3, 100, 300), (2, 2, 132, 8), (1, 2, 256, 64), (8, 16, 128, 128)])
def test_delta_fronts(dtype, taps, Hk, H, D, E):
    from umbrella_amd import _lib
    lens, first = [1, 9, 2, 17, 8, 3, 1], [0, 5, 1, 0, 2, 40, 3]
    T, C, Dp = sum(lens), 2 * Hk * D + H * E, (D + 15) // 16 * 16
    pos, slot = _steps(lens, first)
    g = torch.Generator(device="cuda").manual_seed(D + E + taps)
    cols = C + H * E + 2 * H
    rows = torch.randn(T, cols, generator=g, device="cuda")
    ring = torch.randn(len(lens), taps, C, generator=g, device="cuda")
    conv = torch.randn(C, taps, generator=g, device="cuda").to(dtype)
    dtb, alog = (torch.randn(H, generator=g, device="cuda") for _ in range(2))
    outs = []
    for col0 in (4, 3):
        ld = (cols + col0 + 3) // 4 * 4 + (0 if col0 == 4 else 1)
        proj = torch.full((T, ld), 9.0, device="cuda")
        proj[:, col0:col0 + cols] = rows
        q, k, v = (torch.full(s, 8.0, device="cuda") for s in ((T, Hk * Dp), (T, Hk * Dp), (T, H * E)))
        beta, lg = (torch.empty(T, H, device="cuda") for _ in range(2))
        _lib.seq_call("umb_delta_prep", q, k, Hk * Dp, v, beta, lg, proj, ld, col0, conv, ring, dtb, alog, pos, slot, T, Hk, H, D, E, taps,
                      _lib.seq_dtype_code(dtype))
        outs.append((q, k, v, beta, lg))
    assert torch.equal(outs[0][3], outs[1][3]) and torch.equal(outs[0][4], outs[1][4])
    assert (outs[0][2] - outs[1][2]).abs().max() <= 2e-6 * outs[1][2].abs().max()          # sums of 3 or 4 products
    for a, b in zip(outs[0][:2], outs[1][:2]):                 # unit rows: sums of D squares in another order
        assert (a - b).abs().max() <= 4e-7 * D ** 0.5
