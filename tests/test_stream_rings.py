"""Streaming products at the lines between their rings and grids (launch_stream), against a product in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# blocks of 16 rows around 256, 400, 512, 1024 and beyond, K of two chunks of 512 bytes to some dozens, every token tile
@pytest.mark.parametrize("dtype,K", [(torch.bfloat16, 512), (torch.float16, 768), (torch.bfloat16, 2304), (torch.float32, 384), (torch.float32, 1280)])
@pytest.mark.parametrize("rows", [4096, 4112, 6400, 6401, 8192, 8200, 16384, 16400, 18432, 24577])
@pytest.mark.parametrize("T,gated", [(1, False), (8, True), (9, False), (16, True), (17, True), (32, False)])
def test_rings(dtype, K, rows, T, gated):
    from umbrella_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(rows + K + T)
    N = 2 * rows if gated else rows
    x, w = torch.randn(T, K, generator=g, device="cuda").to(dtype), (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).to(dtype)
    bias = torch.randn(N, generator=g, device="cuda").to(dtype)
    out = torch.full((T + 1, rows), 7.0, dtype=dtype if gated else torch.float32, device="cuda")
    _lib.seq_call("umb_seq_linear", out, x, w, bias, T, N, K, 2 if gated else 0, _lib.seq_dtype_code(dtype))
    want = x.double() @ w.double().T + bias.double()
    size = x.double().abs() @ w.double().abs().T + bias.double().abs()                     # what a sum's rounding goes with
    bound = 2.0 ** -24 * (K / 8 + 16) * size
    if gated:
        gate, up = want[:, :rows], want[:, rows:]
        want = torch.nn.functional.silu(gate) * up
        bound = 1.1 * bound[:, :rows] * up.abs() + bound[:, rows:] * gate.abs() + {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -21}[dtype] * want.abs() + 1e-7
    assert bool((out[T] == 7.0).all())
    assert bool(((out[:T].double() - want).abs() <= bound).all())


# fp32 gate and up of more than 12 chunks, a workgroup a block; single matrices a few blocks beyond two rounds of 32 rows, and of none
@pytest.mark.parametrize("T,K,rows,gated", [(1, 1664, 7184, True), (8, 1792, 12321, True), (4, 2048, 8200, True), (17, 1536, 20480, False), (32, 256, 18000, False), (32, 384, 20496, False)])
def test_rings_of_fp32(T, K, rows, gated):
    test_rings(torch.float32, K, rows, T, gated)


@pytest.mark.parametrize("rows,gated", [(6500, True), (8300, True), (16500, False), (12304, False)])
@pytest.mark.parametrize("T", [1, 9, 24, 40])
def test_a_single_tile_of_a_group(rows, gated, T):
    """a tile list of one tile: its blocks run on inside a unit's workgroups as a dense launch's do"""
    from umbrella_amd import _lib
    K, groups, dtype = 1280, 3, torch.bfloat16
    code, N = _lib.seq_dtype_code(dtype), 2 * rows if gated else rows
    g = torch.Generator(device="cuda").manual_seed(rows + T)
    x, w = torch.randn(T + 5, K, generator=g, device="cuda").to(dtype), (torch.randn(groups, N, K, generator=g, device="cuda") * K ** -0.5).to(dtype)
    made = dtype if gated else torch.float32
    out = torch.full((T + 6, rows), 7.0, dtype=made, device="cuda")
    tiles = torch.tensor([[2, 3, T]], dtype=torch.int32, device="cuda")
    _lib.seq_call("umb_seq_linear_grouped", out, x, w, tiles, 1, 64, N * K, N, K, 2 if gated else 0, code)
    xs = x[3:3 + T].contiguous()
    full, size = xs.double() @ w[2].double().T, xs.double().abs() @ w[2].double().abs().T
    bound = 2.0 ** -24 * (K / 8 + 16) * size
    if gated:
        gate, up = full[:, :rows], full[:, rows:]
        full = torch.nn.functional.silu(gate) * up
        bound = 1.1 * bound[:, :rows] * up.abs() + bound[:, rows:] * gate.abs() + 2.0 ** -8 * full.abs() + 1e-7
    assert bool((out[:3] == 7.0).all()) and bool((out[3 + T:] == 7.0).all()) and bool(((out[3:3 + T].double() - full).abs() <= bound).all())
