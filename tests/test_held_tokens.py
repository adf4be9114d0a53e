"""Streaming products of 33 to 64 tokens whose tokens stay in registers: against a product in 64 bits, and bit by bit against the streaming kernel."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# second blocks of rows for one workgroup, for most and for all; a last block of one row and of all but one; both ends of the token tiles; both K
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,K", [(33, 2048), (48, 2048), (49, 2048), (64, 2048), (33, 4096), (48, 4096), (49, 4096), (64, 4096)])
@pytest.mark.parametrize("rows,epi", [(4097, 2), (8191, 2), (8200, 0), (16385, 1), (24608, 0), (12300, 2)])
def test_products(dtype, T, K, rows, epi):
    from umbrella_amd import _lib
    code, gated = _lib.seq_dtype_code(dtype), epi == 2
    g = torch.Generator(device="cuda").manual_seed(rows + K + T)
    N = 2 * rows if gated else rows
    x, w = torch.randn(T, K, generator=g, device="cuda").to(dtype), (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).to(dtype)
    bias = torch.randn(N, generator=g, device="cuda").to(dtype)
    out = torch.full((T + 1, rows), 7.0, dtype=torch.float32 if epi == 0 else dtype, device="cuda")
    _lib.seq_call("umb_seq_linear", out, x, w, bias, T, N, K, epi, code)
    want, size = x.double() @ w.double().T + bias.double(), x.double().abs() @ w.double().abs().T + bias.double().abs()
    bound = 2.0 ** -24 * (K / 8 + 16) * size                       # four waves' chains of K / 4 products, 32 of them a step
    half = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    if gated:
        gate, up = want[:, :rows], want[:, rows:]
        want = torch.nn.functional.silu(gate) * up
        bound = 1.1 * bound[:, :rows] * up.abs() + bound[:, rows:] * gate.abs() + half * want.abs() + 1e-7
    elif epi == 1:
        bound = bound + half * want.abs() + 1e-7
    assert bool((out[T] == 7.0).all()) and bool(((out[:T].double() - want).abs() <= bound).all())
    few = torch.empty((32, rows), dtype=out.dtype, device="cuda")  # a token's sums do not depend on how many stand beside it
    _lib.seq_call("umb_seq_linear", few, x, w, bias, 32, N, K, epi, code)
    assert torch.equal(out[:32], few)


def test_capped_logits():
    from umbrella_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(0)
    T, N, K = 40, 9001, 2048
    x, w = torch.randn(T, K, generator=g, device="cuda").bfloat16(), (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).bfloat16()
    out = torch.full((T + 1, N), 7.0, device="cuda")
    _lib.seq_call("umb_seq_linear_cap", out, x, w, None, T, N, K, 30.0, _lib.seq_dtype_code(torch.bfloat16))
    want = 30.0 * torch.tanh(x.double() @ w.double().T / 30.0)
    assert bool((out[T] == 7.0).all()) and float((out[:T].double() - want).abs().max()) <= 2.0 ** -24 * (K / 8 + 64) * float((x.double().abs() @ w.double().abs().T).max())


# chunks of 256 from the fewest on (5), either side of eight and of the ten that stay beyond 48 tokens; the squared activation
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T", [33, 48, 49, 64])
@pytest.mark.parametrize("K", [1280, 1792, 2304, 2560, 2816, 3072, 3840])
@pytest.mark.parametrize("rows,epi", [(4097, 2), (8200, 0), (16385, 4), (5121, 2), (10241, 0)])
def test_products_of_any_chunks(dtype, T, K, rows, epi):
    if epi != 4:
        return test_products(dtype, T, K, rows, epi)
    from umbrella_amd import _lib
    code = _lib.seq_dtype_code(dtype)
    g = torch.Generator(device="cuda").manual_seed(rows + K + T)
    x, w = torch.randn(T, K, generator=g, device="cuda").to(dtype), (torch.randn(rows, K, generator=g, device="cuda") * K ** -0.5).to(dtype)
    out, few = torch.full((T + 1, rows), 7.0, dtype=dtype, device="cuda"), torch.empty((32, rows), dtype=dtype, device="cuda")
    _lib.seq_call("umb_seq_linear", out, x, w, None, T, rows, K, 4, code)
    want, size = (x.double() @ w.double().T).relu(), x.double().abs() @ w.double().abs().T
    bound = 2.0 ** -24 * (K / 8 + 16) * size                       # of a sum, as above; of its square twice the sum's times it
    bound = 2.1 * bound * want + bound * bound + {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype] * want * want + 1e-7
    assert bool((out[T] == 7.0).all()) and bool(((out[:T].double() - want * want).abs() <= bound).all())
    _lib.seq_call("umb_seq_linear", few, x, w, None, 32, rows, K, 4, code)
    assert torch.equal(out[:32], few)


@pytest.mark.parametrize("T,K,epi", [(48, 2048, 0), (64, 4096, 2), (49, 2816, 4)])
def test_infinities_and_nan_stay_in_their_rows(T, K, epi):
    from umbrella_amd import _lib
    code, rows, bad, odd = _lib.seq_dtype_code(torch.bfloat16), 12300, (5, 20, 31, T - 1), (0, 4100, 12299)
    g = torch.Generator(device="cuda").manual_seed(K + T)
    N = 2 * rows if epi == 2 else rows
    x, w = torch.randn(T, K, generator=g, device="cuda").bfloat16(), (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).bfloat16()
    out, few, clean = (torch.empty((t, rows), dtype=torch.bfloat16 if epi else torch.float32, device="cuda") for t in (T, 32, T))
    _lib.seq_call("umb_seq_linear", clean, x, w, None, T, N, K, epi, code)
    for t, v in zip(bad, (float("inf"), float("nan"), float("-inf"), float("nan"))):
        x[t, (t * 37) % K] = v
    for n, v in zip(odd, (float("nan"), float("inf"), float("nan"))):
        w[n, K - 1 - n % 7] = v
    _lib.seq_call("umb_seq_linear", out, x, w, None, T, N, K, epi, code)
    _lib.seq_call("umb_seq_linear", few, x, w, None, 32, N, K, epi, code)
    same = torch.isnan(out[:32]) == torch.isnan(few)
    assert bool(same.all()) and torch.equal(out[:32][~torch.isnan(few)], few[~torch.isnan(few)])
    rest = torch.ones(T, rows, dtype=torch.bool, device="cuda")
    rest[list(bad)] = False
    rest[:, list(odd)] = False
    assert torch.equal(out[rest], clean[rest]) and bool(torch.isfinite(clean).all())
    assert epi == 4 or not bool(torch.isfinite(out[:, 0]).any())         # (relu squared: fmaxf gives 0 for NaN, in every kernel)
