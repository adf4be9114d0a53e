"""Latent attention of few tokens: waves of 16 keys, and a token's keys over several workgroups where there is room for their partial results."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("sink", [True, False])
@pytest.mark.parametrize("H,Dc,R", [(32, 512, 64), (3, 512, 0), (6, 256, 32), (16, 256, 64), (8, 128, 32), (5, 64, 64), (2, 64, 0),
                                    (4, 128, 24), (4, 96, 32), (4, 512, 160)])                       # the last three: another kernel's
@pytest.mark.parametrize("window", [2 ** 30, 700, 33])
def test_latent_attention_of_few_tokens(dtype, H, Dc, R, window, sink):
    """against float64: fp32 queries, weights and sums, so the result's own rounding and little more"""
    from umbrella_amd import _lib
    from umbrella_amd.attn.cache import PagedSeqCache
    Dk, code = Dc + R, _lib.seq_dtype_code(dtype)
    g = torch.Generator(device="cuda").manual_seed(H + Dc + R)
    for lens in ([1], [16, 17, 255], [256, 257], [5, 1030, 513, 40], [2000]):
        B = len(lens)
        c = PagedSeqCache([], [], sum(lens) + 2000, B, "cuda", dtype, page=48, latent_layers=(Dk,))
        c.latent[0].copy_(torch.randn(c.latent[0].shape, generator=g, device="cuda"))
        for b, n in enumerate(lens):
            c.open(b), c.extend(b, n)
        slot = torch.tensor([c.slot(b) for b in range(B)], dtype=torch.int32, device="cuda")
        pos = torch.tensor([n - 1 for n in lens], dtype=torch.int32, device="cuda")
        qa, s = 2.0 * torch.randn(B, H, Dk, generator=g, device="cuda"), torch.randn(H, generator=g, device="cuda").to(dtype)
        whole = B * H * 16 * (Dc + 2)
        for floats in (0, whole // 8, whole):
            part = torch.full((floats + 64,), 9.0, device="cuda")
            out = torch.full((B + 1, H * Dc), 3.0, dtype=dtype, device="cuda")
            _lib.seq_call("umb_lat_attend_split", out, qa, c.latent_struct(0), s if sink else None, pos, slot, B, H, Dc, R, window, Dk ** -0.5,
                          part if floats else None, floats, code)
            assert bool((out[B] == 3.0).all()) and bool((part[floats:] == 9.0).all())
            for b, n in enumerate(lens):
                rows = c.latent_rows(0, b, torch.arange(max(0, n - window), n)).double()
                x = (qa[b].double() @ rows.T) * Dk ** -0.5
                p = torch.softmax(torch.cat([x, (s.double() if sink else torch.full((H,), -torch.inf, device="cuda", dtype=torch.float64))[:, None]], 1), 1)[:, :-1]
                o, size = p @ rows[:, :Dc], p @ rows[:, :Dc].abs()
                u = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
                # scores of some 10 from Dk products in fp32 (2^-24 Dk of their size), then the exponent's and the sums' roundings
                tol = 1.01 * u * o.abs() + 2.0 ** -24 * (Dk * 8 + n + 64) * size + 1e-7
                assert bool(((out[b].double().view(H, Dc) - o).abs() <= tol).all()), (lens, b, floats)
