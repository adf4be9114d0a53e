"""Gated linear attention of single tokens in one launch (umb_gla_step) against decays, recurrence and gate as launches of their own."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("T,H,D,Dv,rank,pad", [(1, 8, 128, 256, 16, 0), (16, 16, 128, 256, 16, 0), (3, 3, 40, 56, 10, 0), (5, 2, 17, 4, 1, 3), (2, 4, 256, 128, 33, 1),
                                               (7, 1, 64, 64, 8, 0), (4, 5, 100, 132, 7, 2)])
def test_step_as_three_launches(dtype, T, H, D, Dv, rank, pad):
    from umbrella_amd import _lib
    code, HD, ld = _lib.seq_dtype_code(dtype), H * D, 2 * H * D + 2 * H * Dv + rank + pad
    g = torch.Generator(device="cuda").manual_seed(T + H + D + Dv)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")                                              # noqa: E731
    proj, w2, b2, wn = rnd(T, ld), (0.5 * rnd(HD, rank)).to(dtype), rnd(HD).to(dtype), (1.0 + 0.1 * rnd(Dv)).to(dtype)
    slots = torch.randperm(T + 2, generator=torch.Generator().manual_seed(1))[:T].to(torch.int32).cuda()
    pos = torch.arange(T, dtype=torch.int32, device="cuda")                                                   # the first one starts afresh
    start = rnd(T + 2, H, D, Dv)
    a, b = start.clone(), start.clone()
    one, row = torch.ones(T, dtype=torch.int32, device="cuda"), torch.arange(T, dtype=torch.int32, device="cuda")
    alpha, o = torch.empty(T, HD, device="cuda"), torch.empty(T, H * Dv, device="cuda")
    want, got = torch.empty(T, H * Dv, dtype=dtype, device="cuda"), torch.full((T + 1, H * Dv), 3.0, dtype=dtype, device="cuda")
    _lib.seq_call("umb_gla_decay", alpha, proj, ld, 2 * HD + 2 * H * Dv, w2, b2, T, HD, rank, 16.0, code)
    _lib.seq_call("umb_gla_scan", o, a, proj, ld, alpha, slots, row, pos, one, T, H, D, Dv, D ** -0.5)
    _lib.seq_call("umb_gla_gate", want, o, proj, ld, 2 * HD + H * Dv, wn, T, H, Dv, 1e-6, code)
    _lib.seq_call("umb_gla_step", got, b, proj, ld, w2, b2, wn, pos, slots, T, H, D, Dv, rank, 16.0, D ** -0.5, 1e-6, code)
    assert bool((got[T] == 3.0).all())
    # the decay's exponent and the update by other contractions: a few fp32 steps of the state; the read-out's sum of D of them in its own order
    assert bool(((a - b).abs() <= 2.0 ** -21 * (a.abs() + start.abs() + 4.0)).all())
    step = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10, torch.float32: 2.0 ** -18}[dtype]
    assert bool(((want.float() - got[:T].float()).abs() <= step * want.float().abs() + 2.0 ** -19 * float(want.float().abs().max()) + 1e-6).all())
