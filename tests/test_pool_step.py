"""Pooled blocks that single tokens complete, in the launch that prepares the tokens: against the two launches."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("B,H,G,D,rot,pool,page", [(1, 6, 2, 24, 16, 7, 16), (5, 8, 2, 64, 64, 16, 64), (3, 4, 4, 128, 0, 1, 48), (4, 3, 1, 25, 10, 5, 64),
                                                   (2, 2, 1, 256, 200, 70, 32), (17, 16, 8, 64, 32, 16, 16), (460, 32, 8, 64, 64, 3, 16)])
def test_completed_blocks(dtype, B, H, G, D, rot, pool, page):
    from umbrella_amd import _lib
    from umbrella_amd.attn.cache import PagedSeqCache
    g = torch.Generator(device="cuda").manual_seed(B + D)
    code, ld = _lib.seq_dtype_code(dtype), (H + G) * D + H
    lens = [1 + (pool * (i % 5) + pool - 1 - i % 3) % (4 * pool + 40) for i in range(B)]           # most complete a block, some do not
    stores = []
    for _ in range(2):
        c = PagedSeqCache([(G, D, pool)], [], sum(lens), B, "cuda", dtype, page=page)
        for b, n in enumerate(lens):
            c.open(b), c.extend(b, n)
        stores.append(c)
    for name in ("k", "v"):
        stores[0].kv[0][name].copy_(torch.randn(stores[0].kv[0][name].shape, generator=g, device="cuda"))
        stores[1].kv[0][name].copy_(stores[0].kv[0][name])
    proj, freq = torch.randn(B, ld, generator=g, device="cuda"), torch.rand(max(rot // 2, 1), generator=g, device="cuda")
    pos = torch.tensor([n - 1 for n in lens], dtype=torch.int32, device="cuda")
    slot, one = torch.arange(B, dtype=torch.int32, device="cuda"), torch.ones(B, dtype=torch.int32, device="cuda")
    slot = torch.tensor([stores[0].slot(b) for b in range(B)], dtype=torch.int32, device="cuda")
    q = [torch.zeros(B, H * D, device="cuda") for _ in range(2)]
    _lib.seq_call("umb_pwa_prep", q[0], stores[0].struct(0), proj, ld, pos, slot, freq, B, H, G, D, rot, 1e-6, code)
    _lib.seq_call("umb_pwa_pool", stores[0].struct(0), slot, pos, one, B, 1, G, D, pool, code)
    _lib.seq_call("umb_pwa_prep_step", q[1], stores[1].struct(0), proj, ld, pos, slot, freq, slot, pos, one, B, H, G, D, rot, pool, 1e-6, code)
    a, b = stores[0].kv[0], stores[1].kv[0]
    assert torch.equal(q[0], q[1]) and torch.equal(a["k"], b["k"]) and torch.equal(a["v"], b["v"])
    assert float(a["kp"].abs().sum()) > 0.0 and torch.equal(a["vp"], b["vp"])
    # the token's own key may be rounded the other way (another contraction of the rotation): one step of one of `pool` keys, sizes below 16; and so may the
    # last of the fp32 sums behind it (sizes below 16: a step of 2^-20, half of it on either side), and the mean (2^-24 of itself on either side)
    ulp = {torch.bfloat16: 2.0 ** -4, torch.float16: 2.0 ** -7, torch.float32: 2.0 ** -20}[dtype]
    assert float((a["kp"] - b["kp"]).abs().max()) <= (ulp + 2.0 ** -20) / pool + 2.0 ** -23 * float(a["kp"].abs().max())
