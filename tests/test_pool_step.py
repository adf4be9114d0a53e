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


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("H,G,D,rot,window,pool,lens", [(32, 8, 64, 64, 512, 16, [2000]), (32, 8, 128, 128, 64, 16, [96 + i for i in range(16)]),
                                                        (6, 2, 64, 32, 40, 7, [1, 7, 14, 41, 48, 49, 300]), (4, 4, 256, 0, 16, 16, [16, 17, 32, 33, 1024]),
                                                        (8, 1, 128, 64, 2 ** 30, 3, [3, 50, 600]), (16, 2, 64, 64, 33, 16, [30 + i for i in range(120)]),
                                                        (6, 2, 24, 16, 40, 7, [42, 49, 5])])
def test_step_as_three_launches(dtype, H, G, D, rot, window, pool, lens):
    """the whole of a step in one launch; the cache holds NaN at the tokens' own positions until they are appended"""
    from umbrella_amd import _lib
    from umbrella_amd.attn.cache import PagedSeqCache
    code, T, ld = _lib.seq_dtype_code(dtype), len(lens), (H + G) * D + H
    g = torch.Generator(device="cuda").manual_seed(H + D + T)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")                                              # noqa: E731
    proj, freq, bias = rnd(T, ld), torch.rand(max(rot // 2, 1), generator=g, device="cuda"), rnd(H).to(dtype)
    pos, one = torch.tensor([n - 1 for n in lens], dtype=torch.int32, device="cuda"), torch.ones(T, dtype=torch.int32, device="cuda")
    fill, outs = None, []
    for step in (False, True):
        c = PagedSeqCache([(G, D, pool)], [], sum(lens) + 50, T, "cuda", dtype, page=32)
        for b, n in enumerate(lens):
            c.open(b), c.extend(b, n)
        kv = c.kv[0]
        fill = fill or {z: rnd(*kv[z].shape).to(kv[z].dtype) for z in ("k", "v", "kp", "vp")}
        for z in fill:
            kv[z].copy_(fill[z])
        for b, n in enumerate(lens):
            page = c.seqs[b]["pages"][(n - 1) // 32]
            kv["k"][page, :, (n - 1) % 32], kv["v"][page, :, (n - 1) % 32] = float("nan"), float("nan")
        slot = torch.tensor([c.slot(b) for b in range(T)], dtype=torch.int32, device="cuda")
        q, out = torch.zeros(T, H * D, device="cuda"), torch.full((T + 1, H * D), 3.0, dtype=dtype, device="cuda")
        if step:
            _lib.seq_call("umb_pwa_step", out, q, c.struct(0), proj, ld, (H + G) * D, bias, pos, slot, freq, slot, pos, one, T, H, G, D, rot, window, pool,
                          D ** -0.5, 1e-6, code)
        else:
            _lib.seq_call("umb_pwa_prep", q, c.struct(0), proj, ld, pos, slot, freq, T, H, G, D, rot, 1e-6, code)
            _lib.seq_call("umb_pwa_pool", c.struct(0), slot, pos, one, T, 1, G, D, pool, code)
            _lib.seq_call("umb_pwa_attend", out, q, c.struct(0), proj, ld, (H + G) * D, bias, pos, slot, T, H, G, D, window, pool, D ** -0.5, code)
        assert bool((out[T] == 3.0).all()) and bool(torch.isfinite(out).all())
        outs.append((out[:T].float(), kv["k"].float(), kv["v"].float(), kv["kp"].clone(), kv["vp"].clone()))
    a, b = outs
    step_of = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10, torch.float32: 2.0 ** -22}[dtype]           # one step of the storage type, of keys below 16
    assert torch.equal(a[2], b[2]) and torch.equal(a[4], b[4])
    assert bool(((a[1] - b[1]).abs() <= step_of * a[1].abs()).all()) and bool(((a[3] - b[3]).abs() <= 16 * step_of / pool + 2.0 ** -19).all())
    # the rotation and the norm may be contracted otherwise, the sums are of up to 600 weights below 1 in the same order
    assert bool(((a[0] - b[0]).abs() <= 2 * step_of * a[0].abs() + 2.0 ** -18 * min(window, max(lens))).all())


def test_sequences_that_bring_nothing_stand_in_front(monkeypatch):
    """a caller of the library may list sequences of length 0: the blocks of those behind them are pooled too, also where pooling is a launch over the
    list (from 16384 head slots on)"""
    import types
    from umbrella_amd import _lib
    import seqmix_helpers
    B, pool = 2100, 3
    cfg = seqmix_helpers.config([seqmix_helpers.attn_layer(heads=6, kv_heads=2, dim=12, window=2, pool=pool, ff=16)], width=16, vocab=20, groups=1)
    m, _ = seqmix_helpers.build(cfg, torch.float32, batch=B + 1, max_length=16, max_tokens=16 * (B + 1))
    real, keep, got = _lib.load_seq(), [], []

    def forward(model, work, step, stream):
        s = step._obj
        if s.max_len == 1:
            for k, first in (("seq_slot", m.kv_cache.slot("empty")), ("seq_row0", 0), ("seq_pos0", 0), ("seq_len", 0)):
                own = (m._keep[3 * s.T + ("seq_slot", "seq_row0", "seq_pos0", "seq_len").index(k) * s.B:][:s.B])
                keep.append(torch.cat([torch.tensor([first], dtype=torch.int32, device="cuda"), own]))
                setattr(s, k, keep[-1].data_ptr())
            s.B += 1
        return real.umb_seq_forward(model, work, step, stream)
    for listed in (False, True):
        m.clear()
        for i in ["empty"] + list(range(B)):
            m.open(i)
        m.forward_batch([(i, [i % 7, i % 5]) for i in range(B)])
        if listed:
            monkeypatch.setattr(_lib, "load_seq", lambda: types.SimpleNamespace(umb_seq_forward=forward))
        m.kv_cache.kv[0]["kp"].fill_(9.0)
        m.forward_batch([(i, [i % 11]) for i in range(B)])
        got.append([m.kv_cache.pooled_rows(0, i, [0])[0] for i in (0, B // 2, B - 1)])
    assert len(keep) == 4
    for a, b in zip(*got):
        assert torch.equal(a, b) and bool((a != 9.0).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,G,D,rot", [(32, 8, 64, 64), (16, 4, 128, 128), (4, 4, 256, 0), (8, 2, 256, 200), (6, 2, 96, 40)])
def test_step_appends_what_a_launch_of_its_own_does(dtype, H, G, D, rot):
    """keys and values bit by bit: a token's cached rows do not depend on the launch that prepared them"""
    from umbrella_amd import _lib
    from umbrella_amd.attn.cache import PagedSeqCache
    code, T, ld, pool = _lib.seq_dtype_code(dtype), 150, (H + G) * D + H, 16
    g = torch.Generator(device="cuda").manual_seed(H + D)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")                                              # noqa: E731
    proj, freq, bias = rnd(T, ld), torch.rand(max(rot // 2, 1), generator=g, device="cuda"), rnd(H).to(dtype)
    lens = [1 + i % 70 for i in range(T)]
    pos, one, outs = torch.tensor([n - 1 for n in lens], dtype=torch.int32, device="cuda"), torch.ones(T, dtype=torch.int32, device="cuda"), []
    for step in (False, True):
        c = PagedSeqCache([(G, D, pool)], [], sum(lens) + 50, T, "cuda", dtype, page=32)
        for b, n in enumerate(lens):
            c.open(b), c.extend(b, n)
        for z in ("k", "v", "kp", "vp"):
            c.kv[0][z].zero_()
        slot = torch.tensor([c.slot(b) for b in range(T)], dtype=torch.int32, device="cuda")
        q, out = torch.zeros(T, H * D, device="cuda"), torch.zeros(T, H * D, dtype=dtype, device="cuda")
        if step:
            _lib.seq_call("umb_pwa_step", out, q, c.struct(0), proj, ld, (H + G) * D, bias, pos, slot, freq, slot, pos, one, T, H, G, D, rot, 64, pool, D ** -0.5,
                          1e-6, code)
        else:
            _lib.seq_call("umb_pwa_prep", q, c.struct(0), proj, ld, pos, slot, freq, T, H, G, D, rot, 1e-6, code)
        outs.append((c.kv[0]["k"], c.kv[0]["v"]))
    assert all(torch.equal(x, y) for x, y in zip(*outs))
