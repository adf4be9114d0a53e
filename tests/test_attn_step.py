"""Single tokens prepared inside their attention (umb_attn_step) against the two launches: the same cache, the same output, nothing read from the cache at the
token's own position, which holds NaN until it is appended."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SHORT, LONG = [1, 15, 16, 17, 40, 256, 257], [1024, 1025, 2049, 3]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("H,G,D,E,maps,lens,window,chunk,keep,append,norm,rot,layout,mixed,temp", [
    (32, 8, 64, 64, 1, SHORT, 2 ** 30, 0, 0, 1, 0, 64, 1, True, 0), (16, 4, 128, 256, 2, [77], 2 ** 30, 64, 0, 1, 0, 128, 0, False, 0),
    (16, 4, 128, 256, 2, [77, 5], 2 ** 30, 64, 0, 0, 0, 128, 0, False, 0), (32, 8, 128, 128, 1, [2000], 512, 0, 64, 1, 1, 0, 0, True, 8),
    (6, 3, 96, 128, 1, LONG, 2 ** 30, 0, 0, 1, 1, 50, 1, False, 0), (8, 1, 64, 64, 1, LONG, 33, 0, 5, 1, 1, 32, 0, True, 0),
    (5, 5, 32, 256, 2, SHORT, 2 ** 30, 0, 0, 1, 0, 32, 1, False, 3), (16, 2, 64, 128, 1, [30 + i for i in range(130)], 2 ** 30, 0, 0, 1, 1, 0, 0, False, 0),
    (4, 2, 24, 40, 1, SHORT, 2 ** 30, 0, 0, 1, 1, 16, 0, True, 0), (4, 2, 512, 64, 1, [300], 2 ** 30, 0, 0, 1, 1, 512, 0, False, 0)])
def test_step_as_two_launches(dtype, H, G, D, E, maps, lens, window, chunk, keep, append, norm, rot, layout, mixed, temp):
    from umbrella_amd import _lib
    from umbrella_amd.attn.cache import PagedSeqCache
    code, T = _lib.seq_dtype_code(dtype), len(lens)
    ld = maps * H * D + append * (maps * G * D + G * E) + H * E
    g = torch.Generator(device="cuda").manual_seed(H + D + E + T)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")                                              # noqa: E731
    proj, freq, bias = rnd(T, ld), torch.rand(max(rot // 2, 1), generator=g, device="cuda"), rnd(H, 40)
    wq, wk, sink = (1.0 + 0.1 * rnd(D)).to(dtype), (1.0 + 0.1 * rnd(D)).to(dtype), rnd(H)
    first = rnd(T, G * E)
    pos = torch.tensor([n - 1 for n in lens], dtype=torch.int32, device="cuda")
    k0 = v0 = None
    outs = []
    for step in (False, True):
        c = PagedSeqCache([(G, maps * D, 0, E)], [], sum(lens) + 100, T, "cuda", dtype, page=32)
        for b, n in enumerate(lens):
            c.open(b), c.extend(b, n)
        if k0 is None:
            k0, v0 = rnd(*c.kv[0]["k"].shape).to(dtype), rnd(*c.kv[0]["v"].shape).to(dtype)
        k, v = c.kv[0]["k"], c.kv[0]["v"]
        k.copy_(k0), v.copy_(v0)
        slot = torch.tensor([c.slot(b) for b in range(T)], dtype=torch.int32, device="cuda")
        if append:
            for b, n in enumerate(lens):
                page = c.seqs[b]["pages"][(n - 1) // 32]
                k[page, :, (n - 1) % 32], v[page, :, (n - 1) % 32] = float("nan"), float("nan")
        q, kept = torch.zeros(T, maps * H * D, device="cuda"), torch.zeros(T, G * E, device="cuda")
        out = torch.full((T + 1, H * E), 3.0, dtype=dtype, device="cuda")
        form = _lib.UmbAttnForm()
        form.maps, form.chunk, form.sink, form.eps, form.keep_first, form.gate_elem = maps, chunk, sink.data_ptr() if maps == 1 else None, 1e-6, keep, 1
        form.lambda_ = 0.3
        mix = _lib.UmbValueMix()
        if mixed:
            mix.first, mix.keep = first.data_ptr(), kept.data_ptr()
            mix.lambda_ = 0.4
        import ctypes as C
        part, gate = torch.zeros(4 << 20, device="cuda"), ld - H * E
        kv, w = c.struct(0), (wq, wk) if norm else (None, None)
        if step:
            _lib.seq_call("umb_attn_step", out, H * E, q, kv, proj, ld, append, *w, norm, 0, freq, rot, layout, 1.1, 0.2, temp, 1e-6, C.byref(mix), gate, bias,
                          40, pos, slot, T, H, G, D, E, window, D ** -0.5, 0.9, 0.0, form, part, part.numel(), code)
        else:
            _lib.seq_call("umb_attn_prep_mix", q, kv, proj, ld, append, *w, norm, 0, pos, slot, freq, rot, layout, 1.1, T, H, G, D, E, maps, 0.2, temp, 1e-6,
                          C.byref(mix), code)
            _lib.seq_call("umb_attn_attend", out, H * E, q, kv, proj, ld, gate, bias, 40, pos, slot, T, H, G, D, E, window, D ** -0.5, 0.9, 0.0, form, part,
                          part.numel(), code)
        assert bool((out[T] == 3.0).all()) and bool(torch.isfinite(out).all())
        outs.append((out[:T].clone(), k.clone(), v.clone(), kept))
    a, b = outs
    # rotation and norms may be contracted otherwise: one step of the storage type on the appended rows, a few fp32 steps through the scores
    step_of = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10, torch.float32: 2.0 ** -22}[dtype]
    for x, y in zip(a[1:], b[1:]):
        assert bool(((x.float() - y.float()).abs() <= step_of * x.float().abs() + 1e-6).all())
    assert bool(((a[0].float() - b[0].float()).abs() <= 2 * step_of * a[0].float().abs() + 1e-5).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,G,D,E,maps,rot,layout,norm_v", [(32, 8, 128, 128, 1, 128, 0, 1), (32, 8, 64, 256, 1, 64, 1, 1), (32, 8, 64, 64, 1, 64, 1, 0), (16, 4, 256, 256, 1, 256, 1, 0),
                                                            (16, 4, 128, 256, 2, 128, 0, 1), (8, 2, 96, 128, 1, 50, 1, 0)])
def test_step_appends_what_a_launch_of_its_own_does(dtype, H, G, D, E, maps, rot, layout, norm_v):
    """keys, values and the first layer's kept ones, bit by bit: a token's cached rows do not depend on the launch that prepared them"""
    import ctypes as C
    from umbrella_amd import _lib
    from umbrella_amd.attn.cache import PagedSeqCache
    code, T = _lib.seq_dtype_code(dtype), 150
    ld = maps * H * D + maps * G * D + G * E
    g = torch.Generator(device="cuda").manual_seed(H + D + E)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")                                              # noqa: E731
    proj, freq, first = rnd(T, ld), torch.rand(rot // 2, generator=g, device="cuda"), rnd(T, G * E)
    wq, wk = (1.0 + 0.1 * rnd(D)).to(dtype), (1.0 + 0.1 * rnd(D)).to(dtype)
    lens = [1 + i % 70 for i in range(T)]
    pos = torch.tensor([n - 1 for n in lens], dtype=torch.int32, device="cuda")
    outs = []
    for step in (False, True):
        c = PagedSeqCache([(G, maps * D, 0, E)], [], sum(lens) + 100, T, "cuda", dtype, page=32)
        for b, n in enumerate(lens):
            c.open(b), c.extend(b, n)
        c.kv[0]["k"].zero_(), c.kv[0]["v"].zero_()
        slot = torch.tensor([c.slot(b) for b in range(T)], dtype=torch.int32, device="cuda")
        q, kept, out = torch.zeros(T, maps * H * D, device="cuda"), torch.zeros(T, G * E, device="cuda"), torch.zeros(T, H * E, dtype=dtype, device="cuda")
        form, mix = _lib.UmbAttnForm(), _lib.UmbValueMix(first.data_ptr(), kept.data_ptr(), 0.4, 0.0)
        form.maps, form.eps, form.lambda_ = maps, 1e-6, 0.3
        kv = c.struct(0)
        if step:
            _lib.seq_call("umb_attn_step", out, H * E, q, kv, proj, ld, 1, wq, wk, 1, norm_v, freq, rot, layout, 1.1, 0.0, 0, 1e-6, C.byref(mix), -1, None, 0, pos,
                          slot, T, H, G, D, E, 2 ** 30, D ** -0.5, 1.0, 0.0, form, None, 0, code)
        else:
            _lib.seq_call("umb_attn_prep_mix", q, kv, proj, ld, 1, wq, wk, 1, norm_v, pos, slot, freq, rot, layout, 1.1, T, H, G, D, E, maps, 0.0, 0, 1e-6,
                          C.byref(mix), code)
        outs.append((kept, c.kv[0]["k"], c.kv[0]["v"]))
    assert float(outs[0][0].abs().sum()) > 0.0 and all(torch.equal(x, y) for x, y in zip(*outs))
