"""Rows of 64 and 128 features that many (token, head) slots are prepared in by quads: against launches of few slots."""
import pytest
import test_prompt_kernels as prompt
import torch

pytestmark = pytest.mark.gpu


# both layouts of pairs; nothing, a part and all of a row turned; one and two maps; rows that end inside a wave's sixteen; queries alone; values of another size
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("H,G,D,E,maps,layout,rot,append,norm,mixed", [(8, 2, 64, 64, 1, 0, 64, 1, 1, True), (9, 3, 128, 64, 2, 1, 80, 1, 0, False),
                                                                       (17, 17, 64, 128, 1, 1, 36, 1, 1, True), (30, 2, 128, 128, 1, 0, 48, 0, 1, False),
                                                                       (15, 1, 128, 128, 1, 0, 128, 1, 0, True), (12, 4, 64, 64, 1, 1, 0, 1, 1, False)])
def test_attention_slots(dtype, H, G, D, E, maps, layout, rot, append, norm, mixed):
    prompt.test_many_slots_are_prepared_as_few_are(dtype, H, G, D, E, maps, layout, rot, append, norm, mixed)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("H,G,D,rot", [(15, 1, 64, 32), (16, 8, 128, 128), (20, 4, 64, 0), (17, 1, 128, 60)])
def test_pooled_slots(dtype, H, G, D, rot):
    prompt.test_many_pooled_slots_are_prepared_as_few_are(dtype, H, G, D, rot)


# heads that quads are aligned in, few of them and many, a last wave in part; a normaliser's column behind a head (rows of Dv + 1), weights for all and of each head
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("T,H,Dv", [(1, 3, 64), (7, 1, 128), (1, 1, 256), (1800, 11, 64), (2467, 7, 128), (601, 9, 256)])
@pytest.mark.parametrize("den,weights,kind", [(False, 0, 0), (True, 1, 1), (True, 2, 0)])
def test_head_gates(dtype, T, H, Dv, den, weights, kind):
    from umbrella_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(T + Dv)
    cols, ld, ldo = Dv + int(den), H * Dv + 5, H * Dv + 4
    o, proj, mrun = (torch.randn(s, generator=g, device="cuda") for s in ((T, H, cols), (T, ld), (T, H)))
    w = torch.randn(Dv if weights == 1 else H * Dv, generator=g, device="cuda").to(dtype) if weights else None
    out = torch.full((T + 1, ldo), 7.0, dtype=dtype, device="cuda")
    _lib.seq_call("umb_head_gate", out, ldo, o, cols, Dv if den else -1, mrun if den else None, proj, ld, 3, w, int(weights == 2), kind, T, H, Dv, 1e-5, 1.2,
                  _lib.seq_dtype_code(dtype))
    v, gate = o[..., :Dv].double(), proj[:, 3:3 + H * Dv].double().view(T, H, Dv)
    if den:
        v = v / (torch.maximum(o[..., Dv].double().abs(), torch.exp(-mrun.double())) + 1e-6)[..., None]
    v = v * 1.2 / torch.sqrt((v * v).mean(-1, keepdim=True) + 1e-5)
    if weights:
        v = v * (w.double() if weights == 1 else w.double().view(H, Dv))
    want = (v * torch.sigmoid(gate) * (gate if kind == 0 else 1.0)).view(T, -1)
    assert bool((out[T] == 7.0).all()) and bool((out[:T, H * Dv:] == 7.0).all())
    eps = torch.finfo(dtype).eps
    assert bool(((out[:T, :H * Dv].double() - want).abs() <= 0.51 * eps * want.abs() + 2e-6 * want.abs() + 1e-7).all())


# ---- the same bits as the kernels that take what quads are not aligned in (an element or a pair a lane)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("H,G,D,E,maps,layout,rot,append,norm,mixed", [(8, 2, 64, 64, 1, 0, 64, 1, 1, True), (9, 3, 128, 64, 2, 1, 80, 1, 0, False),
                                                                       (17, 17, 64, 128, 1, 1, 36, 1, 1, True), (30, 2, 128, 128, 1, 0, 48, 0, 1, False),
                                                                       (32, 8, 128, 128, 2, 0, 128, 1, 1, False), (32, 8, 64, 64, 1, 1, 0, 1, 1, False)])
def test_attention_slots_bit_by_bit(dtype, H, G, D, E, maps, layout, rot, append, norm, mixed, T=2880):
    from umbrella_amd import _lib
    code = _lib.seq_dtype_code(dtype)
    g = torch.Generator(device="cuda").manual_seed(D + E)
    HQ, GK, GV = maps * H, append * maps * G, append * G
    ld = HQ * D + GK * D + GV * E + 5
    proj, freq, firsts = torch.randn(T, ld, generator=g, device="cuda"), torch.rand(64, generator=g, device="cuda"), torch.randn(T, G * E, generator=g, device="cuda")
    wq, wk = (torch.randn(D, generator=g, device="cuda").to(dtype) for _ in range(2))
    pos, slot = torch.arange(T, device="cuda", dtype=torch.int32), torch.zeros(T, device="cuda", dtype=torch.int32)
    outs = []
    for shift in (0, 1):                                       # q 4 bytes behind 16: no quads
        c, _, _, _ = prompt._decode_store([T], G, maps * D, E, 0, dtype, 32, 1)
        q, keep = torch.zeros(T * HQ * D + 4, device="cuda"), torch.zeros(T, G * E, device="cuda")
        m = _lib.UmbValueMix(firsts.data_ptr(), keep.data_ptr(), 0.3, 0.0) if mixed else None
        _lib.seq_call("umb_attn_prep_mix", q[shift:], c.struct(0), proj, ld, append, wq if norm else None, wk if norm else None, norm, norm, pos, slot,
                      freq if rot else None, rot, layout, 1.1, T, H, G, D, E, maps, 0.1, 100, 1e-5, m, code)
        outs.append([q[shift:shift + T * HQ * D].clone(), keep, c.kv[0]["k"], c.kv[0]["v"]])
    assert all(torch.equal(x, y) for x, y in zip(*outs))


# few slots a token: the fewest that go in quads, one fewer, and waves whose last rows are none
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("H,G,D,E,maps,layout,rot,append,norm,mixed", [(3, 1, 128, 128, 1, 0, 128, 1, 1, True), (2, 1, 128, 64, 1, 1, 64, 1, 1, False), (2, 1, 64, 128, 1, 0, 32, 1, 1, True),
                                                                       (1, 1, 64, 64, 1, 1, 64, 1, 1, False), (1, 1, 64, 64, 2, 0, 64, 0, 1, False),
                                                                       (1, 1, 128, 128, 1, 1, 128, 0, 1, False), (3, 3, 64, 64, 1, 1, 64, 1, 0, True)])
def test_few_attention_slots_bit_by_bit(dtype, H, G, D, E, maps, layout, rot, append, norm, mixed):
    slots = maps * (H + append * G) + append * G
    test_attention_slots_bit_by_bit(dtype, H, G, D, E, maps, layout, rot, append, norm, mixed, T=24576 // slots + 7)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("H,G,D,rot", [(32, 8, 64, 64), (16, 8, 128, 128), (20, 4, 64, 0), (17, 1, 128, 60)])
def test_pooled_slots_bit_by_bit(dtype, H, G, D, rot):
    from umbrella_amd import _lib
    T, code = 1700, _lib.seq_dtype_code(dtype)
    g = torch.Generator(device="cuda").manual_seed(D)
    proj, freq = torch.randn(T, (H + G) * D + 3, generator=g, device="cuda"), torch.rand(64, generator=g, device="cuda")
    pos, slot = torch.arange(T, device="cuda", dtype=torch.int32), torch.zeros(T, device="cuda", dtype=torch.int32)
    outs = []
    for shift in (0, 1):
        c, _, _, _ = prompt._decode_store([T], G, D, D, 5, dtype, 32, 1)
        q = torch.zeros(T * H * D + 4, device="cuda")
        _lib.seq_call("umb_pwa_prep", q[shift:], c.struct(0), proj, proj.shape[1], pos, slot, freq if rot else None, T, H, G, D, rot, 1e-5, code)
        outs.append([q[shift:shift + T * H * D].clone(), c.kv[0]["k"], c.kv[0]["v"]])
    assert all(torch.equal(x, y) for x, y in zip(*outs))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("T,H,Dv", [(1800, 11, 64), (2467, 7, 128), (601, 9, 256), (1, 16, 256), (7, 1, 128)])
@pytest.mark.parametrize("den,weights,kind", [(False, 0, 0), (True, 1, 1), (True, 2, 0)])
def test_head_gates_bit_by_bit(dtype, T, H, Dv, den, weights, kind):
    from umbrella_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(T + Dv)
    cols, ld, outs = Dv + int(den), H * Dv + 5, []
    o, proj, mrun = (torch.randn(s, generator=g, device="cuda") for s in ((T, H, cols), (T, ld), (T, H)))
    w = torch.randn(Dv if weights == 1 else H * Dv, generator=g, device="cuda").to(dtype) if weights else None
    for ldo in (H * Dv, H * Dv + 1):
        out = torch.zeros((T, ldo), dtype=dtype, device="cuda")
        _lib.seq_call("umb_head_gate", out, ldo, o, cols, Dv if den else -1, mrun if den else None, proj, ld, 3, w, int(weights == 2), kind, T, H, Dv, 1e-5, 1.2,
                      _lib.seq_dtype_code(dtype))
        outs.append(out[:, :H * Dv])
    assert torch.equal(*outs)


# ---- infinities, NaN and the ends of the range: where the kernels that take an element a lane have them, in no other row
def _ends(x, seed):
    """every eleventh row of x [rows, cols] with one of them somewhere"""
    g = torch.Generator().manual_seed(seed)
    for k, r in enumerate(range(3, x.shape[0], 11)):
        x[r, int(torch.randint(x.shape[1], (1,), generator=g))] = (float("inf"), float("-inf"), float("nan"), 3e38, 0.0)[k % 5]
        if k % 5 == 4:
            x[r] = 0.0
    return x


def _same(a, b):
    return torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(a[~torch.isnan(a)], b[~torch.isnan(b)])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("H,G,D,E,layout,rot,norm,mixed", [(32, 8, 64, 64, 0, 40, 1, True), (32, 8, 128, 128, 1, 64, 0, False), (16, 8, 128, 64, 0, 128, 1, False)])
def test_ends_of_the_range_in_attention_slots(dtype, H, G, D, E, layout, rot, norm, mixed):
    from umbrella_amd import _lib
    T, code, ld = 1600, _lib.seq_dtype_code(dtype), (H + G) * D + G * E
    g = torch.Generator(device="cuda").manual_seed(D + E)
    proj, freq, firsts = torch.randn(T, ld, generator=g, device="cuda"), torch.rand(64, generator=g, device="cuda"), torch.randn(T, G * E, generator=g, device="cuda")
    _ends(proj, D), _ends(firsts, E)
    wq, wk = (torch.randn(D, generator=g, device="cuda").to(dtype) for _ in range(2))
    pos, slot, outs = torch.arange(T, device="cuda", dtype=torch.int32), torch.zeros(T, device="cuda", dtype=torch.int32), []
    for shift in (0, 1):
        c, _, _, _ = prompt._decode_store([T], G, D, E, 0, dtype, 32, 1)
        q, keep = torch.zeros(T * H * D + 4, device="cuda"), torch.zeros(T, G * E, device="cuda")
        m = _lib.UmbValueMix(firsts.data_ptr(), keep.data_ptr(), 0.3, 0.0) if mixed else None
        _lib.seq_call("umb_attn_prep_mix", q[shift:], c.struct(0), proj, ld, 1, wq if norm else None, wk if norm else None, norm, norm, pos, slot, freq, rot, layout,
                      1.1, T, H, G, D, E, 1, 0.1, 100, 1e-5, m, code)
        outs.append([q[shift:shift + T * H * D].clone(), keep, c.kv[0]["k"].float(), c.kv[0]["v"].float()])
    assert all(_same(x, y) for x, y in zip(*outs))
    rows = outs[0][0].view(T, H * D)
    assert bool(torch.isfinite(rows[0]).all()) and 0 < int((~torch.isfinite(rows)).any(1).sum()) <= 4 * (T // 11 + 1) // 5 + 1


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,G,D,rot", [(32, 8, 64, 64), (16, 8, 128, 60)])
def test_ends_of_the_range_in_pooled_slots(dtype, H, G, D, rot):
    from umbrella_amd import _lib
    T, code = 1700, _lib.seq_dtype_code(dtype)
    g = torch.Generator(device="cuda").manual_seed(D)
    proj, freq = _ends(torch.randn(T, (H + G) * D, generator=g, device="cuda"), D), torch.rand(64, generator=g, device="cuda")
    pos, slot, outs = torch.arange(T, device="cuda", dtype=torch.int32), torch.zeros(T, device="cuda", dtype=torch.int32), []
    for shift in (0, 1):
        c, _, _, _ = prompt._decode_store([T], G, D, D, 5, dtype, 32, 1)
        q = torch.zeros(T * H * D + 4, device="cuda")
        _lib.seq_call("umb_pwa_prep", q[shift:], c.struct(0), proj, proj.shape[1], pos, slot, freq, T, H, G, D, rot, 1e-5, code)
        outs.append([q[shift:shift + T * H * D].clone(), c.kv[0]["k"].float(), c.kv[0]["v"].float()])
    assert all(_same(x, y) for x, y in zip(*outs)) and bool(torch.isnan(outs[0][0]).any())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("T,H,Dv", [(1800, 11, 64), (2467, 7, 128), (601, 9, 256)])
@pytest.mark.parametrize("den,kind", [(False, 0), (True, 1)])
def test_ends_of_the_range_in_head_gates(dtype, T, H, Dv, den, kind):
    from umbrella_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(T + Dv)
    cols, outs = Dv + int(den), []
    o, proj, mrun = (torch.randn(s, generator=g, device="cuda") for s in ((T * H, cols), (T, H * Dv), (T, H)))
    _ends(o, Dv), _ends(proj, T)
    mrun[5], mrun[6], mrun[7] = float("inf"), float("-inf"), float("nan")
    for ldo in (H * Dv, H * Dv + 1):
        out = torch.zeros((T, ldo), dtype=dtype, device="cuda")
        _lib.seq_call("umb_head_gate", out, ldo, o, cols, Dv if den else -1, mrun if den else None, proj, H * Dv, 0, None, 0, kind, T, H, Dv, 1e-5, 1.2,
                      _lib.seq_dtype_code(dtype))
        outs.append(out[:, :H * Dv].float())
    assert _same(*outs) and bool(torch.isnan(outs[0]).any()) and bool(torch.isfinite(outs[0]).any())
