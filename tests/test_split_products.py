"""Products of few tokens whose K is summed in slabs, and the seams that add the slabs: against the sum of the slabs in float64."""
import pytest
import torch

U = 2.0 ** -24
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _code(name):
    from umbrella_amd import _lib
    return {"bf16": _lib.BF16, "fp16": _lib.F16, "fp32": _lib.F32}[name]


def test_split_rule_stays_inside_what_the_product_takes():
    from umbrella_amd import _lib
    split = _lib.load_seq().umb_seq_linear_split
    ptr = 1 << 20
    for code, item in ((_lib.BF16, 2), (_lib.F32, 4)):
        for T in (1, 16, 17, 32, 33, 64, 65, 2000):
            for N in (1, 16, 1000, 2048, 2049, 2730, 4096, 4097, 32000):
                for K in (8, 200, 256, 512, 1024, 2048, 2304, 8192, 14336):
                    parts = split(ptr, ptr, T, N, K, code)
                    assert 1 <= parts <= 4 and (parts == 1 or (T <= 64 and K * item % 512 == 0 and parts * 4 <= K * item // 512) or
                                                            (T > 64 and item == 2 and N >= 128 and K % 64 == 0 and parts * 4 <= K // 64)), (T, N, K)
        assert split(ptr + 8, ptr, 1, 2048, 8192, code) == 1 and split(ptr, ptr + 8, 1, 2048, 8192, code) == 1     # no 16-byte pieces


def test_up_to_64_tokens_the_number_of_slabs_follows_from_the_weights():
    """a token's sums are the same whatever else is in its step"""
    from umbrella_amd import _lib
    split = _lib.load_seq().umb_seq_linear_split
    ptr = 1 << 20
    for code in (_lib.BF16, _lib.F16, _lib.F32):
        for N in (16, 192, 1000, 2048, 2049, 2560, 2720, 2721, 3072, 4096, 4097, 5120, 8192, 32000):
            for K in (192, 512, 1024, 2048, 2304, 4096, 8192, 14336):
                assert len({split(ptr, ptr, T, N, K, code) for T in range(1, 65)}) == 1, (N, K)


def test_slabs_fit_the_room_that_a_workspace_has():
    """the number of slabs follows from the step and not from the workspace that earlier steps left: what pays among those that fit"""
    from umbrella_amd import _lib
    split = _lib.load_seq().umb_seq_linear_split
    ptr, seen = 1 << 20, set()
    for T in (1, 64, 65, 300, 2047, 2048, 2049, 2300, 2730, 2731, 4000, 4096, 4097, 6000, 8192, 8193, 20000):
        for N in (128, 1024, 2048, 4096, 8192):
            for K in (512, 2048, 4096, 8192, 14336):
                parts = split(ptr, ptr, T, N, K, _lib.BF16)
                assert parts * T <= max(T, min(4 * T, 8192)), (T, N, K, parts)
                seen.add((T, parts))
    assert (2049, 3) in seen and (2731, 2) in seen and (4096, 2) in seen


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("T,N,chunks,parts", [(1, 16, 2, 2), (1, 2048, 8, 2), (16, 40, 7, 3), (17, 2049, 5, 4), (33, 4096, 16, 2), (48, 130, 32, 4),
                                              (64, 2047, 33, 4), (65, 130, 2, 4), (257, 1001, 3, 4), (300, 2048, 5, 2), (1101, 520, 4, 3)])
def test_slabs_add_up_to_the_product(dtype, T, N, chunks, parts):
    from umbrella_amd import _lib
    dt, K = DTYPES[dtype], chunks * 512 // DTYPES[dtype].itemsize
    if T > 64 and dtype == "fp32":
        pytest.skip("slabs of many tokens are for 16-bit storage")
    g = torch.Generator().manual_seed(T * N + chunks)
    x, w, b = (torch.randn(s, generator=g).to(dt) for s in ((T, K), (N, K), (N,)))
    out = torch.full((parts + 1, T, N), 7.0, device="cuda:0")
    _lib.seq_call("umb_seq_linear_parts", out, x.cuda(), w.cuda(), b.cuda(), T, N, K, parts, _code(dtype))
    assert bool((out[parts] == 7.0).all())                     # and nothing behind the last slab
    want = x.double() @ w.double().T + b.double()
    bound = 4 * U * K ** 0.5 * (x.double().abs() @ w.double().abs().T + b.double().abs())      # fp32 sums of K products
    assert ((out[:parts].double().cpu().sum(0) - want).abs() <= bound).all()


# more row blocks than the chip holds workgroups (16 rows a block up to 32 tokens and in gate/up, 32 beyond): one block past it, ragged, a third
# round; as many chunks as the ring has slots, one less (not run on), and more; 65 tokens: two token tiles
RUNS = [(1, 16 * 768 + 1, 4), (8, 16 * 1600 - 3, 5), (16, 16 * 513, 4), (16, 16 * 512, 9), (17, 16 * 257 - 8, 3), (32, 16 * 530 + 2, 4), (32, 16 * 300, 2),
        (33, 32 * 256 + 2, 3), (48, 32 * 520 - 6, 8), (64, 32 * 257, 7), (65, 32 * 130, 4)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bf16", "fp32"])
@pytest.mark.parametrize("T,N,chunks", RUNS)
def test_streams_run_on_from_block_to_block(dtype, T, N, chunks):
    from umbrella_amd import _lib
    dt, K = DTYPES[dtype], chunks * 512 // DTYPES[dtype].itemsize
    g = torch.Generator(device="cuda").manual_seed(T * N + chunks)
    x, w, b = (torch.randn(s, generator=g, device="cuda").to(dt) for s in ((T, K), (N, K), (N,)))
    want, size = x.double() @ w.double().T + b.double(), x.double().abs() @ w.double().abs().T + b.double().abs()
    bound = 4 * U * K ** 0.5 * size
    out = torch.full((T + 1, N), 7.0, device="cuda")
    _lib.seq_call("umb_seq_linear", out, x, w, b, T, N, K, 0, _code(dtype))
    assert ((out[:T].double() - want).abs() <= bound).all() and bool((out[T] == 7.0).all())
    half = N // 2
    for n in {half, N // 2 * 2}:                               # stacked halves of half and of whole height: silu(gate) * up
        w2 = torch.cat([w[:n], w[:n].flip(0)]).contiguous()
        full = x.double() @ w2.double().T
        size = x.double().abs() @ w2.double().abs().T
        gate, up, tol = full[:, :n], full[:, n:], 4 * U * K ** 0.5 * size
        act = torch.full((T + 1, n), 7.0, dtype=dt, device="cuda")
        _lib.seq_call("umb_seq_linear", act, x, w2, None, T, 2 * n, K, 2, _code(dtype))
        ref = gate * torch.sigmoid(gate) * up
        ulp = {"bf16": 2.0 ** -8, "fp32": 2.0 ** -23}[dtype]
        slack = 1.1 * tol[:, :n] * up.abs() + gate.abs() * tol[:, n:] + 1.02 * ulp * ref.abs() + 1e-6 * ref.abs() + 1e-20
        assert ((act[:T].double() - ref).abs() <= slack).all() and bool((act[T] == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("W,groups", [(64, 1), (4096, 1), (2048, 4), (201, 3), (8200, 1)])
@pytest.mark.parametrize("parts", [1, 2, 3, 4])
def test_seams_add_the_slabs(W, groups, parts):
    """every seam over slabs gives what it gives over their sum, formed in the same order"""
    from umbrella_amd import _lib
    g = torch.Generator().manual_seed(W + parts)
    for T in (1, 5, 450 if W <= 4096 else 3):
        x, w1, w2, w3, w4 = (torch.randn(s, generator=g).cuda() for s in ((T, W), (W,), (W,), (W,), (W,)))
        y, y2 = (torch.randn(parts, T, W, generator=g).cuda() for _ in range(2))

        def total(t):
            s = t[0].clone()
            for p in range(1, parts):
                s += t[p]
            return s
        outs = []
        for slabs in (True, False):
            a, b, n = (y.clone(), y2.clone(), parts) if slabs else (total(y), total(y2), 1)
            xs = [x.clone() for _ in range(3)]
            hs = [torch.empty_like(x) for _ in range(3)]
            _lib.seq_call("umb_seq_resid_norm_parts", xs[0], hs[0], a.clone(), n, w1, w2, T, W, groups, 1e-5, _lib.F32)
            _lib.seq_call("umb_seq_pair_resid_norm_parts", xs[1], hs[1], a.clone(), n, b, n, w1, w2, 0.5, w3, w4, T, W, 1e-5, _lib.F32)
            _lib.seq_call("umb_hc_seam_parts", xs[2], hs[2], a.clone(), n, None, None, 0.5, None, w1, 1.0, T, W, 1, 1e-5, _lib.F32)
            outs.append(xs + hs)
        for got, want in zip(*outs):
            assert torch.equal(got, want)
        xs = torch.randn(T, 2, W, generator=g).cuda()             # several streams: the slabs are summed in front of the seam
        hs = [torch.empty(T, W, device="cuda:0") for _ in range(2)]
        both = [xs.clone(), xs.clone()]
        _lib.seq_call("umb_hc_seam_parts", both[0], hs[0], y.clone(), parts, None, None, 0.5, None, w1, 1.0, T, W, 2, 1e-5, _lib.F32)
        _lib.seq_call("umb_hc_seam", both[1], hs[1], total(y), None, None, 0.5, None, w1, 1.0, T, W, 2, 1e-5, _lib.F32)
        assert torch.equal(both[0], both[1]) and torch.equal(hs[0], hs[1])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bf16", "fp32"])
@pytest.mark.parametrize("N,chunks", [(4134, 2), (4134, 8), (2048, 9), (9000, 12)])
def test_a_row_is_summed_in_one_order_whatever_the_batch(dtype, N, chunks):
    """K from several places, one or two row tiles a workgroup, workgroups that run on: the same bits for a token alone and among others"""
    from umbrella_amd import _lib
    dt, K = DTYPES[dtype], chunks * 512 // DTYPES[dtype].itemsize
    g = torch.Generator(device="cuda").manual_seed(N + chunks)
    x, w = (torch.randn(s, generator=g, device="cuda").to(dt) for s in ((64, K), (N, K)))
    full = torch.empty(64, N, device="cuda")
    _lib.seq_call("umb_seq_linear", full, x, w, None, 64, N, K, 0, _code(dtype))
    for lo, n in ((0, 1), (5, 8), (7, 16), (30, 17), (20, 33), (10, 48)):
        part = torch.empty(n, N, device="cuda")
        _lib.seq_call("umb_seq_linear", part, x[lo:lo + n].contiguous(), w, None, n, N, K, 0, _code(dtype))
        assert torch.equal(part, full[lo:lo + n])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bf16", "fp32"])
@pytest.mark.parametrize("N,K", [(2048, 2048), (2600, 4096), (4096, 4096), (4096, 14336), (4112, 4096)])
def test_a_row_has_one_order_in_slabs_too(dtype, N, K):
    """what a sublayer's last product of up to 64 tokens leaves, slab by slab: the same bits for a token alone and among others"""
    from umbrella_amd import _lib
    dt, lib = DTYPES[dtype], _lib.load_seq()
    g = torch.Generator(device="cuda").manual_seed(N + K)
    x, w = (torch.randn(s, generator=g, device="cuda").to(dt) for s in ((64, K), (N, K)))
    outs = []
    for lo, n in ((0, 64), (0, 1), (5, 8), (7, 16), (30, 32), (20, 33), (10, 48)):
        part = x[lo:lo + n].contiguous()
        parts = lib.umb_seq_linear_split(part.data_ptr(), w.data_ptr(), n, N, K, _code(dtype))
        out = torch.empty(parts, n, N, device="cuda")
        _lib.seq_call("umb_seq_linear_parts", out, part, w, None, n, N, K, parts, _code(dtype))
        outs.append(out)
        assert out.shape[0] == outs[0].shape[0] and torch.equal(out, outs[0][:, lo:lo + n])


# every seam behind a product in slabs, and the one that takes whole sums (a next sublayer that reads through a convolution), in a whole forward: two
# layers whose last products split at these tokens, against the same forward without room for slabs
def _split_models():
    import fidizen_helpers as F
    import potosun_helpers as P
    import seqmix_helpers as G
    import tomopel_helpers as M
    import tutunex_helpers as U
    W, ff = 1024, 4096
    return {"groups": lambda dt, **kw: G.build(G.config([G.attn_layer(heads=16, dim=128, ff=ff), G.gla_layer(heads=8, dim=32, vdim=256, ff=ff)], width=W), dt, **kw),
            "pair": lambda dt, **kw: U.build(U.config([U.layer(U.parallel(heads=16, kv_heads=2, dim=16, vdim=128, r_heads=8, r_kv=2, r_dim=32, r_vdim=256), ff=ff),
                                                       U.layer(U.attention(heads=16, dim=16, vdim=128), ff=ff)], width=W), dt, **kw),
            "forms": lambda dt, **kw: P.build(P.config([P.layer(P.biased(heads=16, dim=16, vdim=128), ff=ff), P.layer(P.latent(heads=16, dim=16, vdim=128), ff=ff)],
                                                       width=W), dt, **kw),
            "convolution": lambda dt, **kw: F.build(F.config([F.layer(heads=16, dim=16, vdim=128, ff=ff), F.layer(heads=16, dim=16, vdim=128, ff=ff)], width=W), dt, **kw),
            "one stream": lambda dt, **kw: M.build(M.config([M.layer(M.mingru(width=2048), ff=ff), M.layer(M.mingru(width=2048), ff=ff)], width=W, streams=1), dt, **kw),
            "two streams": lambda dt, **kw: M.build(M.config([M.layer(M.mingru(width=2048), ff=ff), M.layer(M.mingru(width=2048), ff=ff)], width=W, streams=2), dt, **kw)}


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bf16", "fp32"])
@pytest.mark.parametrize("kind", ["groups", "pair", "forms", "convolution", "one stream", "two streams"])
def test_forwards_in_slabs(kind, dtype):
    from umbrella_amd import _lib
    dt = DTYPES[dtype]
    m, _ = _split_models()[kind](dt, max_length=400)
    m.reserve(600)
    room, split = m._ws.y_rows, _lib.load_seq().umb_seq_linear_split
    assert room == 4 * 600
    g = torch.Generator().manual_seed(3)
    for lens in ([1], [20, 13], [1, 1, 1], [350, 250]):
        T = sum(lens)
        if T <= 64 or dtype == "bf16":
            assert split(1 << 20, 1 << 20, T, 1024, 4096, _code(dtype)) > 1 and split(1 << 20, 1 << 20, T, 1024, 2048, _code(dtype)) > 1
        ids, runs = [torch.randint(0, 90, (n,), generator=g).tolist() for n in lens], []
        for rows in (room, 0):
            m._ws.y_rows = rows
            m.clear()
            for i in range(len(lens)):
                m.open(i)
            logits, trace = m.forward_batch(list(enumerate(ids)), trace=True)
            runs.append([logits.double().clone(), *trace.double().clone()])
        for got, want in zip(*runs):
            # fp32 sums in another order; 16 bits: a rounding of 2^-9 that falls the other way in some of a few dozen places of a layer
            assert (got - want).norm() <= (2e-5 if dtype == "fp32" else 2e-2) * want.norm(), (kind, lens)
        assert T > 64 and dtype == "fp32" or not torch.equal(runs[0][-1], runs[1][-1])        # sums in slabs they were


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["groups", "pair", "one stream"])
def test_a_workspace_of_single_floats(kind):
    """outputs of a sublayer that are not 16-byte aligned: whole sums, as a product without slabs takes them"""
    m, _ = _split_models()[kind](torch.bfloat16, max_length=700)
    m.reserve(600)
    g, runs = torch.Generator().manual_seed(4), []
    ids = torch.randint(0, 90, (600,), generator=g).tolist()
    for off in (0, 1):
        bufs = [torch.full((4 * 600 * 1024 + 4,), 5.0, device="cuda") for _ in range(2)]
        m._ws.y, m._ws.y2 = (b.data_ptr() + 4 * off for b in bufs)
        m.clear()
        m.open(0)
        runs.append(m.forward_batch([(0, ids)]).double().clone())
        assert all(bool((b[:off] == 5.0).all()) and bool((b[off + 4 * 600 * 1024:] == 5.0).all()) for b in bufs)
    # a rounding of 2^-9 that falls the other way in some of a few dozen places of a layer
    assert (runs[0] - runs[1]).norm() <= 2e-2 * runs[0].norm()
