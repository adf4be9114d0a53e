"""Staged matrix products of prompts (csrc/gemm_tile.h) at the edges of their tiles, against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# tile of the launch: (T, N, K).  256 x 256 (0.7 of a round of 256 workgroups, one row / column past a tile); 128 x 128 (more than
# 256 of them); the two K-split forms at whole, ragged and unaligned N; one stage of 64 k, an odd number of stages, two stages
SHAPES = [(2049, 6145, 64), (2048, 6160, 192), (2300, 2592, 128), (2300, 2590, 320), (300, 200, 128), (257, 130, 256), (1024, 2050, 384),
          (256, 128, 64), (1100, 2944, 64)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,N,K", SHAPES)
def test_staged_linear(dtype, T, N, K):
    from umbrella_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(T + N + K)
    x, w, b = (torch.randn(s, generator=g, device="cuda").to(dtype) for s in ((T, K), (N, K), (N,)))
    code = _lib.seq_dtype_code(dtype)
    full, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    # an fp32 sum of K products in any order: at most K roundings of 2^-24 of the sum of sizes (and two more for the bias)
    tol = 2.0 ** -24 * (K + 2) * (size + b.double().abs())
    out = torch.full((T + 1, N), 7.0, device="cuda")
    _lib.seq_call("umb_seq_linear", out, x, w, b, T, N, K, 0, code)
    assert ((out[:T].double() - (full + b.double())).abs() <= tol).all() and bool((out[T] == 7.0).all())
    out_dt = torch.full((T + 1, N), 7.0, dtype=dtype, device="cuda")
    _lib.seq_call("umb_seq_linear", out_dt, x, w, None, T, N, K, 1, code)
    half_ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11       # unit roundoff of 8 and 11 significant bits
    assert ((out_dt[:T].double() - full).abs() <= 1.01 * half_ulp * full.abs() + tol + 2.0 ** -25).all() and bool((out_dt[T] == 7.0).all())
    if N % 2 == 0:                       # stacked halves: silu(gate) * up; |d silu| <= 1.1 |d gate|
        half = N // 2
        gate, up, tg, tu = full[:, :half], full[:, half:], tol[:, :half], tol[:, half:]
        want = gate * torch.sigmoid(gate) * up
        act = torch.full((T + 1, half), 7.0, dtype=dtype, device="cuda")
        _lib.seq_call("umb_seq_linear", act, x, w, None, T, N, K, 2, code)
        bound = 1.02 * half_ulp * want.abs() + 1.1 * tg * up.abs() + gate.abs() * tu + 1e-6 * want.abs() + 2.0 ** -25
        assert ((act[:T].double() - want).abs() <= bound).all() and bool((act[T] == 7.0).all())


# wide products of packed dense weights (csrc/dgemm.hip): every tile (one token past 64, a whole one, ragged, 257 = two of 160), K slabs that
# divide and that do not, a last row tile of 16 rows
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,N,K,S", [(65, 272, 256, 1), (128, 512, 1024, 3), (257, 28672, 128, 1), (300, 4112, 256, 2), (1024, 14336, 128, 1),
                                     (200, 256, 2048, 5), (513, 2064, 384, 1)])
def test_wide_dense_product(dtype, T, N, K, S):
    from umbrella_amd import _lib
    from umbrella_amd.models.llama import PackedLinear
    g = torch.Generator(device="cuda").manual_seed(T + N + K)
    x, w = (torch.randn(s, generator=g, device="cuda").to(dtype) for s in ((T, K), (N, K)))
    full, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    tol = 2.0 ** -24 * (K + S) * size
    lin, code = PackedLinear.from_dense(w), _lib.dtype_code(dtype)
    part = torch.full((S + 1, T, N), 7.0, device="cuda")
    _lib.call("umb_gemm", part, x, x.stride(0), lin.w, None, T, N, K, 0, S, lin.Rtb, 0, code)
    assert ((part[:S].double().sum(0) - full).abs() <= tol).all() and bool((part[S] == 7.0).all())
    half_ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    out = torch.full((T + 1, N), 7.0, device="cuda")
    _lib.call("umb_gemm", out, x, x.stride(0), lin.w, None, T, N, K, 0, 1, lin.Rtb, 1, code)
    assert ((out[:T].double() - full).abs() <= 1.01 * half_ulp * full.abs() + tol + 2.0 ** -25).all() and bool((out[T] == 7.0).all())
    inter = PackedLinear.from_dense(w, interleave=True)               # gate and up rows in pairs
    act = torch.full((T + 1, N // 2), 7.0, dtype=dtype, device="cuda")
    _lib.call("umb_gemm", act, x, x.stride(0), inter.w, None, T, N, K, 0, 1, inter.Rtb, 2, code)
    gate, up, tg, tu = full[:, :N // 2], full[:, N // 2:], tol[:, :N // 2], tol[:, N // 2:]
    want = gate * torch.sigmoid(gate) * up
    # gate, up, silu and the product are each rounded once (|d silu| <= 1.1 |d gate|); 2e-6: the fast exponential
    bound = 1.05 * half_ulp * (1.1 * gate.abs() * up.abs() + 3 * want.abs()) + 1.1 * tg * up.abs() + 1.1 * gate.abs() * tu + 2e-6 * want.abs() + 2.0 ** -24
    assert ((act[:T].double() - want).abs() <= bound).all() and bool((act[T] == 7.0).all())


# the chunked kernel of few tokens: token counts around its tiles (8 / 16 / 32 / 48 / 64 and two token tiles), one chunk of K, fewer chunks than
# ring slots, ragged output rows
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("N,K", [(40, 256), (4134, 512), (272, 1280)])
def test_few_token_linear(dtype, N, K):
    from umbrella_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(N + K)
    code = _lib.seq_dtype_code(dtype)
    x, w, b = (torch.randn(s, generator=g, device="cuda").to(dtype) for s in ((100, K), (N, K), (N,)))
    full, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    tol = 2.0 ** -24 * (K + 2) * (size + b.double().abs())
    unit = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}[dtype]
    rows = None
    for T in (1, 2, 7, 8, 9, 17, 33, 48, 64, 65, 100):
        out = torch.full((T + 1, N), 7.0, device="cuda")
        _lib.seq_call("umb_seq_linear", out, x[:T].contiguous(), w, b, T, N, K, 0, code)
        assert ((out[:T].double() - (full[:T] + b.double())).abs() <= tol[:T]).all() and bool((out[T] == 7.0).all())
        rows = out[:1].clone() if rows is None else rows
        assert torch.equal(out[:1], rows)                      # the sum's order does not depend on the other rows
        half = N // 2
        act = torch.full((T + 1, half), 7.0, dtype=dtype, device="cuda")
        _lib.seq_call("umb_seq_linear", act, x[:T].contiguous(), w, None, T, N, K, 2, code)
        gate, up, tg, tu = full[:T, :half], full[:T, half:], tol[:T, :half], tol[:T, half:]
        want = gate * torch.sigmoid(gate) * up
        bound = 1.02 * unit * want.abs() + 1.1 * tg * up.abs() + gate.abs() * tu + 1e-6 * want.abs() + 2.0 ** -25
        assert ((act[:T].double() - want).abs() <= bound).all() and bool((act[T] == 7.0).all())


UNIT = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}


def _bounded(got, want, tol, unit=0.0):
    """tol: of the fp32 value; unit: its rounding to storage"""
    return bool(((got.double() - want).abs() <= 1.02 * unit * want.abs() + tol + 2.0 ** -25).all())


# whole 512-byte chunks of K in a batch of problems, row strides beyond the row, output gates: launches of few workgroups (the ring) and of more
# than one per unit (the one-tile kernels); one chunk and several
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("B,N,K", [(3, 40, 512), (5, 72, 256), (40, 200, 256), (2, 130, 1280)])
@pytest.mark.parametrize("T", [1, 7, 17, 48, 70, 300])
def test_batched_linear_in_whole_chunks(dtype, B, N, K, T):
    from umbrella_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(T + N + K)
    code, ldx, ldo = _lib.seq_dtype_code(dtype), B * K + 256, B * N + 5
    x, w = torch.randn(T, ldx, generator=g, device="cuda").to(dtype), torch.randn(B, N, K, generator=g, device="cuda").to(dtype)
    gate = torch.randn(T, B * N + 3, generator=g, device="cuda")
    xs = x[:, :B * K].double().view(T, B, K).transpose(0, 1).contiguous()
    wt = w.double().transpose(1, 2).contiguous()
    full, size = (torch.bmm(a, b).transpose(0, 1).reshape(T, B * N) for a, b in ((xs, wt), (xs.abs(), wt.abs())))
    tol = 2.0 ** -24 * (K + 2) * size
    for epi in (0, 1, 3, 7):
        out = torch.full((T + 1, ldo), 7.0, dtype=torch.float32 if epi == 0 else dtype, device="cuda")
        _lib.seq_call("umb_seq_linear_batched", out, x, w, T, N, K, ldx, ldo, B, K, N * K, N, epi, gate if epi > 1 else None, B * N + 3,
                      N if epi == 3 else 1, code)
        f = 1.0
        if epi == 3:
            f = torch.sigmoid(gate[:, :B * N].double())
        elif epi == 7:
            f = torch.sigmoid(gate[:, :B].double()).repeat_interleave(N, 1)
        # a quotient by 1 + e^-gate behind the sum: 2^-22 of it
        assert _bounded(out[:T, :B * N], full * f, tol + 2.0 ** -22 * (full * f).abs(), UNIT[dtype] if epi else 0.0), epi
        assert bool((out[T] == 7.0).all()) and bool((out[:, B * N:] == 7.0).all())


def _glu(kind, gate, up):
    if kind == 5:                                          # limit 1.5, alpha 1.7
        gate, up = gate.clamp(max=1.5), up.clamp(-1.5, 1.5)
        return gate * torch.sigmoid(1.7 * gate) * (up + 1)
    if kind == 6:
        return torch.nn.functional.gelu(gate, approximate="tanh") * up
    return torch.nn.functional.silu(gate) * up


# tile lists in whole chunks: whole, partial and empty tiles, every epilogue; output rows few and many, so that both kernels run
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("tile_rows", [16, 64])
@pytest.mark.parametrize("N,K", [(72, 512), (1500, 256), (40, 1280)])
def test_grouped_linear_in_whole_chunks(dtype, tile_rows, N, K):
    from umbrella_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(tile_rows + N + K)
    code, E = _lib.seq_dtype_code(dtype), 4
    tiles = [(2, 0, tile_rows), (2, tile_rows, 3), (0, tile_rows + 3, 1), (3, tile_rows + 4, tile_rows - 1), (0, 0, 0), (1, 2 * tile_rows + 3, 9)]
    T = 2 * tile_rows + 12
    grp = torch.zeros(T, dtype=torch.long, device="cuda")
    for e, r0, n in tiles:
        grp[r0:r0 + n] = e
    tl = torch.tensor(tiles, dtype=torch.int32, device="cuda")
    x, w = torch.randn(T, K, generator=g, device="cuda").to(dtype), (0.1 * torch.randn(E, 2 * N, K, generator=g, device="cuda")).to(dtype)
    full, size = torch.empty(T, 2 * N, dtype=torch.float64, device="cuda"), torch.empty(T, 2 * N, dtype=torch.float64, device="cuda")
    for e in range(E):
        full[grp == e], size[grp == e] = x[grp == e].double() @ w[e].double().T, x[grp == e].double().abs() @ w[e].double().abs().T
    tol = 2.0 ** -24 * (K + 2) * size
    gate, up, tg, tu = full[:, :N], full[:, N:], tol[:, :N], tol[:, N:]
    for epi in (0, 1, 4, 2, 5, 6):
        dual = epi in (2, 5, 6)
        out = torch.full((T + 1, N if dual else 2 * N), 7.0, dtype=torch.float32 if epi == 0 else dtype, device="cuda")
        if epi == 5:
            _lib.seq_call("umb_seq_linear_grouped_glu", out, x, w, tl, len(tiles), tile_rows, 2 * N * K, 2 * N, K, 1.5, 1.7, code)
        else:
            _lib.seq_call("umb_seq_linear_grouped", out, x, w, tl, len(tiles), tile_rows, 2 * N * K, 2 * N, K, epi, code)
        if dual:                                           # |d act / d gate| <= 1.2 for the three, |act| <= |gate| + 0.3
            want = _glu(epi, gate, up)
            assert _bounded(out[:T], want, 1.2 * tg * (up.abs() + 1) + (gate.abs() + 0.3) * tu + 2e-6 * (want.abs() + up.abs()), UNIT[dtype]), epi
        elif epi == 4:
            want = full.clamp(min=0).pow(2)
            assert _bounded(out[:T], want, 2 * tol * full.abs() + tol * tol + 2.0 ** -23 * want, UNIT[dtype])
        else:
            assert _bounded(out[:T], full, tol, UNIT[dtype] if epi else 0.0)
        assert bool((out[T] == 7.0).all())


# the remaining epilogues of the dense products: the ring (whole chunks, few tokens) and the staged tiles (many tokens)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("T,N,K", [(5, 72, 512), (30, 200, 256), (60, 40, 768), (300, 260, 192), (257, 2304, 128)])
def test_epilogues_of_linears(dtype, T, N, K):
    from umbrella_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(T + N + K)
    code = _lib.seq_dtype_code(dtype)
    x, w, b = torch.randn(T, K, generator=g, device="cuda").to(dtype), (0.1 * torch.randn(N, K, generator=g, device="cuda")).to(dtype), torch.randn(N, generator=g, device="cuda").to(dtype)
    full, size = x.double() @ w.double().T + b.double(), x.double().abs() @ w.double().abs().T + b.double().abs()
    tol = 2.0 ** -24 * (K + 3) * size
    out = torch.full((T + 1, N), 7.0, dtype=dtype, device="cuda")
    _lib.seq_call("umb_seq_linear", out, x, w, b, T, N, K, 4, code)
    want = full.clamp(min=0).pow(2)
    assert _bounded(out[:T], want, 2 * tol * full.abs() + tol * tol + 2.0 ** -23 * want, UNIT[dtype]) and bool((out[T] == 7.0).all())
    cap = torch.full((T + 1, N), 7.0, device="cuda")
    _lib.seq_call("umb_seq_linear_cap", cap, x, w, b, T, N, K, 2.5, code)
    assert _bounded(cap[:T], 2.5 * torch.tanh(full / 2.5), tol + 2e-6) and bool((cap[T] == 7.0).all())      # a tangent of 2^-22 at most
    half = N // 2
    gate, up, tg, tu = full[:, :half], full[:, half:], tol[:, :half], tol[:, half:]
    for epi in (2, 5, 6):
        act = torch.full((T + 1, half), 7.0, dtype=dtype, device="cuda")
        if epi == 5:
            _lib.seq_call("umb_seq_linear_glu", act, x, w, b, T, N, K, 1.5, 1.7, code)
        else:
            _lib.seq_call("umb_seq_linear", act, x, w, b, T, N, K, epi, code)
        want = _glu(epi, gate, up)
        assert _bounded(act[:T], want, 1.2 * tg * (up.abs() + 1) + (gate.abs() + 0.3) * tu + 2e-6 * (want.abs() + up.abs()), UNIT[dtype]), epi
        assert bool((act[T] == 7.0).all())


# rows in quads: every workgroup size (64 ... 1024 threads, up to four quads a thread where rows are many), a group that ends inside the last
# wave, several groups; small groups of many rows, a wave each
@pytest.mark.parametrize("T", [3, 402])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("W,groups", [(192, 3), (8, 1), (200, 1), (1024, 2), (1200, 1), (3072, 3), (2052, 1), (4096, 1), (4100, 1), (8192, 1)])
def test_norms_in_quads(dtype, W, groups, T):
    from umbrella_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(W + groups)
    eps, code = 1e-5, _lib.seq_dtype_code(dtype)
    x, y, y2 = (torch.randn(T, W, generator=g, device="cuda") * s for s in (3.0, 50.0, 0.2))
    w1, w2, w3, w4 = ((1 + 0.2 * torch.randn(W, generator=g, device="cuda")).to(dtype) for _ in range(4))

    def norm(v, w, n=groups):
        v = v.double().view(T, n, -1)
        return (v / (v.pow(2).mean(-1, keepdim=True) + eps).sqrt()).view(T, W) * w.double()
    unit = {torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -22}[dtype]

    def close(got, want, u=2.0 ** -21):              # fp32: a handful of roundings of 2^-24, the sum of squares W of them at most (averaged)
        return bool(((got.double() - want).abs() <= (u + 2.0 ** -20) * want.abs() + 2.0 ** -20).all())
    out, h = torch.empty(T, W, device="cuda"), torch.full((T + 1, W), 7.0, dtype=dtype, device="cuda")
    _lib.seq_call("umb_seq_group_norm", out, h, x, None, w1, T, W, groups, eps, code)
    assert close(out, norm(x, w1)) and close(h[:T], norm(x, w1), unit) and bool((h[T] == 7.0).all())
    xd = x.clone()
    _lib.seq_call("umb_seq_resid_norm", xd, h, y, w1, w2, T, W, groups, eps, code)
    new = x.double() + norm(y, w1)
    assert close(xd, new) and close(h[:T], norm(new, w2), unit + 2.0 ** -18) and bool((h[T] == 7.0).all())
    table = torch.randn(11, W, generator=g, device="cuda").to(dtype)
    ids = torch.tensor([4, 99, -1] * (T // 3), dtype=torch.int32, device="cuda")
    _lib.seq_call("umb_seq_embed_norm", xd, h, table, ids, 1.5, w2, T, W, 11, groups, eps, code)
    rows = table.double()[[4, 10, 0] * (T // 3)] * 1.5
    assert close(xd, rows) and close(h[:T], norm(rows, w2), unit)
    xd = x.clone()
    _lib.seq_call("umb_seq_pair_resid_norm", xd, h, y, y2, w1, w2, 0.5, w3, w4, T, W, eps, code)
    pair = 0.5 * (norm(y, w1, 1) + norm(y2, w2, 1))
    new = x.double() + norm(pair, w3, 1)
    assert close(xd, new, 2.0 ** -19) and close(h[:T], norm(new, w4, 1), unit + 2.0 ** -18)
    xd = x.clone()
    _lib.seq_call("umb_hc_seam", xd, h, y, None, None, 0.5, None, w1, 1.0, T, W, 1, eps, code)
    new = x.double() + 0.5 * y.double()
    assert close(xd, new) and close(h[:T], norm(new, 1.0 + w1.double(), 1), unit + 2.0 ** -18)
    _lib.seq_call("umb_hc_embed", xd, h, table, ids, 1.5, None, w1, 1.0, T, W, 11, 1, eps, code)
    assert close(xd, rows) and close(h[:T], norm(rows, 1.0 + w1.double(), 1), unit)


@pytest.mark.parametrize("W", [1024, 4096, 8192])
def test_scale_of_a_normed_row(W):
    """the error all elements of a row share: a tree of sums, a quotient, a root and a reciprocal"""
    from umbrella_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(W)
    T = 4000
    x, w, h = 3 * torch.randn(T, W, generator=g, device="cuda"), torch.ones(W, device="cuda"), torch.empty(T, W, device="cuda")
    for lo, n in [(200 * i, 200) for i in range(15)] + [(3000, 1000)]:          # launches of few rows and of many
        _lib.seq_call("umb_seq_group_norm", h[lo:], None, x[lo:], None, w, n, W, 1, 1e-6, _lib.seq_dtype_code(torch.float32))
    v = x.double()
    want = v / (v.pow(2).mean(-1, keepdim=True) + 1e-6).sqrt()
    err = (h.double() * want).sum(-1) / want.pow(2).sum(-1) - 1
    # three roundings of up to 2^-24 (0.35 each in the mean) and half the sum's own: 0.70 with a tree of sums, 0.80 with 16 in a row; over 4000
    # rows the mean is known to 1 %
    assert float(err.pow(2).mean().sqrt()) <= 0.75 * 2.0 ** -24


# the chunked recurrence with a decay per channel: one chunk and a token, ragged stretches (one shorter than a block), a carried state, weak and
# strong decays (a channel forgets within a token), sizes up to the LDS limit
@pytest.mark.parametrize("H,D,Dv,lens,strong", [(2, 16, 16, [65], False), (3, 48, 80, [64, 5, 130], False), (2, 128, 256, [200, 1], False),
                                                (2, 128, 64, [70, 129], True), (1, 112, 32, [333], True)])
def test_gla_chunks(H, D, Dv, lens, strong):
    from umbrella_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(D + Dv)
    T, B, HD = sum(lens), len(lens), H * D
    ld = 2 * HD + H * Dv + 8
    proj = torch.randn(T, ld, generator=g, device="cuda")
    la = -torch.rand(T, HD, generator=g, device="cuda") * (0.2 if not strong else 1.0) * torch.where(
        torch.rand(HD, generator=g, device="cuda") < (0.5 if strong else 0.0), 60.0, 1.0)
    state = torch.randn(B + 1, H, D, Dv, generator=g, device="cuda")
    pos0 = [0 if b % 2 else 7 for b in range(B)]
    row0 = [sum(lens[:b]) for b in range(B)]
    slots = [B - b for b in range(B)]
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")                            # noqa: E731
    want_o, want_s, size = torch.zeros(T, H, Dv, dtype=torch.float64, device="cuda"), state.double(), torch.zeros(T, H, Dv, dtype=torch.float64, device="cuda")
    q, k, v = (proj[:, c:c + n].double() for c, n in ((0, HD), (HD, HD), (2 * HD, H * Dv)))
    for b in range(B):
        S = want_s[slots[b]] * (0.0 if pos0[b] == 0 else 1.0)
        A = S.abs()
        for t in range(row0[b], row0[b] + lens[b]):
            a = la[t].double().exp().view(H, D, 1)
            add = k[t].view(H, D, 1) * v[t].view(H, 1, Dv)
            S, A = a * S + add, a * A + add.abs()
            want_o[t], size[t] = (S * q[t].view(H, D, 1)).sum(1), (A * q[t].abs().view(H, D, 1)).sum(1)
        want_s[slots[b]] = S
    need = _lib.load_seq().umb_gla_scan_chunked_floats(T, B, H, D, Dv)
    scratch = torch.full((need + 64,), float("nan"), device="cuda")
    o, st = torch.full((T + 1, H * Dv), 7.0, device="cuda"), state.clone()
    _lib.seq_call("umb_gla_scan_chunked", o, st, proj, ld, la, i32(slots), i32(row0), i32(pos0), i32(lens), T, B, max(lens), H, D, Dv, 0.5,
                  scratch, need)
    # fp32 sums of at most D + 64 products in two stages, every weight an exponential good to 2^-21: far inside 2^-17 of the sum of sizes
    assert ((o[:T].view(T, H, Dv).double() - 0.5 * want_o).abs() <= 2.0 ** -17 * 0.5 * size + 1e-30).all() and bool((o[T] == 7.0).all())
    assert ((st[slots].double() - want_s[slots]).abs() <= 2.0 ** -17 * (want_s[slots].abs().amax() + 1)).all()
    assert torch.equal(st[0], state[0]) and bool(torch.isnan(scratch[need:]).all())


@pytest.mark.parametrize("decay", [0.01, 1.0, 4.0])
@pytest.mark.parametrize("u", [0, 3])
def test_gla_chunks_weigh_as_well_as_token_by_token(decay, u):
    """single weights e^(sum of log decays) inside a block, read out by values of one: relative, however small the weight"""
    from umbrella_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(int(decay * 100) + u)
    D, Dv, T = 16, 16, 64
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")                            # noqa: E731
    need = _lib.load_seq().umb_gla_scan_chunked_floats(T, 1, 1, D, Dv)
    proj, scratch = torch.zeros(T, 2 * D + Dv, device="cuda"), torch.empty(need, device="cuda")
    proj[:, 0], proj[:, D] = 1.0, 1.0
    own = torch.arange(16 * u, 16 * u + 16, device="cuda")
    proj[own, 2 * D + torch.arange(16, device="cuda")] = 1.0
    la = -2 * decay * torch.rand(T, D, generator=g, device="cuda")
    o, st = torch.empty(T, Dv, device="cuda"), torch.zeros(1, 1, D, Dv, device="cuda")
    _lib.seq_call("umb_gla_scan_chunked", o, st, proj, 2 * D + Dv, la, i32([0]), i32([0]), i32([0]), i32([T]), T, 1, T, 1, D, Dv, 1.0, scratch, need)
    c = la[:, 0].double().cumsum(0)[own]
    want = (c[:, None] - c[None]).exp().tril()
    see = want > 2.0 ** -120
    # the exponential unit's last place (2^-23), the exponent's rest to first order (2^-26) and one rounding behind it
    assert float(((o[own].double() - want).abs() / want.clamp(min=1e-300))[see].max()) <= 4 * 2.0 ** -24
    assert bool((o[own][~see].abs() < 2.0 ** -119).all())


@pytest.mark.parametrize("T,at", [(200, 70), (200, 64), (200, 135), (197, 196), (130, 0)])
@pytest.mark.parametrize("kind", ["inf", "nan", "forget"])
def test_gla_chunks_stay_causal_for_values_that_are_not_finite(kind, T, at):
    """an infinite or NaN value spoils its own token and later ones, as token by token; a log decay of -inf is a decay of zero"""
    from umbrella_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(T + at)
    H, D, Dv = 2, 32, 80
    HD, ld = H * D, 2 * H * D + H * Dv + 8
    proj, la = torch.randn(T, ld, generator=g, device="cuda"), -0.2 * torch.rand(T, HD, generator=g, device="cuda")
    state = torch.randn(1, H, D, Dv, generator=g, device="cuda")
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")                            # noqa: E731
    need = _lib.load_seq().umb_gla_scan_chunked_floats(T, 1, H, D, Dv)
    scratch = torch.empty(need, device="cuda")

    def chunked(p, log_decay):
        o, st = torch.empty(T, H * Dv, device="cuda"), state.clone()
        _lib.seq_call("umb_gla_scan_chunked", o, st, p, ld, log_decay, i32([0]), i32([0]), i32([3]), i32([T]), T, 1, T, H, D, Dv, 0.5, scratch, need)
        return o, st
    o0, _ = chunked(proj, la)
    if kind == "forget":
        la[at, ::3] = float("-inf")
        la[min(at + 1, T - 1), 1::3] = float("-inf")
    else:
        proj[at, 2 * HD + 5] = float(kind)
        proj[at, 2 * HD + Dv + 7] = -float(kind)
    o1, s1 = chunked(proj, la)
    o2, s2 = torch.empty(T, H * Dv, device="cuda"), state.clone()
    _lib.seq_call("umb_gla_scan", o2, s2, proj, ld, la.exp(), i32([0]), i32([0]), i32([3]), i32([T]), 1, H, D, Dv, 0.5)
    assert torch.equal(o1.isfinite(), o2.isfinite()) and torch.equal(s1.isfinite(), s2.isfinite())
    assert bool(o1.isfinite().all()) == (kind == "forget")
    fin, size = o2.isfinite(), float(o2[o2.isfinite()].abs().max())
    # sums of a few hundred products in another order: 2^-24 times their number at most, of the largest output
    assert float((o1 - o2)[fin].abs().max()) <= 2.0 ** -14 * size and float((s1 - s2)[s2.isfinite()].abs().max()) <= 2.0 ** -14 * float(state.abs().max() + size)
    if kind != "forget":
        assert torch.equal(o1[:at // 16 * 16], o0[:at // 16 * 16])               # blocks in front are what they were


@pytest.mark.parametrize("H,D,Dv,per_head,groups", [(2, 16, 8, 0, 2), (4, 40, 60, 1, 2), (1, 128, 256, 0, 1), (2, 130, 64, 0, 2), (2, 256, 4, 1, 1)])
def test_single_token_recurrence_follows_the_scan(H, D, Dv, per_head, groups):
    from umbrella_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(D + Dv)
    T = 3
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")                                     # noqa: E731
    q, k, v = r(T, groups * D), r(T, groups * D + 4), r(T, H * Dv + 4)
    alpha = torch.rand(T, H if per_head else H * D, generator=g, device="cuda")
    state, out = r(T + 2, H, D, Dv), []
    pos, slot, row, one = (torch.tensor(x, dtype=torch.int32, device="cuda") for x in ([5, 0, 9], [3, 0, 1], [0, 1, 2], [1, 1, 1]))
    for step in (True, False):
        st, o = state.clone(), torch.full((T + 1, H * Dv), 7.0, device="cuda")
        args = (o, st, q, groups * D, k, groups * D + 4, v, H * Dv + 4, alpha, per_head, groups)
        if step:
            _lib.seq_call("umb_lin_step", *args, pos, slot, T, H, D, Dv, 0.25)
        else:
            _lib.seq_call("umb_lin_scan", *args, slot, row, pos, one, T, H, D, Dv, 0.25)
        out.append((o, st))
    # the sums run in one order; which product of a * S + k * v joins the other unrounded is the compiler's choice
    bound = 2.0 ** -23 * (state[slot.long()].abs() + k.abs().amax() * v.abs().amax())
    assert ((out[0][1] - out[1][1])[slot.long()].abs() <= bound).all() and torch.equal(out[0][1][[2, 4]], state[[2, 4]])
    assert ((out[0][0] - out[1][0]).abs() <= D * q.abs().amax() * bound.amax()).all() and bool((out[0][0][T] == 7.0).all())


@pytest.mark.parametrize("T,C,prefix,end,wide", [(1, 1, 1, 1, True), (1, 65, 65, 65, False), (13, 77, 64, 77, True), (31, 200, 0, 131, True), (40, 640, 600, 640, False),
                                                 (257, 957, 700, 957, True), (5, 64, 63, 64, True)])
def test_boolean_mask_scan_and_bits(T, C, prefix, end, wide):
    from umbrella_amd import _lib
    from umbrella_amd.models.llama import pack_mask_bits
    g = torch.Generator().manual_seed(T + C)
    mask = torch.zeros(T, C + 3, dtype=torch.bool)
    mask[:, :prefix] = True
    mask[:, prefix:end] = torch.rand(T, end - prefix, generator=g) < 0.4
    if end > prefix:
        mask[0, prefix], mask[T - 1, end - 1] = False, True
        if T == 1 and end - prefix == 1:
            mask[0, prefix] = True
    m = mask.cuda()[:, :C]                                                   # rows further apart than their columns
    kind = torch.int64 if wide else torch.int32
    ids, pos, slots = (torch.randint(0, 5000, (T,), generator=g).to(kind).cuda() for _ in range(3))
    nb = (C + 63) // 64
    out = torch.full((2 * nb + 2,), -7, dtype=torch.int32, device="cuda")
    _lib.call("umb_mask_scan", out, m, m.stride(0), T, C, slots, int(wide))
    got = out.tolist()
    cols = mask[:, :C].all(0)
    first = int((~cols).nonzero()[0]) if not bool(cols.all()) else C
    assert min(got[0:2 * nb:2]) == first and got[2 * nb] == int(slots.max()) and got[2 * nb + 1] == -7
    assert max(got[1:2 * nb:2]) == int(mask[:, :C].any(0).nonzero()[-1]) + 1
    pre = max(min(first, C - 1), 0)
    W = (C - pre + 63) // 64
    bits, idx = torch.empty(T + 1, W, dtype=torch.int64, device="cuda").fill_(-7), torch.empty(3 * T + 2, dtype=torch.int32, device="cuda").fill_(-7)
    _lib.call("umb_mask_pack", bits, W, idx, m, m.stride(0), T, C, pre, ids, int(wide), pos, int(wide), slots, int(wide))
    assert torch.equal(bits[:T].cpu(), pack_mask_bits(mask[:, pre:C])) and bool((bits[T] == -7).all())
    assert torch.equal(idx[:3 * T], torch.cat([ids, pos, slots]).int()) and idx[3 * T:].tolist() == [pre, -7]


def test_a_row_that_attends_everything_attends_nothing_else():
    """a mask of ones has no column left for bit rows: the row must not see the slot behind its own, whatever that holds"""
    from umbrella_amd.models.config import LlamaCfg
    from umbrella_amd.models.llama import Llama
    from umbrella_amd.models.synthetic import synth_state_small
    cfg = LlamaCfg(vocab_size=128, hidden_size=256, intermediate_size=256, num_hidden_layers=2, num_attention_heads=4, num_key_value_heads=2,
                   head_dim=64, eos_token_id=[], name="tiny")
    m = Llama("tiny", max_length=128, device="cuda:0", dtype=torch.float16, state_dict=synth_state_small(cfg, 1), config=cfg)
    m.alloc()
    ids = torch.arange(20, 29)[None]
    see = torch.tril(torch.ones(9, 9, dtype=torch.bool))
    m.inference(ids[:, :8], torch.arange(8)[None], see[:8, :8], torch.arange(8))
    m.kv_cache.set_rows([9], torch.full((2, 2, 1, 64), 30.0, device="cuda"), torch.full((2, 2, 1, 64), 50.0, device="cuda"))
    one = m.inference(ids[:, 8:], torch.tensor([[8]]), see[8:], torch.tensor([8]))
    m.clear()
    both = m.inference(ids, torch.arange(9)[None], see, torch.arange(9))
    assert (one[0, 0] - both[0, 8]).abs().max() < 2e-2 * both.abs().max()


def test_masks_that_are_accepted_in_any_layout():
    """one row of any stride, rows and columns to spare, no column: the logits are those of the same mask laid out plainly"""
    from umbrella_amd.models.config import LlamaCfg
    from umbrella_amd.models.llama import Llama
    from umbrella_amd.models.synthetic import synth_state_small
    cfg = LlamaCfg(vocab_size=128, hidden_size=256, intermediate_size=256, num_hidden_layers=2, num_attention_heads=4, num_key_value_heads=2,
                   head_dim=64, eos_token_id=[], name="tiny")
    m = Llama("tiny", max_length=128, device="cuda:0", dtype=torch.float16, state_dict=synth_state_small(cfg, 1), config=cfg)
    m.alloc()
    ids, at = torch.arange(20, 29)[None], torch.arange(9)
    see = torch.tril(torch.ones(9, 9, dtype=torch.bool)).cuda()
    m.inference(ids, at[None], see, at)

    def row(mask, pos=torch.tensor([[8]]), slots=torch.tensor([8])):
        return m.inference(ids[:, 8:], pos, mask, slots).clone()
    some = torch.tensor([1, 0, 1, 1, 0, 1, 1, 0, 1], dtype=torch.bool, device="cuda")
    for one in (torch.ones(9, dtype=torch.bool, device="cuda"), some):
        want = row(one.clone()[None])
        assert torch.equal(row(one[:, None].clone().T), want)                            # strides (1, 1)
        assert torch.equal(row(torch.stack([one, ~one], 1)[:, :1].T), want)              # a column of a wider array
    want = row(torch.ones(1, 9, dtype=torch.bool, device="cuda"))
    assert torch.equal(row(torch.ones(1, 1, dtype=torch.bool, device="cuda").expand(1, 9)), want)     # strides (0, 0)
    full = m.inference(ids, at[None], see, at).clone()
    m.kv_cache.kv_offset = 9
    spare = torch.cat([see, torch.zeros(2, 9, dtype=torch.bool, device="cuda")])
    got = m.inference(ids, torch.arange(11)[None], spare, torch.arange(12))              # rows, positions and slots to spare
    assert torch.allclose(got, full, rtol=0, atol=2e-3 * float(full.abs().max())) and m.kv_cache.kv_offset == 12
    first = m.inference(ids[:, :1], at[None, :1], see[:1, :1], at[:1])
    assert torch.equal(m.inference(ids[:, :1], at[None, :1], see[:1, :0], at[:1]), first)
    with pytest.raises(AssertionError):
        m.inference(ids, at[None], see[:8], at)


def _decode_store(lens, G, DK, E, pool, dtype, page, seed):
    from umbrella_amd.attn.cache import PagedSeqCache
    c = PagedSeqCache([(G, DK, pool, E)], [], sum(lens), len(lens), "cuda", dtype, page=page)
    g = torch.Generator(device="cuda").manual_seed(seed)
    for z in ("k", "v", "kp", "vp"):
        if c.kv[0][z] is not None:
            c.kv[0][z].copy_(torch.randn(c.kv[0][z].shape, generator=g, device="cuda"))
    entries = []
    for b, n in enumerate(lens):
        c.open(b)
        c.extend(b, n, entries)
    c.write_pages(entries)
    pos = torch.tensor([n - 1 for n in lens], dtype=torch.int32, device="cuda")
    return c, pos, torch.tensor([c.slot(b) for b in range(len(lens))], dtype=torch.int32, device="cuda"), g


SHORT, LONG = [1, 15, 16, 17, 40, 65, 256, 257], [1024, 1025, 2049, 3]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,G,D,E,maps,lens,window,chunk,keep,extra", [
    (8, 2, 64, 64, 1, SHORT, 2 ** 30, 0, 0, False), (4, 2, 128, 128, 1, LONG, 2 ** 30, 0, 0, True), (8, 2, 96, 128, 2, SHORT, 100, 0, 0, True),
    (4, 1, 128, 256, 2, LONG, 2 ** 30, 0, 0, False), (3, 1, 160, 64, 1, SHORT + LONG, 30, 0, 5, True), (6, 3, 32, 256, 1, SHORT, 300, 50, 7, True),
    (4, 1, 64, 64, 1, [20 + 3 * i for i in range(70)], 64, 0, 3, True), (32, 8, 64, 128, 1, [33] * 140, 512, 0, 0, False)])
def test_single_token_attention(dtype, H, G, D, E, maps, lens, window, chunk, keep, extra):
    from umbrella_amd import _lib
    code = _lib.seq_dtype_code(dtype)
    c, pos, slot, g = _decode_store(lens, G, maps * D, E, 0, dtype, 16, H + D + E)
    T, nd = len(lens), 40
    q = torch.randn(T, H, maps, D, generator=g, device="cuda")
    gate = torch.randn(T, H * E, generator=g, device="cuda") if extra else None
    sink = torch.randn(H, generator=g, device="cuda") if extra else None
    bias = torch.randn(H, nd, generator=g, device="cuda") if extra else None
    if extra:
        bias[0, nd - 1] = float("-inf")                   # whole rounds of one head see nothing
    cap, lam, eps, scale = (6.0 if extra else 0.0), 0.3, 1e-3, D ** -0.5
    form = _lib.UmbAttnForm(maps, chunk, sink.data_ptr() if extra else None, lam, eps, keep, int(extra))
    for split in (False, True):
        out = torch.full((T, H * E + 8), 3.0, dtype=dtype, device="cuda")
        scratch = torch.empty(T * H * maps * 16 * (E + 2), device="cuda") if split else None
        _lib.seq_call("umb_attn_attend", out, H * E + 8, q, c.struct(0), gate, H * E if extra else 0, 0 if extra else -1, bias, nd if extra else 0, pos,
                      slot, T, H, G, D, E, window, scale, 1.25, cap, form, scratch, scratch.numel() if split else 0, code)
        assert bool((out[:, H * E:] == 3.0).all())
        for t, n in enumerate(lens):
            i = n - 1
            j = torch.arange(n)
            see = i - j < window
            if chunk:
                see &= j // chunk == i // chunk
            j = j[see | (j < keep)]
            k, v = (z.double() for z in c.token_rows(0, t, j))                       # [m, G, maps D], [m, G, E]
            k = k.view(len(j), G, maps, D).repeat_interleave(H // G, 1)
            s = (q[t].double()[None] * k).sum(-1) * scale                            # [m, H, maps]
            if cap:
                s = cap * torch.tanh(s / cap)
            if extra:
                s = s + bias.double()[:, torch.clamp(i - j, max=nd - 1).cuda()].T[..., None]
                p = torch.softmax(torch.cat([s, sink.double()[None, :, None].expand(1, H, maps)]), 0)[:-1]
            else:
                p = torch.softmax(s, 0)
            o = (p[..., None] * v.repeat_interleave(H // G, 1)[:, :, None]).sum(0)   # [H, maps, E]
            if maps == 2:
                o = o[:, 0] - lam * o[:, 1]
                o = o / torch.sqrt(o.pow(2).mean(-1, keepdim=True) + eps)
            else:
                o = o[:, 0]
            o = (1.25 * o).reshape(-1)
            if extra:
                o = o * torch.sigmoid(gate[t].double())
            got = out[t, :H * E].double()
            # storage rounding of the result; scores of up to 7 in fp32 over at most 2049 keys, then a quotient: 1e-4 of the largest output
            tol = 2.0 ** (-8 if dtype == torch.bfloat16 else -11) * o.abs() + 1e-4 * o.abs().max() + 1e-6
            assert bool(((got - o).abs() <= tol).all()), (t, n, split, float((got - o).abs().max()))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,G,D,lens,window,pool", [(8, 2, 64, SHORT, 2 ** 20, 16), (4, 2, 128, SHORT + LONG, 20, 7), (2, 2, 256, LONG, 513, 3),
                                                    (32, 8, 128, [90 + i for i in range(40)], 64, 16), (6, 3, 64, [33] * 400, 16, 1)])
def test_single_token_pooled_attention(dtype, H, G, D, lens, window, pool):
    from umbrella_amd import _lib
    code = _lib.seq_dtype_code(dtype)
    c, pos, slot, g = _decode_store(lens, G, D, D, pool, dtype, 32, H + D + pool)
    T = len(lens)
    q, gate = torch.randn(T, H, D, generator=g, device="cuda"), torch.randn(T, H, generator=g, device="cuda")
    pb = torch.randn(H, generator=g, device="cuda").to(dtype)
    out = torch.empty(T, H * D, dtype=dtype, device="cuda")
    _lib.seq_call("umb_pwa_attend", out, q, c.struct(0), gate, H, 0, pb, pos, slot, T, H, G, D, window, pool, D ** -0.5, code)
    for t, n in list(enumerate(lens))[:50]:
        i = n - 1
        j = torch.arange(max(0, i - window + 1), n)
        k, v = (z.double() for z in c.token_rows(0, t, j))
        nb = max(i - window + 1, 0) // pool
        if nb:
            kp, vp = (z.double() for z in c.pooled_rows(0, t, torch.arange(nb)))
            k, v = torch.cat([kp, k]), torch.cat([vp, v])
        k, v = k.repeat_interleave(H // G, 1), v.repeat_interleave(H // G, 1)
        w = torch.sigmoid((q[t].double()[None] * k).sum(-1) * D ** -0.5 + pb.double())
        o = ((w[..., None] * v).sum(0) * torch.sigmoid(gate[t].double())[:, None]).reshape(-1)
        scale = (w[..., None] * v.abs()).sum(0).max()
        # storage rounding; fp32 sums of up to 2049 terms of that total size (2^-24 each, pairwise over waves and row groups)
        tol = 2.0 ** (-8 if dtype == torch.bfloat16 else -11) * o.abs() + 2e-6 * scale + 1e-6
        assert bool(((out[t].double() - o).abs() <= tol).all()), (t, n, float((out[t].double() - o).abs().max()))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D,pool,page", [(24, 7, 64), (128, 16, 64), (200, 65, 64), (300, 130, 32), (64, 1, 8)])
def test_pooled_blocks(dtype, D, pool, page):
    from umbrella_amd import _lib
    c, pos, slot, g = _decode_store([300, 131, 1], 2, D, D, pool, dtype, page, D + pool)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")                                    # noqa: E731
    p0, n = [64, 0, 0], [236, 131, 1]
    want = {}
    for b in range(3):
        for blk in range((p0[b] + n[b]) // pool):
            rows = c.token_rows(0, b, torch.arange(blk * pool, (blk + 1) * pool))
            new = p0[b] <= blk * pool + pool - 1
            want[b, blk] = [z.float() for z in rows] if new else [z[0].clone() for z in c.pooled_rows(0, b, [blk])]
    _lib.seq_call("umb_pwa_pool", c.struct(0), slot, i32(p0), i32(n), 3, max(n), 2, D, pool, _lib.seq_dtype_code(dtype))
    for (b, blk), rows in want.items():
        for z, r in zip(c.pooled_rows(0, b, [blk]), rows):
            if r.dim() == 3:                              # added in position order in fp32, then times the rounded 1 / pool
                s = torch.zeros_like(r[0])
                for x in r:
                    s = s + x
                r = s * torch.tensor(1.0 / pool, dtype=torch.float32, device="cuda")
            assert torch.equal(z[0], r), (b, blk)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,N,S", [(257, 1024, 3), (300, 36, 1), (259, 2052, 2), (513, 4096, 5), (1024, 4096, 1), (270, 8192, 8), (258, 5120, 4)])
def test_split_reduce_of_many_rows_is_that_of_few(dtype, T, N, S):
    """h bit for bit what the launches of up to 256 rows give; the norm's sum of squares runs in another order (fp32): one rounding step"""
    from umbrella_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(T + N)
    code, eps = _lib.dtype_code(dtype), torch.finfo(dtype).eps
    part = torch.randn(S, T, N, generator=g, device="cuda")
    res, w = torch.randn(T, N, generator=g, device="cuda").to(dtype), torch.randn(N, generator=g, device="cuda").to(dtype)
    for residual, normed in ((res, True), (None, True), (res, False)):
        h, x = torch.full((T + 1, N), 3.0, dtype=dtype, device="cuda"), torch.full((T + 1, N), 3.0, dtype=dtype, device="cuda")
        _lib.call("umb_reduce_residual_norm", part, S, T, N, residual, h, x if normed else None, w, 1e-5, code)
        for lo in range(0, T, 200):
            n = min(200, T - lo)
            h1, x1 = torch.empty(n, N, dtype=dtype, device="cuda"), torch.empty(n, N, dtype=dtype, device="cuda")
            _lib.call("umb_reduce_residual_norm", part[:, lo:lo + n].contiguous(), S, n, N, None if residual is None else residual[lo:lo + n], h1,
                      x1 if normed else None, w, 1e-5, code)
            assert torch.equal(h[lo:lo + n], h1)
            if normed:
                assert bool(((x[lo:lo + n].float() - x1.float()).abs() <= eps * x1.float().abs() + 1e-7).all())
        assert bool((h[T] == 3.0).all()) and bool((x[T] == 3.0).all()) and (normed or bool((x == 3.0).all()))
    if N % 32 == 0:
        tt = (T + 15) // 16
        h2, x2 = torch.empty(T, N, dtype=dtype, device="cuda"), torch.zeros(16 * tt * N, dtype=dtype, device="cuda")
        _lib.call("umb_reduce_residual_norm_fm", part, S, T, N, res, h2, x2, w, 1e-5, tt, code)
        _lib.call("umb_reduce_residual_norm", part, S, T, N, res, h, x, w, 1e-5, code)
        fm = x2.view(N // 32, tt, 4, 16, 8).permute(1, 3, 0, 2, 4).reshape(16 * tt, N)[:T]
        assert torch.equal(fm, x[:T]) and torch.equal(h2, h[:T])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,Hq,Hkv,D,S,paired", [(257, 4, 2, 64, 2, 1), (400, 4, 1, 96, 3, 1), (263, 3, 1, 32, 1, 0), (514, 2, 2, 128, 4, 0), (1024, 5, 1, 256, 8, 1),
    # enough columns and few enough splits for a workgroup per 256 columns of 16 tokens
    (263, 20, 6, 64, 2, 1), (400, 8, 4, 96, 3, 1), (259, 48, 2, 32, 1, 0), (514, 4, 2, 128, 2, 0), (700, 8, 1, 64, 4, 1), (1023, 5, 1, 256, 3, 1), (258, 5, 1, 256, 1, 0)])
def test_split_reduce_and_rotation_of_many_tokens_is_that_of_few(dtype, T, Hq, Hkv, D, S, paired):
    from umbrella_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(T + D)
    N, L, code = (Hq + 2 * Hkv) * D, 1536, _lib.dtype_code(dtype)
    part = torch.randn(S, T, N, generator=g, device="cuda")
    cos, sin = torch.randn(L, D, generator=g, device="cuda").to(dtype), torch.randn(L, D, generator=g, device="cuda").to(dtype)
    pos = torch.randint(0, L, (T,), generator=g, device="cuda", dtype=torch.int32)
    bias = torch.randn(N, generator=g, device="cuda").to(dtype)
    ssq = torch.rand(T, 7, generator=g, device="cuda") + 0.5
    runs = {"in a row": torch.arange(T, device="cuda") + 100, "off the grid": torch.arange(T, device="cuda") + 101,
            "anywhere": torch.randperm(L, generator=g, device="cuda")[:T]}
    for name, slot in runs.items():
        slot = slot.to(torch.int32)
        for b, q2 in ((None, None), (bias, None), (None, ssq), (bias, ssq)):
            outs = []
            for step in (T, 200):
                q = torch.full((T + 1, Hq * D), 3.0, dtype=dtype, device="cuda")
                kc, vt = torch.full((Hkv, L * D), 3.0, dtype=dtype, device="cuda"), torch.full((Hkv, D * (L + 32)), 3.0, dtype=dtype, device="cuda")
                for lo in range(0, T, step):
                    n = min(step, T - lo)
                    _lib.call("umb_reduce_qkv_rope2", part[:, lo:lo + n].contiguous(), S, n, Hq, Hkv, D, L, pos[lo:lo + n], slot[lo:lo + n], cos, sin,
                              q[lo:lo + n], kc, vt, paired, b, None if q2 is None else q2[lo:lo + n], 0 if q2 is None else 5, 0 if q2 is None else 7,
                              0.0 if q2 is None else 40.0, 1e-5, code)
                outs.append((q, kc, vt))
            for x, y in zip(*outs):
                if b is None or q2 is None:
                    assert torch.equal(x, y), (name, b is not None)
                else:       # x / rms + bias may be one fp32 rounding or two: then each of the rotation's two products may round the other way
                    eps = torch.finfo(dtype).eps
                    assert bool(((x.float() - y.float()).abs() <= 4 * eps * y.float().abs().max()).all()) and (x != y).float().mean() < 1e-2


def _stretches(lens, news):
    """rows of a step that brings the last news[b] of lens[b] positions of every sequence"""
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")                                    # noqa: E731
    row0 = [sum(news[:b]) for b in range(len(news))]
    return i32(row0), i32([n - k for n, k in zip(lens, news)]), i32(news), sum(news)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,G,D,E,maps,window,chunk,keep,extra", [
    (8, 2, 64, 64, 1, 2 ** 30, 0, 0, False), (6, 1, 64, 64, 1, 70, 0, 5, True), (4, 1, 128, 128, 1, 90, 0, 40, True), (12, 2, 128, 128, 1, 2 ** 30, 64, 0, False),
    (4, 2, 64, 128, 2, 2 ** 30, 50, 0, False), (2, 1, 128, 256, 2, 100, 0, 3, True), (3, 1, 72, 48, 1, 60, 0, 0, True),
    # every count of 32-feature steps and 16-column tiles, whole and not, each direction first to overflow its size; more heads than a workgroup has waves
    (8, 1, 96, 96, 1, 2 ** 30, 0, 0, False), (5, 1, 80, 32, 1, 50, 0, 2, True), (2, 2, 16, 112, 1, 70, 0, 0, False), (6, 1, 104, 128, 1, 2 ** 30, 30, 0, True),
    (2, 1, 192, 192, 1, 40, 0, 0, True), (3, 1, 136, 48, 1, 2 ** 30, 0, 0, False), (1, 1, 256, 256, 1, 2 ** 30, 0, 0, True), (2, 1, 24, 208, 1, 60, 0, 0, False),
    (2, 1, 40, 48, 2, 2 ** 30, 0, 0, True), (2, 2, 128, 128, 2, 60, 0, 0, False), (1, 1, 72, 144, 2, 2 ** 30, 0, 0, True), (2, 1, 160, 160, 2, 2 ** 30, 40, 0, False),
    (1, 1, 256, 256, 2, 80, 0, 5, True)])
def test_prompt_attention(dtype, H, G, D, E, maps, window, chunk, keep, extra):
    from umbrella_amd import _lib
    code = _lib.seq_dtype_code(dtype)
    lens, news = [16, 33, 250, 95], [16, 17, 250, 30]
    c, _, slot, g = _decode_store(lens, G, maps * D, E, 0, dtype, 16, H + D + E)
    row0, pos0, cnt, T = _stretches(lens, news)
    nd = 40
    q = torch.randn(T, H, maps, D, generator=g, device="cuda")
    gate = torch.randn(T, H, generator=g, device="cuda") if extra else None
    sink = torch.randn(H, generator=g, device="cuda") if extra else None
    bias = torch.randn(H, nd, generator=g, device="cuda") if extra else None
    cap, lam, eps, scale = (6.0 if extra else 0.0), 0.3, 1e-3, D ** -0.5
    form = _lib.UmbAttnForm(maps, chunk, sink.data_ptr() if extra else None, lam, eps, keep, 0)
    out = torch.full((T + 1, H * E + 8), 3.0, dtype=dtype, device="cuda")
    _lib.seq_call("umb_attn_attend_tiled", out, H * E + 8, q, c.struct(0), gate, H if extra else 0, 0 if extra else -1, bias, nd if extra else 0, slot, row0,
                  pos0, cnt, len(lens), max(news), H, G, D, E, window, scale, 1.25, cap, form, code)
    assert bool((out[:, H * E:] == 3.0).all()) and bool((out[T] == 3.0).all())
    for b, (n, k) in enumerate(zip(lens, news)):
        kk, vv = (z.double() for z in c.token_rows(0, b, torch.arange(n)))
        kk = kk.view(n, G, maps, D).repeat_interleave(H // G, 1)
        vv = vv.repeat_interleave(H // G, 1)
        r0 = int(row0[b])
        i, j = torch.arange(n - k, n, device="cuda")[:, None], torch.arange(n, device="cuda")[None]
        see = i - j < window
        if chunk:
            see &= j // chunk == i // chunk
        see = (see | (j < keep)) & (j <= i)
        s, s_size = (torch.einsum("thmd,jhmd->thmj", x.cpu(), y.cpu()).cuda() * scale for x, y in
                     ((q[r0:r0 + k].double(), kk), (q[r0:r0 + k].double().abs(), kk.abs())))
        if cap:
            s = cap * torch.tanh(s / cap)
        if extra:
            s = s + bias.double()[:, (i - j).clamp(0, nd - 1)].permute(1, 0, 2)[:, :, None]
        s = s.masked_fill(~see[:, None, None], float("-inf"))
        if extra:
            p = torch.softmax(torch.cat([s, sink.double()[None, :, None, None].expand(k, H, maps, 1)], -1), -1)[..., :-1]
        else:
            p = torch.softmax(s, -1)
        # o = sum p v, p a quotient of weights: a score's error counts twice, a weight's split once.  A split keeps 2^-17 (bf16) or 2^-22 (fp16) of
        # its number, an fp32 sum of D products D 2^-24 of their size, base-2 scores within 20 round to 2^-20; fp16 weights next to zero lose 2^-25
        split = 2.0 ** (-17 if dtype == torch.bfloat16 else -22)
        s_err = (split + D * 2.0 ** -24) * s_size.masked_fill(~see[:, None, None], 0.0).amax(-1) + 2.0 ** -20
        rel, lost = 2 * s_err + split + 2.0 ** -20, 0.0 if dtype == torch.bfloat16 else 2.0 ** -25
        o, size = (torch.einsum("thmj,jhe->thme", p.cpu(), v.cpu()).cuda() for v in (vv, vv.abs()))
        gone = lost * torch.einsum("tj,jhe->the", see.double(), vv.abs().contiguous())[:, :, None]
        o_err = rel[..., None] * size + gone
        if maps == 2:
            o, o_err = o[:, :, 0] - lam * o[:, :, 1], o_err[:, :, 0] + lam * o_err[:, :, 1]
            rms = torch.sqrt(o.pow(2).mean(-1, keepdim=True) + eps)
            o = o / rms
            o_err = o_err / rms + o.abs() * torch.sqrt(o_err.pow(2).mean(-1, keepdim=True)) / rms
        else:
            o, o_err = o[:, :, 0], o_err[:, :, 0]
        f = 1.25 * (torch.sigmoid(gate[r0:r0 + k].double())[..., None] if extra else 1.0)
        o, o_err = o * f, o_err * f
        tol = 2.0 ** (-8 if dtype == torch.bfloat16 else -11) * o.abs() + o_err + 2.0 ** -20 * o.abs() + 2.0 ** -25
        err = (out[r0:r0 + k, :H * E].double().view(k, H, E) - o).abs()
        assert bool((err <= tol).all()), (b, float(err.max()))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,G,D,window,pool", [(8, 2, 64, 40, 16), (5, 1, 32, 2 ** 20, 4), (4, 2, 128, 17, 3), (6, 1, 96, 64, 1), (2, 1, 256, 33, 7)])
def test_prompt_pooled_attention(dtype, H, G, D, window, pool):
    from umbrella_amd import _lib
    code = _lib.seq_dtype_code(dtype)
    lens, news = [16, 33, 250, 95], [16, 17, 250, 30]
    c, _, slot, g = _decode_store(lens, G, D, D, pool, dtype, 32, H + D + pool)
    row0, pos0, cnt, T = _stretches(lens, news)
    q, gate = torch.randn(T, H, D, generator=g, device="cuda"), torch.randn(T, H, generator=g, device="cuda")
    pb = torch.randn(H, generator=g, device="cuda").to(dtype)
    out = torch.full((T + 1, H * D), 3.0, dtype=dtype, device="cuda")
    _lib.seq_call("umb_pwa_attend_tiled", out, q, c.struct(0), gate, H, 0, pb, slot, row0, pos0, cnt, len(lens), max(news), H, G, D, window, pool, D ** -0.5,
                  code)
    assert bool((out[T] == 3.0).all())
    for b, (n, k) in enumerate(zip(lens, news)):
        nb = max(n - window, 0) // pool
        kk, vv = (z.double() for z in c.token_rows(0, b, torch.arange(n)))
        if nb:
            kp, vp = (z.double() for z in c.pooled_rows(0, b, torch.arange(nb)))
            kk, vv = torch.cat([kp, kk]), torch.cat([vp, vv])
        kk, vv = kk.repeat_interleave(H // G, 1).cpu(), vv.repeat_interleave(H // G, 1).cpu()
        r0 = int(row0[b])
        i, j = torch.arange(n - k, n)[:, None], torch.arange(n)[None]
        see = torch.cat([torch.arange(nb)[None] * pool + pool - 1 <= i - window, (j <= i) & (i - j < window)], 1)
        s = torch.einsum("thd,jhd->thj", q[r0:r0 + k].double().cpu(), kk) * D ** -0.5
        w = torch.sigmoid(s + pb.double().cpu()[None, :, None]) * see[:, None]
        gt = torch.sigmoid(gate[r0:r0 + k].double().cpu())[..., None]
        o, size = torch.einsum("thj,jhd->thd", w, vv) * gt, (torch.einsum("thj,jhd->thd", w, vv.abs()) * gt).max()
        # storage rounding; queries, pooled rows and weights split to 2^-17 each (bf16), scores of up to 7: 3e-5 of the sum of sizes
        tol = 2.0 ** (-8 if dtype == torch.bfloat16 else -11) * o.abs() + 3e-5 * size + 1e-6
        err = (out[r0:r0 + k].double().cpu().view(k, H, D) - o).abs()
        assert bool((err <= tol).all()), (b, float(err.max()), float(size))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,Dc,R,window", [(9, 512, 64, 70), (16, 256, 32, 2 ** 20), (8, 256, 64, 33), (4, 512, 64, 2 ** 20), (9, 64, 24, 50),
    # every count of feature steps and value tiles, whole and not, either first to overflow its size; few heads and more than eight
    (8, 128, 0, 40), (3, 96, 32, 2 ** 20), (5, 144, 8, 60), (16, 256, 48, 2 ** 20), (6, 272, 0, 50), (7, 384, 64, 2 ** 20), (4, 368, 40, 45), (12, 400, 40, 70),
    (2, 512, 0, 2 ** 20)])
def test_latent_attention_of_prompts_and_of_many_tokens(dtype, H, Dc, R, window):
    from umbrella_amd import _lib
    from umbrella_amd.attn.cache import PagedSeqCache
    code, Dk = _lib.seq_dtype_code(dtype), Dc + R
    g = torch.Generator(device="cuda").manual_seed(H + Dc + R)

    def case(lens, news, tiled):
        c = PagedSeqCache([], [], sum(lens), len(lens), "cuda", dtype, page=16, latent_layers=(Dk,))
        c.latent[0].copy_(torch.randn(c.latent[0].shape, generator=g, device="cuda"))
        for b, n in enumerate(lens):
            c.open(b), c.extend(b, n)
        slot = torch.tensor([c.slot(b) for b in range(len(lens))], dtype=torch.int32, device="cuda")
        row0, pos0, cnt, T = _stretches(lens, news)
        qa, sink = torch.randn(T, H, Dk, generator=g, device="cuda"), torch.randn(H, generator=g, device="cuda").to(dtype)
        out = torch.full((T + 1, H * Dc), 3.0, dtype=dtype, device="cuda")
        scale = Dk ** -0.5
        if tiled:
            _lib.seq_call("umb_lat_attend_tiled", out, qa, c.latent_struct(0), sink, slot, row0, pos0, cnt, len(lens), max(news), H, Dc, R, window, scale, code)
        else:
            pos = torch.tensor([n - 1 for n in lens], dtype=torch.int32, device="cuda")
            _lib.seq_call("umb_lat_attend", out, qa, c.latent_struct(0), sink, pos, slot, T, H, Dc, R, window, scale, code)
        assert bool((out[T] == 3.0).all())
        for b, (n, k) in enumerate(zip(lens, news)):
            r0 = int(row0[b])
            rows = c.latent_rows(0, b, torch.arange(n)).double().cpu()
            i, j = torch.arange(n - k, n)[:, None], torch.arange(n)[None]
            x = qa[r0:r0 + k].to(dtype).double().cpu()                       # queries enter in the storage type
            s = (torch.einsum("thd,jd->thj", x, rows) * scale).masked_fill(~((j <= i) & (i - j < window))[:, None], float("-inf"))
            p = torch.softmax(torch.cat([s, sink.double().cpu()[None, :, None].expand(k, H, 1)], -1), -1)[..., :-1]
            o = torch.einsum("thj,jd->thd", p, rows[:, :Dc])
            # weights and the result are rounded to the storage type, each to half a step of its own size
            u = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
            tol = u * o.abs() + u * torch.einsum("thj,jd->thd", p, rows[:, :Dc].abs()) + 1e-4 * o.abs().max()
            err = (out[r0:r0 + k].double().cpu().view(k, H, Dc) - o).abs()
            assert bool((err <= tol).all()), (b, float(err.max()))
    case([16, 33, 250, 95], [16, 17, 250, 30], True)
    if H > 4:                                              # enough workgroups of eight waves
        case([1100, 60, 1100], [1100, 17, 1090], True) if Dc <= 384 else case([330] * 6, [330] * 6, True)
    case([1 + 3 * i for i in range(50)], [1] * 50, False)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("H,G,D,E,maps,layout,rot,append,norm,mixed", [(8, 2, 64, 64, 1, 0, 64, 1, 1, True), (3, 1, 128, 96, 2, 1, 80, 1, 0, False),
                                                                       (7, 7, 24, 128, 1, 1, 0, 1, 1, True), (30, 2, 100, 40, 1, 0, 50, 0, 1, False)])
def test_many_slots_are_prepared_as_few_are(dtype, H, G, D, E, maps, layout, rot, append, norm, mixed):
    """norm, rotation and append of many (token, head) slots against launches of few: an fp32 sum of squares in another order"""
    from umbrella_amd import _lib
    T, step, code = 2880, 60, _lib.seq_dtype_code(dtype)
    g = torch.Generator(device="cuda").manual_seed(D + E)
    c, _, _, _ = _decode_store([T], G, maps * D, E, 0, dtype, 32, 1)
    d, _, _, _ = _decode_store([T], G, maps * D, E, 0, dtype, 32, 2)
    HQ, GK, GV = maps * H, append * maps * G, append * G
    ld = HQ * D + GK * D + GV * E + 5
    proj, freq = torch.randn(T, ld, generator=g, device="cuda"), torch.rand(64, generator=g, device="cuda")
    wq, wk = (torch.randn(D, generator=g, device="cuda").to(dtype) for _ in range(2))
    pos, slot = torch.arange(T, device="cuda", dtype=torch.int32), torch.zeros(T, device="cuda", dtype=torch.int32)
    firsts = torch.randn(T, G * E, generator=g, device="cuda")
    outs = []
    for store, n in ((c, T), (d, step)):
        q, keep = torch.empty(T, HQ * D, device="cuda"), torch.zeros(T, G * E, device="cuda")
        for lo in range(0, T, n):
            m = _lib.UmbValueMix(firsts[lo:].data_ptr(), keep[lo:].data_ptr(), 0.3, 0.0) if mixed else None
            _lib.seq_call("umb_attn_prep_mix", q[lo:], store.struct(0), proj[lo:lo + n], ld, append, wq if norm else None, wk if norm else None, norm, norm,
                          pos[lo:lo + n], slot[lo:lo + n], freq if rot else None, rot, layout, 1.1, n, H, G, D, E, maps, 0.1, 100, 1e-5, m, code)
        outs.append([q, keep] + ([store.kv[0]["k"], store.kv[0]["v"]] if append else []))
    eps = torch.finfo(dtype).eps
    for i, (x, y) in enumerate(zip(*outs)):
        if i >= 2:                                         # pages of the two stores hold the same sequence in the same order
            x, y = x.float()[:T // 32], y.float()[:T // 32]
        size = y.abs().max()
        assert bool(((x - y).abs() <= (4e-6 * size if i < 2 else eps * y.abs() + 4e-6 * size)).all()), i


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,G,D,rot", [(8, 2, 64, 64), (9, 3, 128, 40), (30, 2, 22, 0)])
def test_many_pooled_slots_are_prepared_as_few_are(dtype, H, G, D, rot):
    from umbrella_amd import _lib
    T, code = 1700, _lib.seq_dtype_code(dtype)
    g = torch.Generator(device="cuda").manual_seed(D)
    proj, freq = torch.randn(T, (H + G) * D + 3, generator=g, device="cuda"), torch.rand(64, generator=g, device="cuda")
    pos, slot = torch.arange(T, device="cuda", dtype=torch.int32), torch.zeros(T, device="cuda", dtype=torch.int32)
    outs = []
    for seed, n in ((1, T), (2, 100)):
        c, _, _, _ = _decode_store([T], G, D, D, 5, dtype, 32, seed)
        q = torch.empty(T, H * D, device="cuda")
        for lo in range(0, T, n):
            _lib.seq_call("umb_pwa_prep", q[lo:], c.struct(0), proj[lo:lo + n], proj.shape[1], pos[lo:lo + n], slot[lo:lo + n], freq if rot else None, n, H, G,
                          D, rot, 1e-5, code)
        k, v = c.token_rows(0, 0, torch.arange(T))
        outs.append((q, k.float(), v.float()))
    eps = torch.finfo(dtype).eps
    assert torch.equal(outs[0][2], outs[1][2])
    for i in range(2):
        x, y = outs[0][i], outs[1][i]
        assert bool(((x - y).abs() <= (0 if i == 0 else eps) * y.abs() + 4e-6 * y.abs().max()).all())
