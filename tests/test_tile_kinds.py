"""Staged products of prompts (csrc/gemm_tile.h): every tile that a launch chooses from, at ragged edges, with rows stored as whole lines, in quads
and one by one, with K of one stage, fewer stages than the ring has slots, and more; against float64."""
import pytest
import torch

# (T, N, K) of single matrices by the tile that they get; N % 8 == 0, N % 4 == 0 and odd
TILES = ["256", "192", "160", "128 wide", "96", "128", "64 split"]          # csrc/gemm_tile.h, in its order
SHAPES = [(*shape, tile) for tile, shapes in {
    "256": [(1600, 8184, 64), (2049, 6145, 320), (2049, 6148, 192)],                                  # 256 rows x 256 tokens
    "192": [(1300, 6145, 128), (1300, 8188, 64), (2300, 5124, 320)],
    "160": [(2300, 8184, 192), (900, 8184, 64), (1101, 8190, 192), (2049, 8188, 320)],
    "128 wide": [(1101, 6152, 192), (1300, 5001, 128), (2300, 2592, 320)],
    "96": [(257, 6148, 64), (1025, 4112, 320), (2300, 2050, 192)],
    "128": [(257, 8184, 320), (257, 200, 64), (300, 1001, 192), (1000, 1028, 320)],                   # 128 x 128
    "64 split": [(257, 2048, 128), (300, 1004, 384), (2049, 129, 128)]}.items() for shape in shapes]  # 128 x 64, K over two groups of waves
# packed weights: (T, N, K, S), K in slabs of one stage, of an even and an odd number, and a slab past the last stage
PACKED = [(1600, 8176, 128, 1, "256"), (1300, 6160, 128, 1, "192"), (900, 8176, 128, 1, "160"), (1101, 6160, 128, 1, "128 wide"),
          (257, 8176, 128, 1, "96"), (1025, 4112, 384, 1, "96"), (257, 6160, 128, 1, "64 split"), (300, 1008, 640, 3, "128"),
          (1300, 5008, 384, 4, "192"), (257, 2048, 256, 2, "64 split"), (300, 1008, 128, 2, "128")]


def test_shapes_get_the_tiles_they_are_listed_for():
    from umbrella_amd import _lib
    kind = _lib.load_seq().umb_seq_tile_kind
    for *shape, tile in SHAPES:
        assert TILES[kind(*shape, 1)] == tile, shape
    for *shape, tile in PACKED:
        assert TILES[kind(*shape)] == tile, shape
    assert {s[-1] for s in SHAPES} == {s[-1] for s in PACKED} == set(TILES)


@pytest.mark.gpu
@pytest.mark.parametrize("T,N,K", [s[:3] for s in SHAPES])
def test_every_tile(T, N, K):
    from umbrella_amd import _lib
    dtype = torch.bfloat16 if K % 128 else torch.float16
    code, half_ulp = _lib.seq_dtype_code(dtype), 2.0 ** -8 if K % 128 else 2.0 ** -11
    g = torch.Generator(device="cuda").manual_seed(T + N + K)
    x, w, b = (torch.randn(s, generator=g, device="cuda").to(dtype) for s in ((T, K), (N, K), (N,)))
    full, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    tol = 2.0 ** -24 * (K + 2) * (size + b.double().abs())                     # an fp32 sum of K products in any order, and the bias
    out = torch.full((T + 1, N), 7.0, device="cuda")
    _lib.seq_call("umb_seq_linear", out, x, w, b, T, N, K, 0, code)
    assert ((out[:T].double() - (full + b.double())).abs() <= tol).all() and bool((out[T] == 7.0).all())
    out = torch.full((T + 1, N), 7.0, dtype=dtype, device="cuda")
    _lib.seq_call("umb_seq_linear", out, x, w, None, T, N, K, 1, code)
    assert ((out[:T].double() - full).abs() <= 1.01 * half_ulp * full.abs() + tol + 2.0 ** -25).all() and bool((out[T] == 7.0).all())
    n = N // 2                                                                 # stacked halves: |d silu| <= 1.1 |d gate|
    gate, up, tg, tu = full[:, :n], full[:, n:2 * n], tol[:, :n], tol[:, n:2 * n]
    act = torch.full((T + 1, n), 7.0, dtype=dtype, device="cuda")
    _lib.seq_call("umb_seq_linear", act, x, w[:2 * n].contiguous(), None, T, 2 * n, K, 2, code)
    want = gate * torch.sigmoid(gate) * up
    bound = 1.02 * half_ulp * want.abs() + 1.1 * tg * up.abs() + gate.abs() * tu + 1e-6 * want.abs() + 2.0 ** -25
    assert ((act[:T].double() - want).abs() <= bound).all() and bool((act[T] == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("T,N,K,S", [s[:4] for s in PACKED])
def test_every_tile_of_packed_weights(T, N, K, S):
    from umbrella_amd import _lib
    from umbrella_amd.models.llama import PackedLinear
    dtype = torch.float16 if K > 128 else torch.bfloat16
    half_ulp = 2.0 ** -11 if K > 128 else 2.0 ** -8
    g = torch.Generator(device="cuda").manual_seed(T + N + K)
    x, w = (torch.randn(s, generator=g, device="cuda").to(dtype) for s in ((T, K), (N, K)))
    full, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    tol = 2.0 ** -24 * (K + S) * size
    lin, code = PackedLinear.from_dense(w), _lib.dtype_code(dtype)
    part = torch.full((S + 1, T, N), 7.0, device="cuda")
    _lib.call("umb_gemm", part, x, x.stride(0), lin.w, None, T, N, K, 0, S, lin.Rtb, 0, code)
    assert ((part[:S].double().sum(0) - full).abs() <= tol).all() and bool((part[S] == 7.0).all())
    inter = PackedLinear.from_dense(w, interleave=True)                        # gate and up rows in pairs
    act = torch.full((T + 1, N // 2), 7.0, dtype=dtype, device="cuda")
    _lib.call("umb_gemm", act, x, x.stride(0), inter.w, None, T, N, K, 0, 1, inter.Rtb, 2, code)
    gate, up, tg, tu = full[:, :N // 2], full[:, N // 2:], tol[:, :N // 2], tol[:, N // 2:]
    want = gate * torch.sigmoid(gate) * up
    bound = 1.05 * half_ulp * (1.1 * gate.abs() * up.abs() + 3 * want.abs()) + 1.1 * tg * up.abs() + 1.1 * gate.abs() * tu + 2e-6 * want.abs() + 2.0 ** -24
    assert ((act[:T].double() - want).abs() <= bound).all() and bool((act[T] == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 300])
@pytest.mark.parametrize("epi", [2, 6])
def test_gates_far_from_zero(T, epi):
    """gated epilogues at the ends of their exponential, at infinities and NaN: what torch gives in 64 bits, on few tokens and on tiles"""
    from umbrella_amd import _lib
    K, vals = 64, [0.0, -0.0, 1e-20, 3.0, -3.0, 30.0, -30.0, 86.0, -86.0, 200.0, -200.0, 3e38, float("inf"), float("nan")]
    n = 128
    w = torch.zeros(2 * n, K, device="cuda", dtype=torch.bfloat16)
    w[:n, 0], w[n:, 1] = 1.0, 1.0                              # gate = x[0], up = x[1]
    for v in vals:
        x = torch.zeros(T, K, device="cuda", dtype=torch.bfloat16)
        x[:, 0], x[:, 1] = v, 1.0
        act = torch.empty(T, n, device="cuda", dtype=torch.bfloat16)
        _lib.seq_call("umb_seq_linear", act, x, w, None, T, 2 * n, K, epi, _lib.BF16)
        g = x[0, 0].double().cpu()
        if v == float("inf") or v != v:                        # 0 * inf in the other products of the row: everything is NaN
            assert bool(torch.isnan(act).all())
            continue
        want = g * torch.sigmoid(g) if epi == 2 else torch.nn.functional.gelu(g, approximate="tanh")
        assert ((act.double().cpu() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-30).all(), v


# per-head products on tiles (96 of them and more) and just below, ragged tokens and rows, one stage and several, row strides beyond the row; outputs
# whose rows are no whole 16-byte groups stay where they were
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,T,N,K,pad", [(32, 385, 128, 64, 8), (7, 900, 200, 192, 0), (50, 257, 72, 320, 24), (12, 1024, 64, 128, 8), (24, 500, 130, 64, 2)])
def test_batched_tiles(dtype, B, T, N, K, pad):
    from umbrella_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(T + N + K)
    code, ldx, per = _lib.seq_dtype_code(dtype), B * K + pad, N + pad
    half_ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    x, w = torch.randn(T, ldx, generator=g, device="cuda").to(dtype), torch.randn(B, N, K, generator=g, device="cuda").to(dtype)
    gate = torch.randn(T, B * N, generator=g, device="cuda")
    xs, wt = x[:, :B * K].double().view(T, B, K).transpose(0, 1).contiguous(), w.double().transpose(1, 2).contiguous()
    full, size = (torch.bmm(a, b).transpose(0, 1) for a, b in ((xs, wt), (xs.abs(), wt.abs())))          # [T][B][N]
    tol = 2.0 ** -24 * (K + 2) * size
    for epi in (0, 1, 3, 7):
        out = torch.full((T + 1, B * per), 7.0, dtype=torch.float32 if epi == 0 else dtype, device="cuda")
        _lib.seq_call("umb_seq_linear_batched", out, x, w, T, N, K, ldx, B * per, B, K, N * K, per, epi, gate if epi > 1 else None, B * N,
                      N if epi == 3 else 1, code)
        f = 1.0
        if epi == 3:
            f = torch.sigmoid(gate.double()).view(T, B, N)
        elif epi == 7:
            f = torch.sigmoid(gate[:, :B].double())[..., None]
        got = out[:T].double().view(T, B, per)
        want = full * f
        bound = tol + 2.0 ** -22 * want.abs() + (0.0 if epi == 0 else 1.02 * half_ulp * want.abs() + 2.0 ** -25)
        assert ((got[..., :N] - want).abs() <= bound).all() and bool((got[..., N:] == 7.0).all()) and bool((out[T] == 7.0).all())


# gates whose exponential leaves the normal range, infinities, NaN: fp32 on few tokens and many, 16 bits on tiles
GATES = [0.0, -0.0, 1e-38, 5.0, 88.5, 200.0, 3e38, float("inf"), -86.9, -87.4, -88.0, -88.6, -89.0, -100.0, -200.0, -3e38, float("-inf"), float("nan")]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,T", [(torch.float32, 1), (torch.float32, 300), (torch.bfloat16, 300)])
def test_gates_to_the_ends_of_their_range(dtype, T):
    """silu(gate) * up of the biases alone: the products are zero"""
    from umbrella_amd import _lib
    K, n = 128, 144
    gate = torch.tensor((GATES * n)[:n]).to(dtype)
    x, w = torch.zeros(T, K, device="cuda", dtype=dtype), torch.zeros(2 * n, K, device="cuda", dtype=dtype)
    act = torch.empty(T, n, device="cuda", dtype=dtype)
    _lib.seq_call("umb_seq_linear", act, x, w, torch.cat([gate, torch.ones(n, dtype=dtype)]).cuda(), T, 2 * n, K, 2, _lib.seq_dtype_code(dtype))
    z = gate.double()
    want = (z / (1.0 + torch.exp(-z))).expand(T, n)
    # 3.1 units of 2^-24; e^-z beyond 32 bits (|z| > 88.72) gives 0; one rounding to 16 bits, whose least steps are 2^-133
    half = dtype == torch.bfloat16
    bound = (3.1 * 2.0 ** -24 + (2.0 ** -8 if half else 0.0)) * want.abs() + want.abs() * (z < -88.72) + 2.0 ** (-134 if half else -149)
    got = act.double().cpu()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    ok = ~torch.isnan(want)
    assert torch.equal(got[ok].isinf(), want[ok].isinf()) and ((got - want).abs() <= bound)[ok & ~want.isinf()].all()


@pytest.mark.gpu
@pytest.mark.parametrize("epi", [3, 7])
def test_batched_gates_to_the_ends_of_their_range(epi):
    """the gate of a per-head product on tiles: a gate that is no number is seen in the result"""
    from umbrella_amd import _lib
    B, T, N, K = 32, 300, 128, 64
    g = torch.Generator(device="cuda").manual_seed(epi)
    x, w = (torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16) for s in ((T, B * K), (B, N, K)))
    gate = torch.tensor((GATES * (T * B * N // len(GATES) + 1))[:T * B * N], device="cuda").view(T, B * N).contiguous()
    out = torch.empty(T, B * N, device="cuda", dtype=torch.bfloat16)
    _lib.seq_call("umb_seq_linear_batched", out, x, w, T, N, K, B * K, B * N, B, K, N * K, N, epi, gate, B * N, N if epi == 3 else 1, _lib.BF16)
    xs, wt = x.double().view(T, B, K).transpose(0, 1).contiguous(), w.double().transpose(1, 2).contiguous()
    full, size = (torch.bmm(a, b).transpose(0, 1) for a, b in ((xs, wt), (xs.abs(), wt.abs())))
    s = torch.sigmoid(gate.double()).view(T, B, N) if epi == 3 else torch.sigmoid(gate[:, :B].double())[..., None].expand(T, B, N)
    want, got = full * s, out.double().view(T, B, N)
    assert torch.equal(got.isnan(), want.isnan())
    # the product's sums, one rounding to 16 bits (least steps 2^-133), gates whose exponential is beyond 32 bits
    bound = 2.0 ** -24 * (K + 4) * size * s + 1.02 * 2.0 ** -8 * want.abs() + want.abs() * (s < 2.95e-39) + 2.0 ** -134
    assert ((got - want).abs() <= bound)[~want.isnan()].all()


# whole rounds of 256 x 256 tiles with the columns behind them in another tile: (T, N, K, columns, tile); rows stored as whole lines, in quads, one by one
MIXED = [(1027, 22488, 192, 51, "192"), (1318, 18735, 64, 42, "192"), (1030, 22029, 192, 51, "160"), (1559, 14468, 64, 36, "160"), (486, 37771, 192, 128, "128 wide"),
         (1162, 17976, 320, 51, "128 wide"), (643, 30628, 64, 85, "96"), (491, 32774, 192, 128, "96")]
MIXED_PACKED = [(1308, 18720, 128, 42, "192"), (1540, 14496, 256, 36, "160"), (483, 37152, 128, 128, "128 wide"), (482, 32928, 384, 128, "96")]


def test_mixed_shapes_get_the_tiles_they_are_listed_for():
    from umbrella_amd import _lib
    for T, N, K, columns, tile in MIXED + MIXED_PACKED:
        got = _lib.load_seq().umb_seq_tile_mix(T, N, K)
        assert (got // len(TILES), TILES[got % len(TILES)]) == (columns, tile), (T, N, K)
    assert {m[-1] for m in MIXED} == {m[-1] for m in MIXED_PACKED} == {"192", "160", "128 wide", "96"}
    for T, N, K in [(2048, 16384, 2048), (256, 65536, 64), (1024, 8192, 4096), (300, 1000, 64)]:         # whole rounds, or less than one
        assert _lib.load_seq().umb_seq_tile_mix(T, N, K) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("T,N,K", [s[:3] for s in MIXED])
def test_mixed_tiles(T, N, K):
    test_every_tile(T, N, K)


@pytest.mark.gpu
@pytest.mark.parametrize("T,N,K", [s[:3] for s in MIXED_PACKED])
def test_mixed_tiles_of_packed_weights(T, N, K):
    test_every_tile_of_packed_weights(T, N, K, 1)
