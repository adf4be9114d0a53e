"""A few rows' seam inside the product that reads them (umb_seq_front_linear) against the two launches it stands for: the same bits."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu

# rows, row, groups, slabs, rows of weights, epilogue (0 fp32, 1 stored type, 2 gated, 5 capped gated, 6 gelu gated, 8 capped)
SHAPES = [(1, 4096, 1, 1, 4096, 0), (1, 4096, 4, 1, 16400, 2), (2, 2048, 1, 1, 2592, 0), (1, 2048, 4, 4, 8200, 2), (2, 1024, 1, 4, 48, 5), (4, 1024, 4, 2, 1000, 8),
          (1, 192, 3, 1, 344, 0), (5, 192, 3, 1, 688, 2), (16, 168, 1, 1, 1000, 0), (1, 184, 1, 1, 496, 6), (3, 1000, 1, 1, 130, 1), (1, 2008, 1, 1, 100, 0),
          (1, 1024, 4, 3, 16, 0), (1, 3072, 3, 1, 9232, 0), (1, 1024, 1, 1, 9000, 0), (1, 512, 1, 2, 8300, 0), (1, 2048, 1, 1, 14336, 2), (7, 256, 1, 1, 30, 5), (1, 4096, 1, 1, 17, 8)]


def _front(lib, kind, T, W, groups, parts, dtype, g):
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")                                              # noqa: E731
    t = dict(x=rnd(T, W), y=rnd(parts, T, W), y2=rnd(parts, T, W), embed=rnd(50, W).to(dtype),
             tokens=torch.randint(0, 50, (T,), generator=torch.Generator().manual_seed(T)).to(torch.int32).cuda(), mix=rnd(1), out=rnd(1), in_=rnd(1))
    for n in ("w_post", "w_next", "w1", "w2"):
        t[n] = (1.0 + 0.1 * rnd(W)).to(dtype)
    f = lib.UmbSeqFront(kind=kind, W=W, groups=groups, V=50, parts=parts, parts2=parts, coef=0.5, m=0.7, offset=0.25, scale=1.5, eps=1e-6)
    for n, v in t.items():
        setattr(f, n, v.data_ptr())
    return f, t


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("kind", ["seam", "stream", "pair", "embed", "embed_stream"])
@pytest.mark.parametrize("T,W,groups,parts,N,epi", SHAPES)
def test_as_two_launches(dtype, kind, T, W, groups, parts, N, epi):
    from umbrella_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(T + W + N)
    code, k = _lib.seq_dtype_code(dtype), {"seam": 0, "stream": 1, "pair": 2, "embed": 3, "embed_stream": 3}[kind]
    groups = groups if kind in ("seam", "embed") else 1
    f, t = _front(_lib, k, T, W, groups, parts, dtype, g)
    if kind == "embed":
        f.in_, f.offset = None, 0.0
    dual = epi in (2, 5, 6)
    w, bias = (torch.randn(N, W, generator=g, device="cuda") * W ** -0.5).to(dtype), torch.randn(N, generator=g, device="cuda").to(dtype)
    if not _lib.load_seq().umb_seq_front_ok(C.byref(f), w.data_ptr(), T, N, epi, code):
        sets = T * groups * -(-(W // groups) // 256)
        assert sets > 8 and (dtype == torch.float32 or kind == "pair" or T > 1 and N > 4096) or (dual and W > 1024 and W * w.element_size() % 512)
        return
    x, h = t["x"].clone(), torch.empty(T, W, dtype=dtype, device="cuda")
    if kind == "seam":
        _lib.seq_call("umb_seq_resid_norm_parts", x, h, t["y"], parts, t["w_post"], t["w_next"], T, W, groups, 1e-6, code)
    elif kind == "stream":
        _lib.seq_call("umb_hc_seam_parts", x, h, t["y"], parts, t["mix"], t["out"], 0.7, t["in_"], t["w_next"], 0.25, T, W, 1, 1e-6, code)
    elif kind == "pair":
        _lib.seq_call("umb_seq_pair_resid_norm_parts", x, h, t["y"], parts, t["y2"], parts, t["w1"], t["w2"], 0.5, t["w_post"], t["w_next"], T, W, 1e-6, code)
    elif kind == "embed":
        _lib.seq_call("umb_seq_embed_norm", x, h, t["embed"], t["tokens"], 1.5, t["w_next"], T, W, 50, groups, 1e-6, code)
    else:
        _lib.seq_call("umb_hc_embed", x, h, t["embed"], t["tokens"], 1.5, t["in_"], t["w_next"], 0.25, T, W, 50, 1, 1e-6, code)
    cols = N // 2 if dual else N
    made = dtype if dual or epi == 1 else torch.float32
    want, got = torch.empty(T, cols, dtype=made, device="cuda"), torch.full((T + 1, cols), 3.0, dtype=made, device="cuda")
    x_out = torch.full((T + 1, W), 5.0, device="cuda")
    if epi == 5:
        _lib.seq_call("umb_seq_linear_glu", want, h, w, bias, T, N, W, 2.0, 1.7, code)
    elif epi == 8:
        _lib.seq_call("umb_seq_linear_cap", want, h, w, bias, T, N, W, 2.0, code)
    else:
        _lib.seq_call("umb_seq_linear", want, h, w, bias, T, N, W, epi, code)
    _lib.seq_call("umb_seq_front_linear", got, x_out, f, w, bias, T, N, epi, 2.0, 1.7, code)
    assert bool((got[T] == 3.0).all()) and bool((x_out[T] == 5.0).all())
    assert torch.equal(x_out[:T], x) and torch.equal(got[:T], want)


def test_refuses_what_it_does_not_cover():
    from umbrella_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(0)
    w, out = torch.zeros(32, 2048, dtype=torch.bfloat16, device="cuda"), torch.zeros(17, 32, device="cuda")

    def rc(T, change=lambda f, t: None, epi=0, W=2048, x_out=None):
        f, t = _front(_lib, 0, T, W, 1, 1, torch.bfloat16, g)
        change(f, t)
        x_out = torch.zeros(T, W, device="cuda") if x_out is None else t["x"]
        return _lib.load_seq().umb_seq_front_linear(out.data_ptr(), x_out.data_ptr(), C.byref(f), w.data_ptr(), None, T, 32, epi, 0.0, 0.0, 1,
                                                    torch.cuda.current_stream().cuda_stream)
    assert rc(2) == 0
    assert rc(3) != 0 and rc(17, W=64) != 0                    # more than 16 sets of 64 quads, more than a token tile
    assert rc(1, epi=5) != 0 and rc(1, epi=3) != 0             # a bound of zero, an epilogue with a gate of its own
    assert rc(1, x_out="x") != 0                               # the residual in place
    assert rc(1, lambda f, t: setattr(f, "w_next", None)) != 0
    assert rc(1, lambda f, t: setattr(f, "y", t["y"].data_ptr() + 4)) != 0
    assert rc(1, lambda f, t: setattr(f, "parts", 5)) != 0
    assert rc(1, lambda f, t: setattr(f, "groups", 3)) != 0


@pytest.mark.parametrize("width,groups", [(64, 1), (192, 3)])
def test_residuals_at_any_address(width, groups, monkeypatch):
    """a step of a few rows whose workspace is not 16-byte aligned runs its seams by themselves"""
    import types
    import seqmix_helpers
    from umbrella_amd import _lib
    cfg = seqmix_helpers.config([seqmix_helpers.attn_layer(heads=6, kv_heads=2, dim=12, window=20, pool=3, ff=32)] * 2, width=width, vocab=50, groups=groups)
    m, _ = seqmix_helpers.build(cfg, torch.float32, batch=2, max_length=32, max_tokens=64)
    real, got, shifted = _lib.load_seq(), [], []

    def forward(model, work, step, stream):
        w = work._obj
        shifted.append(torch.full((w.Tmax * width + 4,), 3.0, device="cuda"))
        was, w.x = w.x, shifted[-1].data_ptr() + 4
        try:
            return real.umb_seq_forward(model, work, step, stream)
        finally:
            w.x = was
    for shift in (False, True):
        m.clear()
        m.open(0)
        if shift:
            monkeypatch.setattr(_lib, "load_seq", lambda: types.SimpleNamespace(umb_seq_forward=forward))
        got.append(torch.cat([m.forward_batch([(0, [7, 8, 9])]).clone(), m.forward_batch([(0, [5])]).clone()]).float())
    assert len(shifted) == 2 and all(float(x[0]) == 3.0 and bool((x[-3:] == 3.0).all()) for x in shifted)
    assert bool(torch.isfinite(got[0]).all()) and float((got[0] - got[1]).norm() / got[0].norm()) <= 1e-5


@pytest.mark.parametrize("T,W,several", [(1, 4096, False), (410, 1024, False), (410, 2048, True), (600, 4096, True), (3, 6144, True)])
def test_roundings_of_a_seams_two_products(T, W, several):
    """written down, not the compiler's choice: which product of a sum of two is rounded by itself follows from how many quads a thread has"""
    from umbrella_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(T + W)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")                                              # noqa: E731
    x, y, mix, out, one, h = rnd(T, W), rnd(1, T, W), rnd(1), rnd(1), torch.ones(W, dtype=torch.bfloat16, device="cuda"), torch.empty(T, W, dtype=torch.bfloat16, device="cuda")
    new = x.clone()
    _lib.seq_call("umb_hc_seam_parts", new, h, y, 1, mix, out, 0.7, None, one, 0.0, T, W, 1, 1e-6, 1)
    my = torch.tensor(0.7, device="cuda") * y[0]
    want = [(mix.double() * x.double() + (out * my).double()).float(), (out.double() * my.double() + (mix * x).double()).float()]
    # the fused product in 64 bits, rounded twice: another value than one rounding's in one of 2^29 sums
    wrong = [int((new != w).sum()) for w in want]
    assert wrong[not several] <= 2 < wrong[several], wrong


# fp32 products that run on in two workgroups a unit; the last rows of weights that the one-tile kernel takes
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("kind", ["seam", "stream"])
@pytest.mark.parametrize("T,W,groups,parts,N,epi", [(4, 512, 1, 1, 12304, 0), (1, 2048, 1, 1, 16400, 1), (2, 1024, 1, 2, 8208, 8), (1, 1000, 1, 1, 16384, 0), (5, 384, 1, 3, 20000, 4)])
def test_long_products_as_two_launches(dtype, kind, T, W, groups, parts, N, epi):
    test_as_two_launches(dtype, kind, T, W, groups, parts, N, epi)


def test_where_rows_are_formed_inside():
    """the lines of the rule, either side"""
    from umbrella_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(0)

    def ok(dtype, T, W, N, epi=0):
        f, _ = _front(_lib, 0, T, W, 1, 1, dtype, g)
        return _lib.load_seq().umb_seq_front_ok(C.byref(f), 1 << 20, T, N, epi, _lib.seq_dtype_code(dtype))
    B, S = torch.bfloat16, torch.float32
    assert ok(B, 1, 1000, 16384) and not ok(B, 1, 1000, 16385) and ok(S, 1, 1000, 16385)
    assert ok(B, 1, 768, 65536) and not ok(B, 1, 768, 65537) and ok(B, 1, 640, 128256)
    assert ok(B, 1, 512, 32768, 2) and not ok(B, 1, 512, 32770, 2) and ok(B, 1, 1024, 32770, 2) and ok(B, 1, 2048, 128256)
    assert ok(S, 1, 4096, 8192) and not ok(S, 1, 4096, 8193) and ok(S, 1, 4096, 32768, 2) and ok(S, 1, 2048, 32000) and ok(B, 1, 4096, 32000)
    assert ok(B, 2, 2048, 4096) and not ok(B, 2, 2048, 4097)


def test_where_a_pairs_rows_are_formed_inside():
    """a pair's are more than a seam's: fewer rows of weights where every 16 of them form the rows"""
    from umbrella_amd import _lib
    g = torch.Generator(device="cuda").manual_seed(0)

    def ok(dtype, T, W, N, epi=0, kind=2):
        f, _ = _front(_lib, kind, T, W, 1, 1, dtype, g)
        return _lib.load_seq().umb_seq_front_ok(C.byref(f), 1 << 20, T, N, epi, _lib.seq_dtype_code(dtype))
    B, S = torch.bfloat16, torch.float32
    assert ok(B, 1, 256, 8192) and not ok(B, 1, 256, 8193) and ok(B, 1, 256, 8193, kind=0) and ok(S, 1, 128, 8192) and not ok(S, 1, 128, 8193)
    assert ok(B, 1, 384, 12288) and not ok(B, 1, 384, 12289) and ok(B, 1, 384, 16384, 2) and not ok(B, 1, 384, 16386, 2) and not ok(S, 1, 200, 8193)
    assert ok(S, 1, 384, 32000) and ok(B, 1, 2048, 32000) and ok(B, 1, 4096, 28672, 2)               # a ring that runs on forms them once a workgroup
