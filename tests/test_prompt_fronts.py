"""What stands between a prompt's projection and its mixer, walked in quads: against the kernels of single channels, which take the same numbers from
columns that are not 16-byte aligned.  And attention of more than 1024 query tiles against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _steps(lens, first, dev="cuda"):
    """positions and slots of stretches of `lens` tokens that start at `first`, in slots of their own in mixed order"""
    slots = [(3 * i + 1) % len(lens) if len(lens) % 3 else i for i in range(len(lens))]
    pos = [p for n, f in zip(lens, first) for p in range(f, f + n)]
    slot = [s for n, s in zip(lens, slots) for _ in range(n)]
    return torch.tensor(pos, dtype=torch.int32, device=dev), torch.tensor(slot, dtype=torch.int32, device=dev)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("taps", [3, 4])
@pytest.mark.parametrize("Hk,H,D,E", [(2, 4, 24, 40), (1, 1, 128, 128), (3, 3, 100, 300), (2, 2, 132, 8), (1, 2, 256, 64), (8, 16, 128, 128)])
@pytest.mark.parametrize("many", [False, True])              # a wave each, and enough of them for quads
def test_delta_fronts(dtype, taps, Hk, H, D, E, many):
    from umbrella_amd import _lib
    lens, first = [1, 9, 2, 17, 8, 3, 1], [0, 5, 1, 0, 2, 40, 3]
    C, Dp = 2 * Hk * D + H * E, (D + 15) // 16 * 16
    if many:
        n = min(1200000 // C + 1, 20000 // (2 * Hk + H + 1) + 1)
        lens, first = lens + [n // 2 + 3, 5, n // 2], first + [0, 7, 2]
    T = sum(lens)
    pos, slot = _steps(lens, first)
    g = torch.Generator(device="cuda").manual_seed(D + E + taps)
    cols = C + H * E + 2 * H
    rows = torch.randn(T, cols, generator=g, device="cuda")
    ring = torch.randn(len(lens), taps, C, generator=g, device="cuda")
    conv = torch.randn(C, taps, generator=g, device="cuda").to(dtype)
    dtb, alog = (torch.randn(H, generator=g, device="cuda") for _ in range(2))
    outs = []
    for col0 in (4, 3):
        ld = (cols + col0 + 3) // 4 * 4 + (0 if col0 == 4 else 1)
        proj = torch.full((T, ld), 9.0, device="cuda")
        proj[:, col0:col0 + cols] = rows
        q, k, v = (torch.full(s, 8.0, device="cuda") for s in ((T, Hk * Dp), (T, Hk * Dp), (T, H * E)))
        beta, lg = (torch.empty(T, H, device="cuda") for _ in range(2))
        _lib.seq_call("umb_delta_prep", q, k, Hk * Dp, v, beta, lg, proj, ld, col0, conv, ring, dtb, alog, pos, slot, T, Hk, H, D, E, taps,
                      _lib.seq_dtype_code(dtype))
        outs.append((q, k, v, beta, lg))
    assert torch.equal(outs[0][3], outs[1][3]) and torch.equal(outs[0][4], outs[1][4])
    assert (outs[0][2] - outs[1][2]).abs().max() <= 2e-6 * outs[1][2].abs().max()          # sums of 3 or 4 products
    for a, b in zip(outs[0][:2], outs[1][:2]):                 # unit rows: sums of D squares in another order
        assert (a - b).abs().max() <= 4e-7 * D ** 0.5


# more than 1024 tiles of 16 rows, and heads of 64 and 32 also more than 1791 (four waves share the keys of causal prompts from there on; trees have a
# wave or two a tile): ragged rows, prefixes around a 64-key step and none, a cache that ends inside one (Lmax an odd multiple of 32), stale keys behind
# the valid ones
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D,Hq,Hkv,T,prefix,spare", [(128, 64, 8, 257, 63, 0), (128, 32, 8, 530, 0, 32), (64, 32, 8, 515, 65, 32), (64, 12, 4, 1400, 1, 0),
                                                     (32, 32, 32, 529, 130, 96), (32, 40, 8, 430, 0, 32), (64, 32, 8, 900, 65, 32),
                                                     (64, 24, 8, 1200, 1, 0), (32, 32, 32, 900, 130, 96), (32, 40, 8, 720, 0, 32)])
def test_attention_of_many_tiles(dtype, D, Hq, Hkv, T, prefix, spare):
    import numpy as np
    from umbrella_amd.attn.cache import VT_PAD, k_to_frag, vt_to_frag
    from umbrella_amd import _lib
    from umbrella_amd.models.llama import pack_mask_bits
    S, g = prefix + T, Hq // Hkv
    Lmax = (S + 31) // 32 * 32 + spare
    gen = torch.Generator().manual_seed(T + D)
    q, k, v = (torch.randn(n, h, D, generator=gen).to(dtype) for n, h in ((T, Hq), (S, Hkv), (S, Hkv)))
    kc, vt = torch.full((Hkv, Lmax, D), 7.0, dtype=dtype), torch.full((Hkv, D, Lmax + VT_PAD), -9.0, dtype=dtype)
    kc[:, :S], vt[:, :, :S] = k.permute(1, 0, 2), v.permute(1, 2, 0)
    kc, vt, qd = k_to_frag(kc).cuda(), vt_to_frag(vt).cuda(), q.cuda()
    rs = np.random.RandomState(T)
    tree = torch.zeros(T, T, dtype=torch.bool)
    for i in range(T):
        if i:
            tree[i] = tree[max(0, i - 1 - rs.randint(0, min(i, 24)))]
        tree[i, i] = True
    pre = torch.tensor([prefix], dtype=torch.int32, device="cuda")
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for bits, see in ((pack_mask_bits(tree).cuda(), tree), (None, torch.ones(T, T).tril().bool())):
        out = torch.full((T + 1, Hq, D), 3.0, dtype=dtype, device="cuda")
        _lib.call("umb_tree_attn", out, qd, kc, vt, None, None, pre, bits, 0 if bits is None else bits.shape[1], T, T, Hq, Hkv, D, Lmax, 256, 1,
                  D ** -0.5, None, _lib.dtype_code(dtype))
        mask = torch.cat([torch.ones(T, prefix, dtype=torch.bool), see], dim=1).cuda()
        for h in range(Hkv):
            kd, vd = k[:, h].double().cuda(), v[:, h].double().cuda()
            for a in range(h * g, h * g + g):
                p = torch.softmax(((q[:, a].double().cuda() @ kd.T) * D ** -0.5).masked_fill(~mask, -torch.inf), dim=-1)
                want = p @ vd
                # weights rounded to storage (a relative unit each), the result rounded once
                bound = 1.1 * unit * (p @ vd.abs()) + 1.1 * unit * want.abs() + 1e-5
                assert ((out[:T, a].double() - want).abs() <= bound).all()
        assert bool((out[T] == 3.0).all())


@pytest.mark.parametrize("D,Hq,Hkv,T,prefix", [(128, 32, 8, 530, 0), (64, 32, 8, 900, 65), (32, 40, 8, 720, 20)])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_values_that_are_not_finite_reach_one_tile_of_keys(D, Hq, Hkv, T, prefix, bad):
    """prompts of many query tiles: a value that a token does not see is weighted with zero inside its tile of 32 keys, and read nowhere else"""
    from umbrella_amd.attn.cache import VT_PAD, k_to_frag, vt_to_frag
    from umbrella_amd import _lib
    S, g, dtype = prefix + T, Hq // Hkv, torch.bfloat16
    Lmax = (S + 31) // 32 * 32
    gen = torch.Generator().manual_seed(T + D)
    q, k, v = (torch.randn(n, h, D, generator=gen).to(dtype) for n, h in ((T, Hq), (S, Hkv), (S, Hkv)))
    pre, outs = torch.tensor([prefix], dtype=torch.int32, device="cuda"), []
    for key in (None, (prefix + 32) // 64 * 64 + 40, (prefix + 300) // 64 * 64 + 32):       # in the later half of 64 keys
        kc, vt = torch.zeros(Hkv, Lmax, D, dtype=dtype), torch.zeros(Hkv, D, Lmax + VT_PAD, dtype=dtype)
        kc[:, :S], vt[:, :, :S] = k.permute(1, 0, 2), v.permute(1, 2, 0)
        if key is not None:
            vt[:, :, key] = bad
        out = torch.empty(T, Hq, D, dtype=dtype, device="cuda")
        _lib.call("umb_tree_attn", out, q.cuda(), k_to_frag(kc).cuda(), vt_to_frag(vt).cuda(), None, None, pre, None, 0, T, T, Hq, Hkv, D, Lmax, 256, 1,
                  D ** -0.5, None, _lib.dtype_code(dtype))
        outs.append(out)
        if key is not None:
            # a tile of 16 rows ends with the token of its last row: those whose keys end in front of the bad one's tile
            ends = [prefix + min((16 * (r // 16) + 15) // g, T - 1) + 1 for r in range(T * g)]
            clean = [t for t in range(T) if max(ends[t * g:t * g + g]) <= key // 32 * 32]
            assert clean and torch.equal(out[clean], outs[0][clean])
            assert bool((~out[key - prefix:].isfinite()).any())


# every count of 16-row tiles a wave (full, ragged, none), chunks of one token, whole and with a tail, heads that do not fill the eight XCDs
@pytest.mark.parametrize("D,E,Hk,H", [(16, 16, 1, 3), (33, 24, 2, 2), (64, 40, 1, 2), (80, 16, 3, 3), (96, 130, 1, 1), (128, 128, 4, 8), (144, 20, 1, 2),
                                      (208, 48, 1, 1), (256, 33, 1, 2)])
def test_delta_chunks(D, E, Hk, H):
    from umbrella_amd import _lib
    lens, first = [64, 1, 63, 200, 129], [0, 7, 3, 0, 64]
    T, B, Dp = sum(lens), len(lens), (D + 15) // 16 * 16
    g = torch.Generator(device="cuda").manual_seed(D + E)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")                   # noqa: E731
    ldqk = Hk * Dp + 8
    q, k = (torch.nn.functional.normalize(rnd(T, Hk, D), dim=-1) for _ in range(2))
    v, beta, lg, state = rnd(T, H, E), torch.rand(T, H, generator=g, device="cuda"), -0.2 * torch.rand(T, H, generator=g, device="cuda"), rnd(B, H, D, E)
    qd, kd = torch.full((2, T, ldqk), 5.0, device="cuda")
    for dst, src in ((qd, q), (kd, k)):
        dst[:, :Hk * Dp] = torch.nn.functional.pad(src, (0, Dp - D)).reshape(T, Hk * Dp)
    row0 = [sum(lens[:i]) for i in range(B)]
    meta = [torch.tensor(x, dtype=torch.int32, device="cuda") for x in ([2, 0, 4, 1, 3], row0, first, lens)]
    got, out = state.clone(), torch.full((T + 1, H, E), 3.0, device="cuda")
    scratch = torch.full((_lib.load_seq().umb_delta_scan_floats(T, H, D, E),), 6.0, device="cuda")
    _lib.seq_call("umb_delta_scan", out, got, qd, kd, ldqk, v, beta, lg, *meta, T, B, max(lens), Hk, H, D, E, scratch, scratch.numel())
    for b, slot in enumerate([2, 0, 4, 1, 3]):
        S = torch.zeros(H, D, E, dtype=torch.float64, device="cuda") if first[b] == 0 else state[slot].double()
        want = torch.empty(lens[b], H, E, dtype=torch.float64, device="cuda")
        for i in range(lens[b]):
            t = row0[b] + i
            qt, kt = (z[t].double().repeat_interleave(H // Hk, dim=0) for z in (q, k))
            S = S * lg[t].double().exp()[:, None, None]
            u = beta[t].double()[:, None] * (v[t].double() - (S * kt[:, :, None]).sum(1))
            S = S + kt[:, :, None] * u[:, None, :]
            want[i] = (S * qt[:, :, None]).sum(1)
        # sums of D + 64 products of 32-bit numbers through a triangular system of unit keys
        bound = 3e-5
        assert (out[row0[b]:row0[b] + lens[b]] - want).norm() <= bound * want.norm() and (got[slot] - S).norm() <= bound * S.norm()
    assert bool((out[T] == 3.0).all())


# the rows of a step come from several pages, whole and cut anywhere: what the cache's page size is must not show
@pytest.mark.parametrize("D,E,maps,keep,chunk", [(128, 128, 1, 0, 0), (72, 48, 1, 37, 0), (64, 128, 2, 0, 61), (24, 16, 1, 3, 0), (256, 208, 1, 0, 0)])
def test_prompt_attention_of_any_page_size(D, E, maps, keep, chunk):
    from umbrella_amd import _lib
    from umbrella_amd.attn.cache import PagedSeqCache
    lens, news, H, G, window, Dc, R = [201, 40, 131], [201, 1, 97], 4, 2, 90, E // 16 * 16, D // 8 * 8
    T, dtype = sum(news), torch.bfloat16
    g = torch.Generator(device="cuda").manual_seed(D)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")                   # noqa: E731
    keys, vals, lat = ([rnd(n, *s).to(dtype) for n in lens] for s in ((G, maps * D), (G, E), (Dc + R,)))
    q, qa = rnd(T, H, maps, D), rnd(T, H, Dc + R)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")              # noqa: E731
    row0, pos0, cnt = i32([sum(news[:b]) for b in range(3)]), i32([n - k for n, k in zip(lens, news)]), i32(news)
    outs = []
    for page in (16, 7, 1, 256):
        c = PagedSeqCache([(G, maps * D, 0, E)], [], sum(lens) + 3 * page, 3, "cuda", dtype, page=page, latent_layers=(Dc + R,))
        entries = []
        for b, n in enumerate(lens):
            c.open(b)
            c.extend(b, n, entries)
        c.write_pages(entries)
        for b, n in enumerate(lens):
            at = torch.arange(n, device="cuda")
            pg = c.pages_dev[c.slot(b)].long()[at // page]
            c.kv[0]["k"][pg, :, at % page] = keys[b]
            c.kv[0]["v"][pg, :, at % page] = vals[b]
            c.latent[0][pg, at % page] = lat[b]
        slot = i32([c.slot(b) for b in range(3)])
        out, lout = torch.full((T + 1, H * E), 3.0, dtype=dtype, device="cuda"), torch.full((T + 1, H * Dc), 3.0, dtype=dtype, device="cuda")
        form = _lib.UmbAttnForm(maps, chunk, None, 0.3, 1e-3, keep, 0)
        _lib.seq_call("umb_attn_attend_tiled", out, H * E, q, c.struct(0), None, 0, -1, None, 0, slot, row0, pos0, cnt, 3, max(news), H, G, D, E, window,
                      D ** -0.5, 1.0, 0.0, form, _lib.seq_dtype_code(dtype))
        _lib.seq_call("umb_lat_attend_tiled", lout, qa, c.latent_struct(0), None, slot, row0, pos0, cnt, 3, max(news), H, Dc, R, window, (Dc + R) ** -0.5,
                      _lib.seq_dtype_code(dtype))
        outs.append((out, lout))
    assert bool((outs[0][0][T] == 3.0).all()) and bool((outs[0][1][T] == 3.0).all()) and bool(outs[0][0].isfinite().all())
    for o in outs[1:]:
        assert torch.equal(o[0], outs[0][0]) and torch.equal(o[1], outs[0][1])


@pytest.mark.parametrize("D,E,maps,n", [(128, 128, 1, 1), (64, 64, 1, 129), (128, 256, 2, 70), (128, 128, 1, 192)])
def test_single_token_in_a_cache_of_one_span(D, E, maps, n):
    """a page table of less than one span of keys: no splits and no merge behind them, the bits of a large cache"""
    from umbrella_amd import _lib
    from umbrella_amd.attn.cache import PagedSeqCache
    H, G, dtype = 8, 2, torch.bfloat16
    g = torch.Generator(device="cuda").manual_seed(n)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")                   # noqa: E731
    keys, vals, q = rnd(n, G, maps * D).to(dtype), rnd(n, G, E).to(dtype), rnd(1, H, maps, D)
    pos, scratch, outs = torch.tensor([n - 1], dtype=torch.int32, device="cuda"), torch.full((H * maps * 16 * (E + 2),), 4.0, device="cuda"), []
    for room in (n, 4000):
        c = PagedSeqCache([(G, maps * D, 0, E)], [], room, 1, "cuda", dtype, page=16)
        entries = []
        c.open(0)
        c.extend(0, n, entries)
        c.write_pages(entries)
        at = torch.arange(n, device="cuda")
        pg = c.pages_dev[c.slot(0)].long()[at // 16]
        c.kv[0]["k"][pg, :, at % 16], c.kv[0]["v"][pg, :, at % 16] = keys, vals
        out, slot = torch.full((2, H * E), 3.0, dtype=dtype, device="cuda"), torch.tensor([c.slot(0)], dtype=torch.int32, device="cuda")
        _lib.seq_call("umb_attn_attend", out, H * E, q, c.struct(0), None, 0, -1, None, 0, pos, slot, 1, H, G, D, E, 2 ** 30, D ** -0.5, 1.0, 0.0,
                      _lib.UmbAttnForm(maps, 0, None, 0.3, 1e-3, 0, 0), scratch, scratch.numel(), _lib.seq_dtype_code(dtype))
        assert bool((out[1] == 3.0).all()) and bool(out.isfinite().all())
        outs.append(out)
    assert torch.equal(outs[0], outs[1])
