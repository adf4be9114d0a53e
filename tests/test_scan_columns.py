"""The token-by-token scan with more columns a thread (umb_lin_scan_rows) against one column a thread and against 64 bits."""
import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("H,groups,D,Dv,per_head", [(16, 16, 128, 256, 0), (16, 16, 128, 68, 0), (32, 8, 64, 84, 1), (9, 3, 256, 132, 0), (64, 64, 52, 16, 1), (24, 24, 184, 100, 0)])
@pytest.mark.parametrize("lens", [[17, 1, 16, 0], [33] * 5, [20] * 40])
def test_columns_of_a_thread(lens, H, groups, D, Dv, per_head):
    from umbrella_amd import _lib
    T, B = sum(lens), len(lens)
    g = torch.Generator(device="cuda").manual_seed(T + H + D + Dv)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")                                              # noqa: E731
    q, k, v = rnd(T, groups * D), rnd(T, groups * D + 4), rnd(T, H * Dv + 8)
    alpha = torch.rand(T, H if per_head else H * D, generator=g, device="cuda")
    start = rnd(B + 1, H, D, Dv)
    slot, row, pos, n = (torch.tensor(x, dtype=torch.int32, device="cuda")
                         for x in (list(range(B, 0, -1)), [sum(lens[:b]) for b in range(B)], [b % 2 for b in range(B)], lens))
    out = []
    for longest in (0, max(lens)):
        s, o = start.clone(), torch.full((T + 1, H * Dv), 7.0, device="cuda")
        args = (o, s, q, groups * D, k, groups * D + 4, v, H * Dv + 8, alpha, per_head, groups, slot, row, pos, n)
        if longest:
            _lib.seq_call("umb_lin_scan_rows", *args, T, B, longest, H, D, Dv, 0.25)
        else:
            _lib.seq_call("umb_lin_scan", *args, B, H, D, Dv, 0.25)
        out.append((o, s))
    S = start.double()
    a64 = (alpha.double()[:, :, None].expand(T, H, D) if per_head else alpha.double().view(T, H, D))
    kk, qq = (x.double()[:, :groups * D].view(T, groups, D).repeat_interleave(H // groups, 1) for x in (k, q))
    want = torch.empty(T, H, Dv, dtype=torch.float64, device="cuda")
    for b in range(B):
        sb = S[B - b] if b % 2 else torch.zeros_like(S[0])
        for t in range(sum(lens[:b]), sum(lens[:b]) + lens[b]):
            sb = a64[t][:, :, None] * sb + kk[t][:, :, None] * v[t, :H * Dv].double().view(H, 1, Dv)
            want[t] = (qq[t][:, :, None] * sb).sum(1) * 0.25
        if lens[b]:
            S[B - b] = sb
    # rounding: two a token in an element of the state, and a read-out's sum of D; measured against the largest values
    for o, s in out:
        assert float((s.double() - S).abs().max()) <= max(lens) * 2.0 ** -23 * float(S.abs().max())
        assert float((o[:T].double().view(T, H, Dv) - want).abs().max()) <= (max(lens) + D ** 0.5) * 2.0 ** -23 * float(want.abs().max())
        assert bool((o[T] == 7.0).all())
    if D % 64 == 0:                              # whole quads of rows: the same sums, whatever a thread's columns (contractions aside)
        assert float((out[0][0] - out[1][0]).abs().max()) <= 2.0 ** -20 * float(want.abs().max())


def test_the_plain_scan_is_one_column():
    """umb_lin_scan asks with max_len 0, of which no rows that fill the chip follow, however many heads; (rows, longest): the lines of the rule"""
    from umbrella_amd import _lib
    cols = _lib.load_seq().umb_lin_scan_columns
    for H, D, Dv in ((64, 256, 256), (32, 256, 256), (16, 128, 256), (1024, 52, 64)):
        assert cols(1, 0, H, D, Dv) == 1
    assert [cols(n * 96, 96, 16, 128, 256) for n in (1, 3, 4, 7, 8)] == [1, 1, 2, 2, 4]
    assert cols(800, 96, 16, 120, 256) == 4 and cols(800, 96, 16, 112, 256) == 1           # a lane's rows in whole quads
    assert cols(0, 1, 1, 1, 1) < 0 and cols(1, 1, 1, 257, 1) < 0
