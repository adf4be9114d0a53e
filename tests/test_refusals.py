"""What the step paths refuse, as the launches they replaced did: before anything is launched (the addresses are never read)."""
import ctypes as C

import pytest

from umbrella_amd import _lib

EINVAL, AT = -22, 1 << 20


def gla_step(rank, ld=None, **kw):
    a = dict(T=1, H=2, D=64, Dv=64)
    a.update(kw)
    ld = ld or 2 * a["H"] * a["D"] + 2 * a["H"] * a["Dv"] + rank
    return _lib.load_seq().umb_gla_step(AT, AT, AT, ld, AT, None, AT, AT, AT, a["T"], a["H"], a["D"], a["Dv"], rank, 16.0, 0.125, 1e-6, 1, None)


@pytest.mark.parametrize("kw", [dict(rank=8193), dict(rank=0), dict(rank=16, D=257), dict(rank=16, Dv=260), dict(rank=16, Dv=66), dict(rank=16, T=65536),
                                dict(rank=16, ld=527)])
def test_gla_step(kw):
    """decays of a rank above 8192 are refused for prompts too"""
    assert gla_step(**kw) == EINVAL


@pytest.mark.parametrize("rows", [None, AT])
@pytest.mark.parametrize("streams,block", [(0, 0), (1, 0), (0, 1)])
def test_logits_without_a_final_norm(rows, streams, block):
    """also where every row is wanted and the last seam norms them: nothing would write what the head reads"""
    layer, m, ws, s = _lib.UmbSeqLayer(), _lib.UmbSeqModel(), _lib.UmbSeqWork(), _lib.UmbSeqStep()
    m.dtype, m.L, m.W, m.V, m.groups, m.eps, m.streams, m.block = 1, 1, 64, 64, 1, 1e-6, streams, block
    m.embed, m.layers = AT, C.pointer(layer)
    layer.norm1 = AT
    for k in ("x", "h", "proj", "aux", "o", "mix", "act", "y", "logits", "h2", "y2"):
        setattr(ws, k, AT)
    ws.Tmax, ws.Rmax, ws.aux_floats, ws.y_rows = 16, 16, 1 << 20, 16
    s.T, s.B, s.R, s.max_len = 1, 1, 1, 1
    for k in ("tokens", "pos", "slot", "seq_slot", "seq_row0", "seq_pos0", "seq_len"):
        setattr(s, k, AT)
    s.logit_rows = rows
    assert _lib.load_seq().umb_seq_forward(C.byref(m), C.byref(ws), C.byref(s), None) == EINVAL


EHIP = -5


def one_row(streams, x, h=AT):
    layer, m, ws, s = _lib.UmbSeqLayer(), _lib.UmbSeqModel(), _lib.UmbSeqWork(), _lib.UmbSeqStep()
    m.dtype, m.L, m.W, m.V, m.groups, m.eps, m.streams, m.embed_scale = 1, 1, 64, 64, 1, 1e-6, streams, 1.0
    m.embed, m.layers = AT, C.pointer(layer)
    layer.norm1, layer.kind, layer.heads, layer.dim, layer.vdim = AT, 1, 1, 16, 16
    layer.proj.w, layer.proj.N, layer.proj.K = AT, 64, 64
    for k in ("proj", "aux", "o", "mix", "act", "y", "logits", "h2", "y2"):
        setattr(ws, k, AT)
    ws.x, ws.h = x, h
    ws.Tmax, ws.Rmax, ws.aux_floats, ws.y_rows = 16, 16, 1 << 20, 16
    s.T, s.B, s.R, s.max_len = 1, 1, 0, 1
    for k in ("tokens", "pos", "slot", "seq_slot", "seq_row0", "seq_pos0", "seq_len"):
        setattr(s, k, AT)
    return _lib.load_seq().umb_seq_forward(C.byref(m), C.byref(ws), C.byref(s), None)


def no_device():
    import torch
    return not torch.cuda.is_available()


@pytest.mark.skipif("not __import__('test_refusals').no_device()", reason="the addresses are nobody's: a device would read them")
@pytest.mark.parametrize("streams", [0, 1])
def test_residuals_at_any_address(streams):
    """a few rows whose residual is not 16-byte aligned run their seam by itself (EHIP: the launch was reached, without a device); one that is not there is
    refused in front of any launch, with its scratch rows"""
    assert one_row(streams, AT) == EHIP and one_row(streams, AT + 4) == EHIP
    assert one_row(streams, None) == EINVAL and (streams or one_row(streams, AT, None) == EINVAL)
