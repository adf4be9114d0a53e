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
