"""A step that names one sequence several times: its parts are one stretch of it.  The launches for single tokens append a token's key and value
beside the attention of the step's other rows, and a recurrent state has one owner a step: two rows of a sequence may not be two stretches."""
import ctypes as C
import types

import pytest
import torch

from umbrella_amd import _lib
from umbrella_amd._lib import UmbSeqModel, UmbSeqWork
from umbrella_amd.attn.cache import PagedSeqCache
from umbrella_amd.models import seqmix

PARTS = [("a", [7]), ("b", [1, 2, 3]), ("a", [8]), ("c", [4]), ("b", [5]), ("a", [9, 10])]
WANT = [[0], [2, 0], [0], [0], [0], [1, 0]]


def host_model(monkeypatch, steps):
    """a model whose launches are written down and not run"""
    m = seqmix.SeqMixLM.__new__(seqmix.SeqMixLM)
    m.kv_cache = PagedSeqCache([(1, 4, 0)], [], max_tokens=256, max_seqs=4, device="cpu", dtype=torch.float32, page=4)
    m.device, m.max_length, m.use_graph = "cpu", 64, False
    m.config = types.SimpleNamespace(layers=[0], width=2)
    m._bufs = {"logits": torch.zeros(64, 3)}
    m._m, m._ws = UmbSeqModel(), UmbSeqWork()
    m.reserve = lambda *a: None

    def forward(model, work, step, stream):
        s = step._obj
        read = lambda p, n: (C.c_int32 * n).from_address(p)[:]                            # noqa: E731
        got = {k: read(getattr(s, k), s.T) for k in ("tokens", "pos", "slot")}
        got.update({k: read(getattr(s, k), s.B) for k in ("seq_slot", "seq_row0", "seq_pos0", "seq_len")})
        got.update(max_len=s.max_len, rows=read(s.logit_rows, s.R) if s.logit_rows else list(range(s.R)))
        if s.trace:                                                                        # a row's trace: its token
            torch.frombuffer((C.c_float * (s.T * 2)).from_address(s.trace), dtype=torch.float32).copy_(
                torch.tensor(got["tokens"], dtype=torch.float32).repeat_interleave(2))
        steps.append(got)
        return 0
    monkeypatch.setattr(_lib, "load_seq", lambda: types.SimpleNamespace(umb_seq_forward=forward))
    monkeypatch.setattr(_lib, "stream_ptr", lambda: None)
    return m


@pytest.mark.parametrize("parts,want", [([("a", [7]), ("a", [8])], [[0], [0]]), (PARTS, WANT), (PARTS, None), ([("b", [1]), ("a", [2])], None),
                                        ([("b", [1]), ("a", [2])], [[0, 0], []]), ([("b", [1]), ("c", [2]), ("a", [3])], [[0], [0], [0]])])
def test_each_sequence_is_one_stretch(monkeypatch, parts, want):
    steps, before = [], {"a": 3, "b": 0, "c": 6}
    m = host_model(monkeypatch, steps)
    for sid, n in before.items():
        m.open(sid)
        if n:
            m.forward_batch([(sid, list(range(n)))])
    del steps[:]
    _, trace = m.forward_batch(parts, want, trace=True)
    (s,) = steps
    assert len(set(s["seq_slot"])) == len(s["seq_slot"])
    assert s["max_len"] == max(s["seq_len"]) and sum(s["seq_len"]) == len(s["tokens"])
    of = {m.kv_cache.slot(sid): sid for sid in before}
    tokens, positions = {sid: [] for sid in before}, {sid: [] for sid in before}
    for slot, row0, pos0, n in zip(s["seq_slot"], s["seq_row0"], s["seq_pos0"], s["seq_len"]):
        assert s["slot"][row0:row0 + n] == [slot] * n
        tokens[of[slot]] += s["tokens"][row0:row0 + n]
        positions[of[slot]] += s["pos"][row0:row0 + n]
        assert pos0 == s["pos"][row0]
    for sid in before:
        mine = [t for other, ids in parts for t in ids if other == sid]
        assert tokens[sid] == mine and positions[sid] == list(range(before[sid], before[sid] + len(mine)))
    # the wanted rows and the trace: in the order of the parts
    asked = [ids[k] for i, (_, ids) in enumerate(parts) for k in (want[i] if want else [len(ids) - 1])]
    assert [s["tokens"][r] for r in s["rows"]] == asked
    assert trace[0, :, 0].tolist() == [t for _, ids in parts for t in ids]


@pytest.mark.gpu
@pytest.mark.parametrize("family", ["gitopel", "tutunex", "potosun"])
def test_parts_of_a_sequence_are_that_stretch_in_one_part(family):
    import potosun_helpers
    import seqmix_helpers
    import tutunex_helpers
    built = {"gitopel": lambda: seqmix_helpers.build(seqmix_helpers.config([seqmix_helpers.attn_layer(), seqmix_helpers.gla_layer(ff=40)]), torch.bfloat16),
             "tutunex": lambda: tutunex_helpers.build(tutunex_helpers.config([tutunex_helpers.layer(tutunex_helpers.attention()),
                                                                              tutunex_helpers.layer(tutunex_helpers.parallel())]), torch.bfloat16),
             "potosun": lambda: potosun_helpers.build(potosun_helpers.config([potosun_helpers.layer(potosun_helpers.biased()),
                                                                              potosun_helpers.layer(potosun_helpers.latent())]), torch.bfloat16)}[family]()
    m = built[0] if isinstance(built, tuple) else built
    outs = []
    for parts, want in (([("a", [5]), ("b", [4]), ("a", [9])], [[0], [0], [0]]), ([("a", [5, 9]), ("b", [4])], [[0, 1], [0]])):
        for sid in "ab":
            m.open(sid)
        m.forward_batch([("a", list(range(3, 40))), ("b", list(range(6)))])
        step = m.forward_batch(parts, want=want).clone()
        outs.append([step if len(parts) == 2 else step[[0, 2, 1]], m.forward_batch([("a", [11]), ("b", [12])]).clone()])
        for sid in "ab":
            m.close(sid)
    for a, b in zip(*outs):
        assert torch.equal(a, b)
