"""Steps whose every row's logits are wanted, in order (the last seam norms them for the head), against the same rows asked for otherwise."""
import pytest
import torch

import potosun_helpers
import seqmix_helpers
import tomopel_helpers
import tutunex_helpers
import zusuvik_helpers

pytestmark = pytest.mark.gpu

MODELS = {"grouped norms": lambda dt: seqmix_helpers.build(seqmix_helpers.config([seqmix_helpers.attn_layer(), seqmix_helpers.gla_layer(ff=40)]), dt),
          "no feed-forward at the end": lambda dt: seqmix_helpers.build(seqmix_helpers.config([seqmix_helpers.attn_layer(), seqmix_helpers.gla_layer()]), dt),
          "two mixers": lambda dt: tutunex_helpers.build(tutunex_helpers.config([tutunex_helpers.layer(tutunex_helpers.attention()),
                                                                                  tutunex_helpers.layer(tutunex_helpers.parallel())]), dt),
          "one stream": lambda dt: potosun_helpers.build(potosun_helpers.config([potosun_helpers.layer(potosun_helpers.biased()),
                                                                                 potosun_helpers.layer(potosun_helpers.latent())]), dt),
          # the null row list of these goes to the launch that reads the sum of the streams, or the one stream of parallel blocks
          "two streams": lambda dt: tomopel_helpers.build(tomopel_helpers.config([tomopel_helpers.layer(tomopel_helpers.parallel()),
                                                                                  tomopel_helpers.layer(tomopel_helpers.mingru())]), dt),
          "parallel blocks": lambda dt: zusuvik_helpers.build(zusuvik_helpers.config([zusuvik_helpers.layer(zusuvik_helpers.retention()),
                                                                                      zusuvik_helpers.layer(zusuvik_helpers.parallel(), mlp=None)]), dt)}


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("name", MODELS)
def test_every_row_and_the_same_rows_out_of_order(name, dtype):
    built = MODELS[name](dtype)
    m = built[0] if isinstance(built, tuple) else built
    V = m.config.vocab_size
    g = torch.Generator().manual_seed(5)
    seqs = {k: torch.randint(0, V, (n,), generator=g).tolist() for k, n in (("a", 19), ("b", 1), ("c", 33))}

    def play(tag, order):
        """a scored prompt and two single tokens, rows wanted by `order`; back in their places"""
        out = []
        for s in seqs:
            m.open(tag + s)
        for parts in ([(s, t[:-2] or t) for s, t in seqs.items()], [(s, t[-2:-1] or t) for s, t in seqs.items()], [(s, t[-1:]) for s, t in seqs.items()]):
            want = [order(list(range(len(t)))) for _, t in parts]
            got = m.forward_batch([(tag + s, t) for s, t in parts], want=want).clone()
            for w in want:
                for k in sorted(range(len(w)), key=w.__getitem__):
                    out.append(got[k])
                got = got[len(w):]
        for s in seqs:
            m.close(tag + s)
        return torch.stack(out)
    whole = play("x", lambda rows: rows)
    turned = play("y", lambda rows: rows[::-1] + rows[:1])         # one row more, so not every row in order even for single tokens
    keep, at = [], 0
    for parts in ([max(len(t) - 2, 1) for t in seqs.values()], [1] * 3, [1] * 3):
        for n in parts:                                            # sorted: row 0 twice, then the others
            keep += [at] + list(range(at + 2, at + n + 1))
            at += n + 1
    got = turned[keep]
    assert whole.shape == got.shape and torch.isfinite(whole).all()
    assert (whole - got).abs().max() <= (1e-5 if dtype == torch.float32 else 2e-2) * whole.abs().max()      # the same norm by another kernel, rounded to `dtype`
