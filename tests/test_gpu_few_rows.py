"""Steps of up to 64 rows of a sequential hybrid decoder (bf16): the row kernels that carry the router's or the token input's products, and the expert
products that find their rows in the choices, against the plain restatement (oracle/serotar_ref.py, float64).

``TOL``: bf16 activations (2^-9 relative each) through the two layers' dozen products, as in test_gpu_serotar.py; positions at which a choice of experts is
close are left out (``clear_choices``)."""
import pytest
import torch

from onebit_amd import hybrid
from oracle import serotar_ref as R
from test_gpu_serotar import BF, TOL, build, clear_choices, err, only, rows_err, run, tokens
from test_serotar_cpu import dense, layer, moe, raw_config

pytestmark = pytest.mark.gpu

# width, mixture, columns of the token input: one and several waves of columns, a last wave that is not full, padded k tiles; router of 1 .. 4 column tiles, the
# largest (64 entries); more experts than choices; no shared expert; the longest sums of a row kernel's products (64 and 128 k tiles) and one beyond
FORMS = {"one wave": (64, moe(6, 2, 2, (4, 2), 24, 32), 10), "four tiles": (260, moe(60, 5, 4, (8, 3), 40, 100), 33), "two tiles, no shared": (300, moe(20, 3, 0, None, 72, 0), 32),
         "full": (2048, moe(32, 6, 8, (8, 4), 64, 128), 64), "router only": (2052, moe(12, 2, 4, (4, 2), 40, 24), 20), "wide router": (4096, moe(30, 4, 2, None, 32, 64), 40),
         "wider than any": (4100, moe(10, 2, 0, None, 32, 0), 12)}


def clear_tokens(raw, w, T):
    """T tokens, their logits, and at which of them no choice of experts is close: more than a third of the positions (the first seed with one)."""
    for seed in (T, T + 1000, T + 2000):
        toks = tokens(T, 130, seed)
        ref, ok = clear_choices(raw, w, toks, 0.04)
        if bool(ok.any()):
            break
    assert int(ok.sum()) > T // 3
    return toks, ref, ok


@pytest.mark.parametrize("name", FORMS)
def test_rows_of_a_step(name):
    width, mlp, side = FORMS[name]
    raw = raw_config([layer(mlp), layer(dense(40)), layer(mlp)], width=width, side=side, vocab=130)
    m, w = build(raw, BF)
    eng = m.step_engine(2, 80)
    for T in (1, 2, 16, 17, 33, 64):
        toks, ref, ok = clear_tokens(raw, w, T)
        assert err(run(eng, 0, 0, toks), ref, ok) < TOL[BF], T


def test_decoded_rows_with_idle_ones():
    """17 requests in a bucket of 20 rows: the idle rows choose no expert and change nothing."""
    raw = raw_config([layer(moe(12, 3, 4, (4, 2), 40, 64)), layer(moe(12, 3, 4, (4, 2), 40, 64))], width=192, vocab=140)
    m, w = build(raw, BF)
    eng = m.step_engine(20, 40)
    prompts = [tokens(5 + i % 9, 140, i) for i in range(17)]
    eng.launch([(i, 0, p[:-1]) for i, p in enumerate(prompts)])
    eng.launch([(i, len(p) - 1, p[-1:]) for i, p in enumerate(prompts)])
    got, seen = eng.logits[:17].clone(), 0
    for i, p in enumerate(prompts):
        ref, ok = clear_choices(raw, w, p, 0.04)
        if bool(ok[-1]):
            seen += 1
            assert float(rows_err(got[i:i + 1], ref[-1:])) < 2 * TOL[BF], i       # (one row against its own rms instead of the whole reference's)
    assert seen > 4


def test_rows_do_not_change_each_other():
    """A row of a step is the same bits alone (with rows without a request beside it, and as an engine's only row), among 15 others and in a step of other
    order: sums run over a row, whatever its neighbours.  (Sums of six k tiles at most: none is split here, however many rows there are.)"""
    raw = raw_config([layer(moe(12, 3, 4, (4, 2), 40, 64))], width=192, vocab=140)
    m, _ = build(raw, BF)
    eng = m.step_engine(16, 40)
    prompts = [tokens(6, 140, i) for i in range(16)]
    eng.launch([(i, 0, p) for i, p in enumerate(prompts)])
    eng.launch([(i, 6, [i + 3]) for i in range(16)])
    together = eng.logits[:16].clone()
    eng.launch([(i, 6, [i + 3]) for i in reversed(range(16))])
    assert torch.equal(eng.logits[:16].flip(0), together)
    eng.launch([(9, 6, [12])])
    assert torch.equal(eng.logits[0], together[9])
    one = m.step_engine(1, 40)
    one.launch([(0, 0, prompts[9])])
    one.launch([(0, 6, [12])])
    assert torch.equal(one.logits[0], together[9])


# heads, sizes and ranks: rp 64 .. 512, padded columns everywhere, heads beyond a group of 16, more n tiles than waves, absorbing products of 1, 4 and 5 k tiles,
# a rank beyond the registers' 1024 columns, ranks that are no multiple of 4 (the launches by themselves)
LATENTS = {"rp 64": dict(heads=3, dim=24, vdim=40, q_rank=20, kv_rank=36, scale=0.4), "rp 128": dict(heads=17, dim=64, vdim=56, q_rank=100, kv_rank=112, scale=0.1),
           "rp 256": dict(heads=16, dim=128, vdim=128, q_rank=768, kv_rank=256, scale=0.08), "rp 512": dict(heads=20, dim=128, vdim=64, q_rank=96, kv_rank=500, scale=0.09),
           "wide heads": dict(heads=2, dim=144, vdim=136, q_rank=64, kv_rank=300, scale=0.08), "long rank": dict(heads=2, dim=32, vdim=32, q_rank=1236, kv_rank=64, scale=0.2),
           "odd ranks": dict(heads=5, dim=32, vdim=32, q_rank=39, kv_rank=61, scale=0.2)}


@pytest.mark.parametrize("name", LATENTS)
def test_decoded_rows_of_latent_attention(name):
    """1 .. 33 requests at contexts from one key to many splits, one token each."""
    raw = raw_config([layer(**LATENTS[name])], width=96, side=0)
    m, w = build(raw, BF, edit=only("mix"))
    toks = tokens(720, 61)
    ref = R.forward(raw, w, toks)
    for n in (1, 2, 9, 16, 17, 32, 33):
        at = [int(round(x)) for x in torch.linspace(719 if n == 1 else 1, 719, n).tolist()]
        eng = m.step_engine(n, 768, max_rows=sum(at))
        eng.launch([(i, 0, toks[:p]) for i, p in enumerate(at)])
        eng.launch([(i, p, toks[p:p + 1]) for i, p in enumerate(at)])
        assert err(eng.logits[:n], ref[at]) < TOL[BF], n


@pytest.mark.parametrize("pad", [512, 33024])
def test_more_padding_than_the_width_needs(pad, monkeypatch):
    """A model whose rows are padded by whole waves of columns, and beyond what a workgroup's default LDS holds: both are the C interface's to accept."""
    true_up = hybrid._up
    monkeypatch.setattr(hybrid, "_up", lambda n, m: pad if (n, m) == (68, 32) else true_up(n, m))
    raw = raw_config([layer(moe(4, 4, 2, None, 24, 32)), layer(dense(40)), layer(moe(4, 4, 2, None, 24, 32))], width=68, vocab=130)
    m, w = build(raw, BF)
    assert m.width_pad == pad
    eng = m.step_engine(2, 80)
    for T in (1, 16, 64, 70):
        toks, ref, ok = clear_tokens(raw, w, T)
        got = run(eng, 0, 0, toks)
        assert bool(torch.isfinite(got).all()), T
        assert err(got, ref, ok) < TOL[BF], T
