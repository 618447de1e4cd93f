"""The end of a sequential layer with more than 64 rows (feed-forward's row kernel, token input, depth average, next norm in one launch), bf16, against the
plain restatement (oracle/serotar_ref.py, float64).

``TOL``: bf16 activations (2^-9 relative each) through the three layers' dozen products, as in test_gpu_serotar.py, where their roundings average over a
row's columns; in rows of one k tile they need not: 12 products x 2 operands x 2^-9 = 0.047."""
import pytest

from oracle import serotar_ref as R
from test_gpu_serotar import BF, TOL, build, err, run, tokens
from test_serotar_cpu import dense, layer, moe, raw_config

pytestmark = pytest.mark.gpu

# width, mixture, columns of the token input: one k tile, a last wave that is not full, waves without columns, both register forms full and with one k tile
# more; two and four n tiles of the gate product, their columns padded; one, odd and many choices (all there are: none can fall differently), identity
# experts; the first width of the separate launches, one that is no whole number of k tiles
FORMS = {"one tile": (32, moe(4, 6, 2, None, 24, 32), 10), "half a wave": (544, moe(3, 3, 0, None, 72, 0), 33), "two a wave": (1024, moe(5, 9, 4, None, 40, 24), 32),
         "one more": (1056, moe(2, 4, 2, None, 40, 24), 64), "full": (2048, moe(7, 8, 1, None, 64, 128), 64), "few columns": (2048, moe(1, 1, 0, None, 32, 0), 20),
         "beyond": (2080, moe(2, 2, 0, None, 32, 0), 12), "not whole tiles": (1044, moe(2, 2, 0, None, 32, 0), 12)}


@pytest.mark.parametrize("name", FORMS)
def test_rows_of_a_prompt(name):
    width, mlp, side = FORMS[name]
    raw = raw_config([layer(mlp), layer(dense(40)), layer(mlp)], width=width, side=side, vocab=130)
    m, w = build(raw, BF)
    eng = m.step_engine(2, 160)
    for T in (65, 80, 97, 144):                                        # (one row a workgroup; the last band of 16 with one row, whole)
        toks = tokens(T, 130, T)
        assert err(run(eng, 0, 0, toks), R.forward(raw, w, toks)) < (TOL[BF] if width > 32 else 0.047), T


@pytest.mark.parametrize("name", ["half a wave", "one more", "full"])
def test_rows_of_a_workgroup(name):
    """Steps of 4096 rows (16 a workgroup on 256 CUs), 4100 (nine, two rounds; the last workgroup with five) and 700 (three) against the same prompts one at a
    time, one to six rows a workgroup.  Products split otherwise move single bf16 roundings (2^-9) of what follows: 2 % of a row's norm, as in
    test_gpu_hybrid_rows.py; a row in another's place shows as 100 %."""
    width, mlp, side = FORMS[name]
    m, _ = build(raw_config([layer(mlp), layer(dense(40))], width=width, side=side, vocab=130), BF)
    eng = m.step_engine(4, 1408, max_rows=4100)
    prompts = [tokens(n, 130, n) for n in (1404, 1300, 1000, 396)]
    for lens in ((1400, 1300, 1000, 396), (1404, 1300, 1000, 396), (240, 222, 170, 68)):
        batch = [p[:n] for p, n in zip(prompts, lens)]
        eng.launch([(i, 0, p, len(p)) for i, p in enumerate(batch)])
        whole, row = eng.logits[:sum(map(len, batch))].clone(), 0
        for i, p in enumerate(batch):
            eng.launch([(i, 0, p, len(p))])
            few, many = eng.logits[:len(p)], whole[row:row + len(p)]
            assert float(((many - few).norm(dim=1) / few.norm(dim=1)).max()) < 2e-2, (lens, i)
            row += len(p)
