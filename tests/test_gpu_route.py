"""Rows of a mixture's experts in steps of more than 64 tokens, against the plain restatement (oracle/serotar_ref.py, float64): float32, so that only choices
closer than its rounding can fall differently (left out, ``clear_choices``); a token in a wrong row, twice or not at all is another output altogether."""
import pytest

from test_gpu_serotar import F32, TOL, build, clear_choices, err, run, tokens
from test_serotar_cpu import layer, moe, raw_config

pytestmark = pytest.mark.gpu


# experts, choices, identity experts, tokens: one expert; as many threads a count as there are (3 experts, 341 runs); few tokens more than one workgroup's; counts
# of 16 tokens up to the last size that has them (16 K counts) and of 64 beyond; two counts a thread's share; one run (more than 512 experts)
@pytest.mark.parametrize("experts,top,identity,T", [(1, 1, 0, 65), (3, 2, 1, 500), (6, 2, 2, 80), (32, 6, 8, 129), (256, 4, 0, 1024), (256, 4, 0, 1040), (300, 3, 20, 200),
                                                    (600, 5, 8, 437), (600, 2, 0, 450)])
def test_rows_of_experts(experts, top, identity, T):
    raw = raw_config([layer(moe(experts, top, identity, None, 8, 16))], width=32, side=0, vocab=200)
    m, w = build(raw, F32)
    eng = m.step_engine(1, T + 8, max_rows=T)
    toks = tokens(T, 200, experts)
    ref, ok = clear_choices(raw, w, toks, 1e-3)
    assert int(ok.sum()) > T // 3
    assert err(run(eng, 0, 0, toks), ref, ok) < TOL[F32]
