"""Latent attention's norms of many rows (a wave per row), against the plain restatement (oracle/serotar_ref.py, float64): the prompt's rows, and the token
after it, which reads the cache entries they left."""
import pytest

from oracle import serotar_ref as R
from test_gpu_serotar import BF, F32, TOL, build, err, only, run, tokens
from test_serotar_cpu import layer, raw_config

pytestmark = pytest.mark.gpu


# ranks, rows: one piece a lane, padded; whole and last part-filled pieces at either end of both register forms; one column too many; one row too few;
# workgroups with one to four rows
@pytest.mark.parametrize("q_rank,kv_rank,T", [(20, 36, 1025), (764, 260, 1026), (764, 260, 1023), (768, 260, 1539), (1548, 500, 1536), (1548, 500, 1535), (1552, 500, 1537)])
@pytest.mark.parametrize("dtype", [BF, F32], ids=["bf16", "f32"])
def test_norms_of_many_rows(q_rank, kv_rank, T, dtype):
    raw = raw_config([layer(heads=2, dim=32, vdim=32, q_rank=q_rank, kv_rank=kv_rank, scale=0.2)], width=64, side=0, vocab=200)
    m, w = build(raw, dtype, edit=only("mix"))
    toks = tokens(T + 1, 200, T)
    ref = R.forward(raw, w, toks)
    eng = m.step_engine(1, T + 8, max_rows=T)
    assert err(run(eng, 0, 0, toks[:T]), ref[:T]) < TOL[dtype]
    assert err(run(eng, 0, T, toks[T:]), ref[T:]) < TOL[dtype]
