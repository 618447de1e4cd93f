"""The many-row products of the hybrid decoders whose weights go straight to registers (csrc/ob_dense.h, ob_dense_wr_kernel) with what their outputs become -- the
layer's input product, the logits, a sequential feed-forward's activation, keys and values of a prompt by head -- at every height of a tile these forms have
(64, 80, 96, 112 and 128 rows at these numbers of rows), the last rows and columns partly filled, sums shorter than a turn of the loop's steps and longer.
``onebit_hybrid_gemm`` reaches plain sums only (test_gpu_hybrid).  Against the restatement in float64 on the same weights; ``TOL`` is those tests'."""
import pytest
import torch

import test_gpu_hybrid as lebepel
import test_gpu_serotar as serotar
from oracle import lebepel_ref, serotar_ref
from test_hybrid_cpu import att, raw_config as lebepel_config
from test_serotar_cpu import dense, layer, raw_config as serotar_config

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
ROWS = pytest.mark.parametrize("T", [395, 460, 570, 680, 790])         # (513-528 tiles of 16 columns: 4, 5, 6, 7 and 8 tiles of 16 rows)


@ROWS
@pytest.mark.parametrize("width", [72, 230])
def test_input_product_and_logits(T, width):
    raw = lebepel_config([att(ff=4100, heads=2, kv_heads=1)], width=width, vocab=8203)
    raw["max_positions"] = 800
    m, w = lebepel.build(raw, BF)
    toks = lebepel.tokens(T, 8203, T)
    assert lebepel.err(lebepel.run(m.step_engine(1, 800, max_rows=T), 0, 0, toks), lebepel_ref.forward(raw, w, toks)) < lebepel.TOL[BF]


@ROWS
@pytest.mark.parametrize("width", [72, 230])
def test_activation_of_a_feed_forward(T, width):
    raw = serotar_config([layer(dense(8210))], width=width, side=0, vocab=203)
    m, w = serotar.build(raw, BF, edit=serotar.only("mlp"))
    toks = serotar.tokens(T, 203, T)
    assert serotar.err(serotar.run(m.step_engine(1, 800, max_rows=T), 0, 0, toks), serotar_ref.forward(raw, w, toks)) < serotar.TOL[BF]


@ROWS
@pytest.mark.parametrize("kv_rank", [64, 200])
def test_keys_and_values_by_head(T, kv_rank):
    raw = serotar_config([layer(heads=33, dim=100, vdim=128, q_rank=33, kv_rank=kv_rank, scale=0.1)], width=72, side=0)
    m, w = serotar.build(raw, BF, edit=serotar.only("mix"))
    toks = serotar.tokens(T, 61, T)
    assert serotar.err(serotar.run(m.step_engine(1, 800, max_rows=T), 0, 0, toks), serotar_ref.forward(raw, w, toks)) < serotar.TOL[BF]
