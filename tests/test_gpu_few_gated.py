"""Decode steps of a state-space layer whose output product applies the mixer's norm (bf16, up to 32 rows), against the plain restatement
(oracle/lebepel_ref.py, float64).

``TOL`` (test_gpu_hybrid.py): bf16 activations, 2^-9 relative each; the product's operand is rounded before the row's factor 1 / rms instead of after it, once
either way."""
import pytest
import torch

from oracle import lebepel_ref as R
from test_gpu_hybrid import BF, TOL, build, err, tokens
from test_hybrid_cpu import att, raw_config, ssm

pytestmark = pytest.mark.gpu

# state-space layer, width: as few square sums as there can be, one k split; a split and a wave with k tiles of both kinds; eight splits, whole ones of either
# kind; no feed-forward columns behind the mixer's; and what keeps the norm's launch: heads of a part slice, two groups, sums that are no multiple of four
FORMS = {"small": (dict(heads=2, groups=1, state=16, vdim=64, norm_groups=1), 40), "both kinds": (dict(heads=12, groups=2, state=20, vdim=64, norm_groups=1, ff=1000), 264),
         "long": (dict(heads=64, groups=1, state=32, vdim=64, norm_groups=1, ff=5632), 96), "mixer only": (dict(heads=24, groups=1, state=16, vdim=32, norm_groups=1, ff=None), 72),
         "part slice": (dict(heads=4, groups=1, state=16, vdim=48, norm_groups=1), 40), "two groups": (dict(heads=8, groups=2, state=16, vdim=32, norm_groups=2), 40),
         "odd sums": (dict(heads=3, groups=1, state=16, vdim=32, norm_groups=1), 40)}


@pytest.mark.parametrize("name", FORMS)
def test_decoded_rows(name):
    """1 .. 64 requests, one token each at positions from the first on, in engines of as many slots and of more: then rows without a request, behind which the
    prompts' operands and square sums lie, share a token tile with live ones."""
    mix, width = FORMS[name]
    raw = raw_config([ssm(**mix), att(heads=2, kv_heads=2), ssm(**mix)], width=width, max_positions=64)
    m, w = build(raw, BF)
    toks = tokens(60, 61)
    ref = R.forward(raw, w, toks)
    for n, slots in ((1, 1), (1, 16), (2, 2), (2, 16), (16, 16), (17, 17), (17, 20), (17, 32), (32, 32), (33, 33), (33, 48), (64, 64)):
        at = [int(round(x)) for x in torch.linspace(59 if n == 1 else 0, 59, n).tolist()]
        eng = m.step_engine(slots, 64, max_rows=max(slots, sum(at)))
        if any(at):
            eng.launch([(i, 0, toks[:p]) for i, p in enumerate(at) if p])
        if slots > n:                                                  # (and a step of every row)
            eng.launch([(i, at[i] if i < n else 0, toks[at[i]:at[i] + 1] if i < n else toks[:1]) for i in range(slots)])
            for i, p in enumerate(at):
                eng.launch([(i, 0, toks[:p])] if p else [(i, 0, toks[:1])])
        eng.launch([(i, p, toks[p:p + 1]) for i, p in enumerate(at)])
        assert err(eng.logits[:n], ref[at]) < TOL[BF], (n, slots)
