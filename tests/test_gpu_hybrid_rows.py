"""The hybrid decoders' row kernels of many rows (four rows a workgroup, from 1024 rows on) against the kernels of few rows: the same prompts as one
step of more than 1024 rows, and one request at a time.

A row's squares are added in the same order whatever the number of rows, so a step of 1024 rows equals, bit for bit, the same step without its last row
(everything else, the number of K splits among it, is the same in both).  One request at a time the products are split otherwise: float32 ulps that move
single bf16 roundings (2^-9) of what follows; 1 % of the logits' norm is asserted of every row (a row, or a quarter of one, that is wrong shows as 10 %
and more)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _equal_without_last_row(model, prompts):
    """Every row's logits of a step of 1024 rows are those of the same step of 1023."""
    eng = model.step_engine(4, 352, max_rows=1024)
    assert sum(len(p) for p in prompts) == 1024
    eng.launch([(i, 0, p, len(p)) for i, p in enumerate(prompts)])
    whole = eng.logits[:1024].clone()
    eng.launch([(i, 0, p[:len(p) - (i == 3)], len(p) - (i == 3)) for i, p in enumerate(prompts)])
    wrong = (whole[:1023] != eng.logits[:1023]).any(1).nonzero()
    assert not len(wrong), wrong[:8].flatten().tolist()


# widths of one, two and four pieces per thread and beyond (4100: the general kernel); groups of 24, 2048 and 4096 columns; not a whole piece (20)
@pytest.mark.parametrize("width,heads,vdim,groups,dtype", [(80, 4, 24, 4, torch.bfloat16), (1028, 32, 64, 1, torch.bfloat16), (2056, 64, 64, 1, torch.bfloat16),
                                                           (4096, 4, 20, 4, torch.bfloat16), (4100, 4, 24, 1, torch.bfloat16), (264, 4, 24, 1, torch.float32)])
def test_many_rows_equal_few(width, heads, vdim, groups, dtype):
    from onebit_amd.lebepel import LebepelConfig, build_synthetic_model
    mlp = {"kind": "dense", "ff": 64}
    cfg = LebepelConfig(vocab_size=96, width=width, norm_eps=1e-5, residual_mult=0.5, logit_softcap=20.0, max_positions=400, loop={"start": 0, "stop": 2, "times": 2},
                        layers=[{"type": "mamba2", "mixer": dict(heads=heads, groups=groups, state=16, vdim=vdim, conv=4, norm_groups=groups), "mlp": mlp},
                                {"type": "attention", "mixer": dict(heads=4, kv_heads=2, dim=24, vdim=32, scale=0.2), "mlp": mlp}])
    model = build_synthetic_model(cfg, seed=3, device="cuda", dtype=dtype)
    g = torch.Generator().manual_seed(width)
    prompts = [torch.randint(0, 96, (n,), generator=g).tolist() for n in (350, 349, 217, 111)]        # 1027 rows
    eng = model.step_engine(4, 352, max_rows=1027)
    eng.launch([(i, 0, p, len(p)) for i, p in enumerate(prompts)])
    whole = eng.logits[:1027].clone()
    row = 0
    for i, p in enumerate(prompts):
        eng.launch([(i, 0, p, len(p))])
        few, many = eng.logits[:len(p)], whole[row:row + len(p)]
        assert float(((many - few).norm(dim=1) / few.norm(dim=1)).max()) < (1e-2 if dtype == torch.bfloat16 else 1e-4), i
        row += len(p)
    _equal_without_last_row(model, prompts[:3] + [prompts[3][:108]])


# the same widths; experts all chosen (no choice can flip), six a token = one and a half rounds of four; identity expert, shared expert, none; depth
# averages over up to five results, token input.  (bf16, 2e-2: where few rows keep the experts' outputs in 32 bits, many rows round each to 2^-9)
@pytest.mark.parametrize("width,dtype", [(80, torch.bfloat16), (1028, torch.bfloat16), (2056, torch.bfloat16), (4100, torch.bfloat16), (1100, torch.float32)])
def test_many_sequential_rows_equal_few(width, dtype):
    from onebit_amd.serotar import SerotarConfig, build_synthetic_model
    mixer = dict(heads=2, dim=32, vdim=32, q_rank=32, kv_rank=32, scale=0.2)
    moe = lambda n, identity: {"kind": "moe", "expert": {"ff": 24}, "router": dict(experts=n, top=n + identity, identity=identity)}
    cfg = SerotarConfig(vocab_size=96, width=width, norm_eps=1e-5, embed_scale=2.0, bigram={"buckets": 64, "mul_prev": 7, "mul_cur": 5}, side_dim=16, layers=[
        {"type": "latent_attention", "mixer": mixer, "mlp": mlp} for mlp in ({"kind": "dense", "ff": 64}, dict(moe(5, 1), shared={"ff": 24}), None, moe(2, 0))])
    model = build_synthetic_model(cfg, seed=4, device="cuda", dtype=dtype)
    g = torch.Generator().manual_seed(width)
    prompts = [torch.randint(0, 96, (n,), generator=g).tolist() for n in (350, 349, 217, 111)]        # 1027 rows
    eng = model.step_engine(4, 352, max_rows=1027)
    eng.launch([(i, 0, p, len(p)) for i, p in enumerate(prompts)])
    whole = eng.logits[:1027].clone()
    row = 0
    for i, p in enumerate(prompts):
        eng.launch([(i, 0, p, len(p))])
        few, many = eng.logits[:len(p)], whole[row:row + len(p)]
        assert float(((many - few).norm(dim=1) / few.norm(dim=1)).max()) < (2e-2 if dtype == torch.bfloat16 else 1e-4), i
        row += len(p)
    _equal_without_last_row(model, prompts[:3] + [prompts[3][:108]])
