"""Decode attention of many (row, head) pairs, one to two per CU and more, against attention in float32, at contexts around the splits' ends; a row's
result does not depend on the other rows: the splits are the caller's, whatever the batch.

Bound: the kernel rounds scores to float16 twice (2^-11 of |s| <= 6: 3e-3 in a weight's exponent, averaged over the keys) and its output once:
4e-3 absolute for outputs of unit variance, as for single splits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("rows,H,Hkv", [(8, 32, 32), (23, 32, 8), (64, 8, 8)])
@pytest.mark.parametrize("chunk", [64, 128, 192, 256])
def test_many_pairs(rows, H, Hkv, chunk):
    from onebit_amd import _lib
    from onebit_amd.bitnet import _stream_ptr
    D, max_len = 128, 1500
    lib, g = _lib.load(), torch.Generator(device=DEV).manual_seed(rows + chunk)
    ctx = [1, chunk, chunk + 1, 511, 512, 513, 1023, 1024, 1025, 1500, 2 * chunk, 5 * chunk + 3]
    ctx = [min(ctx[r % len(ctx)], max_len) for r in range(rows)]
    q = torch.randn(rows, H, D, generator=g, device=DEV).half()
    k = (0.7 * torch.randn(rows, Hkv, max_len, D, generator=g, device=DEV)).half()
    v = torch.randn(rows, Hkv, max_len, D, generator=g, device=DEV).half()
    pos = torch.tensor([c - 1 for c in ctx], dtype=torch.int32, device=DEV)

    def run(q, k, v, pos):
        rows, ns = len(pos), -(-max_len // chunk)
        scratch = torch.zeros(int(lib.onebit_attention_decode_scratch_bytes(rows, H, ns)) + 16, dtype=torch.uint8, device=DEV)
        o = torch.empty(rows, H, D, dtype=torch.float16, device=DEV)
        for _ in range(2):                      # (the tickets are back at zero)
            assert lib.onebit_attention_decode_rows(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), None, None, pos.data_ptr(), rows, H, Hkv, D, rows,
                                                    max_len, chunk, ns, scratch.data_ptr(), scratch.numel(), _stream_ptr(o.device)) == 0
        return o
    o = run(q, k, v, pos)
    for r, c in enumerate(ctx):
        kk, vv = (t[r, :, :c].float().repeat_interleave(H // Hkv, 0) for t in (k, v))
        w = ((q[r].float()[:, None] @ kk.transpose(1, 2)) / D ** 0.5).softmax(-1)
        assert float((o[r].float() - (w @ vv)[:, 0]).abs().max()) < 4e-3, (r, c)
        assert torch.equal(o[r:r + 1], run(q[r:r + 1], k[r:r + 1], v[r:r + 1], pos[r:r + 1])), (r, c)
