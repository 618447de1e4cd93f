"""Prompt attention of several sequences: query blocks taken one by one where their pairs leave slots of the chip free and the XCDs' shares stay even,
in pairs elsewhere and from 512 pairs on.
Which workgroup sweeps a block does not enter its arithmetic: every segment's rows are, bit for bit, the single-sequence kernel's (always pairs)."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# (rows, past) of the segments; H x blocks: all resident (<= 512 blocks), dealt in rounds (equal segments, <= 511 pairs), pairs (from 512 on; unequal
# segments of more than 512 blocks; a block far back in its cache the longest either way); odd block counts, heads the groups do not divide evenly,
# one head, a segment of one row, a segment past a full cache
@pytest.mark.parametrize("spec,H,Hkv,D", [
    ([(1, 0)], 1, 1, 64), ([(700, 0)], 5, 1, 128), ([(129, 70), (1, 130), (640, 0), (385, 315)], 12, 4, 64), ([(512, 0)] * 4, 32, 8, 128),
    ([(513, 0), (700, 0), (127, 5)], 40, 40, 64), ([(640, 60), (640, 0), (256, 3)], 73, 73, 64), ([(700, 0)] * 6, 28, 28, 64), ([(257, 0)] * 8, 32, 4, 128),
    ([(640, 0)] * 4, 32, 8, 128), ([(300, 0), (600, 0)], 60, 12, 128), ([(256, 0), (106, 590), (31, 600)], 40, 8, 128)])
def test_blocks_and_pairs(spec, H, Hkv, D):
    from onebit_amd import _lib
    from onebit_amd.bitnet import _stream_ptr
    from onebit_amd.engine import _Seg as Seg
    lib, g = _lib.load(), torch.Generator(device=DEV).manual_seed(H + D)
    max_len, slots, T = 700, len(spec), sum(n for n, _ in spec)
    q = torch.randn(T, H, D, generator=g, device=DEV).half()
    k, v = (torch.randn(slots, Hkv, max_len, D, generator=g, device=DEV).half() for _ in range(2))
    segs, row = (Seg * slots)(), 0
    for i, (n, past) in enumerate(spec):
        segs[i] = Seg(row, n, slots - 1 - i, past)
        row += n
    o = torch.full((T, H, D), float("nan"), dtype=torch.float16, device=DEV)
    assert lib.onebit_attention_ragged(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), None, ctypes.cast(segs, ctypes.c_void_p), slots, H, Hkv, D,
                                       slots, max_len, _stream_ptr(o.device)) == 0
    for i, (n, past) in enumerate(spec):
        s, r0 = segs[i].slot, segs[i].row0
        one = torch.empty(n, H, D, dtype=torch.float16, device=DEV)
        assert lib.onebit_attention_prefill(q[r0:r0 + n].data_ptr(), k[s].data_ptr(), v[s].data_ptr(), one.data_ptr(), None, 1, n, H, Hkv, D, past, max_len,
                                            _stream_ptr(o.device)) == 0
        assert torch.equal(o[r0:r0 + n], one), (n, past)
