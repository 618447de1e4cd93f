"""The 1-bit LDS-DMA products at row counts around every tile they choose from (96, 112, 128 tokens): unsliced, K-sliced and grouped launches.

Bound: u = fp16(fp16(z) g): two roundings of 2^-11, and the float32 sum of z behind them: K / 32 additions, 2^-24 sqrt(K) |a|_2 with a factor 4."""
import ctypes

import pytest
import torch
from torch import nn

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _layer(K, N, g):
    from onebit_amd import BitLinearInf
    m = BitLinearInf(K, N, device=DEV, dtype=torch.float16)
    m.weight.data = torch.randint(0, 256, (N, K // 8), generator=g, device=DEV, dtype=torch.uint8).view(torch.int8)
    m.input_factor.data = (0.05 + 0.1 * torch.rand(K, generator=g, device=DEV)).half()
    m.weight_scale.data = (0.05 + 0.1 * torch.rand(N, generator=g, device=DEV)).half()
    return m


def _check(m, a, u):
    s = 1.0 - 2.0 * ((m.weight.view(torch.uint8)[:, :, None] >> torch.arange(8, device=DEV, dtype=torch.uint8)) & 1).reshape(m.out_features, -1).double()
    ref = (a.double() @ s.T) * m.weight_scale.double()
    bound = 1.1 * 2.0 ** -10 * ref.abs() + 4 * 2.0 ** -24 * a.shape[1] ** 0.5 * a.double().norm(dim=1, keepdim=True) * m.weight_scale.double() + 2.0 ** -24
    assert ((u.double() - ref).abs() <= bound).all(), float(((u.double() - ref).abs() / bound).max())


@pytest.mark.parametrize("K,N", [(4096, 4096), (2048, 11008), (1024, 4100)])
@pytest.mark.parametrize("T", [97, 130, 192, 193, 224, 225, 337, 389, 449, 575, 577, 673, 701, 897, 1153, 1300, 1537, 1540, 2100])
def test_one_projection(T, K, N):
    g = torch.Generator(device=DEV).manual_seed(T + K)
    m = _layer(K, N, g)
    m.layernorm = nn.Identity()
    x = torch.randn(T, K, generator=g, device=DEV).half()
    _check(m, x * m.input_factor, m(x))


# fewer than 256 columns: K slices from 2048 of K on, the 128 x 128 kernel below
@pytest.mark.parametrize("K,N", [(2048, 128), (4096, 8), (4096, 248), (11008, 200), (1792, 128), (4096, 124)])
@pytest.mark.parametrize("T", [65, 96, 97, 129, 300, 2100])
def test_one_projection_of_few_columns(T, K, N):
    test_one_projection(T, K, N)


# up to 768 columns, either side of the rows from which on the 128 x 128 kernel is the faster one; K that is padded, and not
@pytest.mark.parametrize("T,K,N", [(2049, 1024, 260), (8001, 2048, 136), (3001, 2048, 136), (9000, 1376, 320), (2100, 1376, 320), (20001, 4064, 260), (4001, 4064, 768)])
def test_many_rows_of_few_columns(T, K, N):
    test_one_projection(T, K, N)


def _group(T, K, Ns):
    """(status, layers, rows, outputs) of one grouped launch; a row more than the outputs have is there to see that it stays."""
    from onebit_amd import _lib
    from onebit_amd.bitnet import _stream_ptr
    from onebit_amd.engine import _Proj, _proj
    lib = _lib.load()
    g = torch.Generator(device=DEV).manual_seed(T)
    ms = [_layer(K, N, g) for N in Ns]
    xs = [torch.randn(T, K, generator=g, device=DEV).half() for _ in ms]
    us = [torch.full((T + 1, N), 7.0, dtype=torch.float16, device=DEV) for N in Ns]
    arr = (_Proj * len(ms))(*[_proj(m) for m in ms])
    up, ap = ((ctypes.c_void_p * 3)(*[t.data_ptr() for t in ts]) for ts in (us, xs))
    return lib.onebit_linear_group_prescaled(ctypes.cast(arr, ctypes.c_void_p), up, ap, len(ms), T, _stream_ptr(xs[0].device)), ms, xs, us


def _check_group(T, K, Ns):
    rc, ms, xs, us = _group(T, K, Ns)
    assert rc == 0
    for m, x, u in zip(ms, xs, us):
        _check(m, x, u[:T])
        assert (u[T] == 7.0).all()                 # nothing behind the last row


@pytest.mark.parametrize("Ns", [(4096, 4096, 4096), (11008, 11008), (5120, 1028, 260)])
@pytest.mark.parametrize("T", [65, 96, 97, 129, 192, 577, 673, 897, 1025, 1153, 1540])
def test_grouped_projections(T, Ns):
    _check_group(T, 1024, Ns)


# members of fewer than 256 columns (keys and values of one head) and K below 1024: at any row count from 65 on with K >= 2048, else from half a round of
# 256 x 128 tiles on
@pytest.mark.parametrize("T,K,Ns", [(65, 2048, (2048, 128, 128)), (1153, 2048, (2048, 128, 128)), (193, 4096, (4096, 64, 64)), (1540, 1024, (4096, 128, 124)),
                                    (1540, 512, (1408, 1408)), (2100, 768, (768, 768, 768)), (1025, 256, (4100, 260)), (193, 256, (16384, 8))])
def test_grouped_projections_of_few_columns(T, K, Ns):
    _check_group(T, K, Ns)


@pytest.mark.parametrize("T,K,Ns", [(200, 512, (512, 512)), (191, 512, (16384, 16384)), (1540, 512, (250, 1408)), (1540, 1056, (4096, 4096))])
def test_groups_that_are_refused(T, K, Ns):
    assert _group(T, K, Ns)[0] == -2
