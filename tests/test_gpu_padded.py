"""K that is no whole number of the LDS-DMA product's K steps (csrc/onebit_hip.hip, ob_g3_padded: rows and signs padded in the workspace), and rows of N % 8 == 4 values
through its epilogue and the LayerNorm: against the same sums in 64 bits."""
import pytest
import torch
from torch import nn

from onebit_amd import BitLinearInf, _lib

pytestmark = pytest.mark.gpu


def _layer(T, K, N, bias):
    g = torch.Generator(device="cuda").manual_seed(T * 7 + K + N)
    m = BitLinearInf(K, N, bias=bias, device="cuda", dtype=torch.float16)
    m.weight.data = torch.randint(0, 256, (N, K // 8), generator=g, device="cuda", dtype=torch.uint8).view(torch.int8)
    m.input_factor.data = torch.randn(K, generator=g, device="cuda").half()
    m.weight_scale.data = (0.1 * torch.randn(N, generator=g, device="cuda")).half()
    if bias:
        m.bias.data = torch.randn(N, generator=g, device="cuda").half()
    x = torch.randn(T, K, generator=g, device="cuda").half()
    x[:, -1] = 30.0                                   # the last column counts, what lies behind it does not
    return m, x


def _z64(m, x):
    K = x.shape[1]
    a = (x * m.input_factor).double()
    s = 1.0 - 2.0 * ((m.weight.view(torch.uint8)[:, :, None] >> torch.arange(8, device="cuda", dtype=torch.uint8)) & 1).reshape(-1, K).double()
    # (the bound of K / 32 float32 additions in any order)
    return a @ s.T, 4 * 2.0 ** -24 * K ** 0.5 * a.norm(dim=-1, keepdim=True)


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("K,N", [(1056, 256), (1376, 4100), (4064, 1000), (1248, 260), (2272, 8196), (1504, 12292), (1280, 4100)])
@pytest.mark.parametrize("T", [1, 3, 64, 65, 97, 129, 257])
def test_layer(T, K, N, bias):
    m, x = _layer(T, K, N, bias)
    z, err = _z64(m, x)
    g = m.weight_scale.double()
    y = m(x)
    m.layernorm = nn.Identity()
    u = m(x)
    # u (a bias is no part of it): z, then z * g, each rounded to float16
    assert ((u.double() - z * g).abs() <= 2.01 * 2.0 ** -11 * (z * g).abs() + err * g.abs() + 2.0 ** -24).all()
    # the LayerNorm of those very rows: float32 statistics (error within 2^-13 of a row's deviation), one rounding, and another behind the bias
    d = u.double() - u.double().mean(-1, keepdim=True)
    y64 = d / (d.square().mean(-1, keepdim=True) + 1e-5).sqrt()
    b = m.bias.double() if bias else torch.zeros_like(g)
    assert ((y.double() - (y64 + b)).abs() <= 2.0 ** -11 * (2 * y64.abs() + b.abs()) + 2.0 ** -13).all()


@pytest.mark.parametrize("T,K,N,pitch", [(65, 1376, 260, 1376), (130, 1376, 4100, 11008), (257, 1056, 1000, 2112)])
def test_partial_of_a_slice(T, K, N, pitch):
    m, _ = _layer(T, K, N, False)
    x = torch.randn(T, pitch, generator=torch.Generator(device="cuda").manual_seed(T), device="cuda").half()
    lib = _lib.load()
    ws = torch.empty(lib.onebit_linear_workspace_bytes(T, K, N, _lib.ONEBIT_F16), dtype=torch.uint8, device="cuda")
    assert ws.numel() > T * K * 2
    out = torch.empty(T, N, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    z, err = _z64(m, x[:, :K])
    for w in (ws, None):                              # with the workspace, and without
        out.fill_(float("nan"))
        _lib.check(lib.onebit_matmul_partial_ws(m.weight.data_ptr(), K // 8, x.data_ptr(), pitch, m.input_factor.data_ptr(), out.data_ptr(),
                                                None if w is None else w.data_ptr(), 0 if w is None else w.numel(), T, K, N, _lib.ONEBIT_F16, s), "partial")
        assert ((out.double() - z).abs() <= err + 2.0 ** -24).all()


# few columns, N % 8 == 4: rows of eight values a load up to 1024 of them and from 128 columns on, beside the other form
@pytest.mark.parametrize("T", [1024, 1025])
@pytest.mark.parametrize("N", [12, 124, 132])
@pytest.mark.parametrize("bias", [False, True])
def test_rows_of_few_values(T, N, bias):
    test_layer(T, 128, N, bias)
