"""Layer calls of 2 to 64 rows whose product goes through K in slices (csrc/onebit_hip.hip, ob_skinny_slices), and their neighbours that do not: against the same sums in
64 bits, ragged last phases and column tiles, with and without a bias and the workspace."""
import pytest
import torch
from torch import nn

from onebit_amd import BitLinearInf, _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,N", [(4096, 1000), (4224, 72), (7168, 4096), (7296, 2056), (11008, 4096), (6656, 8)])
@pytest.mark.parametrize("T", [2, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("bias", [False, True])
def test_layer(T, K, N, bias):
    g = torch.Generator(device="cuda").manual_seed(T + K + N)
    m = BitLinearInf(K, N, bias=bias, device="cuda", dtype=torch.float16)
    m.weight.data = torch.randint(0, 256, (N, K // 8), generator=g, device="cuda", dtype=torch.uint8).view(torch.int8)
    m.input_factor.data = torch.randn(K, generator=g, device="cuda").half()
    m.weight_scale.data = (0.1 * torch.randn(N, generator=g, device="cuda")).half()
    if bias:
        m.bias.data = torch.randn(N, generator=g, device="cuda").half()
    x = torch.randn(T, K, generator=g, device="cuda").half()
    lib, s = _lib.load(), torch.cuda.current_stream().cuda_stream
    sliced = lib.onebit_linear_workspace_bytes(T, K, N, _lib.ONEBIT_F16) > 0
    assert sliced == (T > 32 or K > 13 * 512)
    a = (x * m.input_factor).double()
    z = a @ (1.0 - 2.0 * ((m.weight.view(torch.uint8)[:, :, None] >> torch.arange(8, device="cuda", dtype=torch.uint8)) & 1).reshape(N, K).double()).T
    # K / 32 float32 additions in any order; z, then z * g, each rounded to float16
    err, gs = 4 * 2.0 ** -24 * K ** 0.5 * a.norm(dim=-1, keepdim=True), m.weight_scale.double()
    y = m(x)
    m.layernorm = nn.Identity()
    u = m(x)
    assert ((u.double() - z * gs).abs() <= 2.01 * 2.0 ** -11 * (z * gs).abs() + err * gs.abs() + 2.0 ** -24).all()
    # float32 statistics (error within 2^-13 of a row's deviation), one rounding, and another behind the bias
    d = u.double() - u.double().mean(-1, keepdim=True)
    y64 = d / (d.square().mean(-1, keepdim=True) + 1e-5).sqrt()
    b = m.bias.double() if bias else torch.zeros_like(gs)
    assert ((y.double() - (y64 + b)).abs() <= 2.0 ** -11 * (2 * y64.abs() + b.abs()) + 2.0 ** -13).all()
    # both outputs, and a call without the workspace
    p = lambda t: None if t is None else t.data_ptr()
    for n in {lib.onebit_linear_workspace_bytes(T, K, N, _lib.ONEBIT_F16), 0}:
        ws = torch.empty(n, dtype=torch.uint8, device="cuda") if n else None
        y2, u2 = torch.full_like(y, float("nan")), torch.full_like(y, float("nan"))
        _lib.check(lib.onebit_linear_forward(p(m.weight), K // 8, p(x), p(m.input_factor), p(m.weight_scale), p(m.bias) if bias else None, p(y2), p(u2), p(ws), n, T, K, N,
                                             _lib.ONEBIT_F16, 1e-5, 0, s), "forward")
        assert ((u2.double() - z * gs).abs() <= 2.01 * 2.0 ** -11 * (z * gs).abs() + err * gs.abs() + 2.0 ** -24).all()
        if n:
            assert torch.equal(u2, u) and torch.equal(y2, y)


# a second output that no 16-byte store can take, a bias that no 16-byte load can: the kernels that ask for neither, the same layer
@pytest.mark.parametrize("T,K,N", [(18, 11008, 4096), (100, 11008, 4096), (130, 2816, 1000)])
@pytest.mark.parametrize("what", ["u", "bias"])
def test_unaligned_second_output_and_bias(T, K, N, what):
    g = torch.Generator(device="cuda").manual_seed(T)
    w = torch.randint(0, 256, (N, K // 8), generator=g, device="cuda", dtype=torch.uint8)
    h, scale, bias = (0.1 + torch.rand(n, generator=g, device="cuda").half() for n in (K, N, N))
    x = torch.randn(T, K, generator=g, device="cuda").half()
    lib, s, p = _lib.load(), torch.cuda.current_stream().cuda_stream, lambda t: t.data_ptr()
    n = lib.onebit_linear_workspace_bytes(T, K, N, _lib.ONEBIT_F16)
    ws, res = torch.empty(n, dtype=torch.uint8, device="cuda"), []
    for off in (0, 1):
        u, b = torch.full((T * N + 16,), 7.0, dtype=torch.float16, device="cuda"), torch.empty(N + 8, dtype=torch.float16, device="cuda")
        uo, bo = off if what == "u" else 0, off if what == "bias" else 0
        b[bo:bo + N] = bias
        y = torch.empty(T, N, dtype=torch.float16, device="cuda")
        _lib.check(lib.onebit_linear_forward(p(w), K // 8, p(x), p(h), p(scale), p(b) + 2 * bo, p(y), p(u) + 2 * uo, p(ws), n, T, K, N, _lib.ONEBIT_F16, 1e-5, 0, s), "forward")
        assert bool((u[:uo] == 7).all()) and bool((u[uo + T * N:] == 7).all())
        res.append((u[uo:uo + T * N].double(), y.double()))
    # sums in another order: a rounding to float16 apart here and there
    for a, b in zip(*res):
        assert float((a - b).norm() / a.norm()) <= 2.0 ** -10
