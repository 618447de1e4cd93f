"""The float32 layer on the matrix cores (csrc/ob_f32.h) against the same sums in 64 bits.

The three bf16 parts of an activation are the activation, the signs are exact, so what is left is the order of float32 additions.  Bound of the
pre-LayerNorm output u = g sum_k s a: K / 32 additions into the upper parts' accumulators, each off by half an ulp of the running sum at most --
that is below |a|_2 sqrt(K) in the worst case used here by far -- so 2^-24 * sqrt(K) * |a|_2 * |g| with a factor 4, and 2 ulps of u itself."""
import numpy as np
import pytest
import torch
from torch import nn

pytestmark = pytest.mark.gpu


def _layer(K, N, seed, bias, pitch=0):
    from onebit_amd import BitLinearInf
    g = torch.Generator(device="cuda").manual_seed(seed)
    m = BitLinearInf(K, N, bias=bias, device="cuda", dtype=torch.float32)
    m.weight.data = torch.randint(0, 256, (N, K // 8 + pitch), generator=g, device="cuda", dtype=torch.uint8).view(torch.int8)[:, :K // 8]
    for p in (m.input_factor, m.weight_scale) + ((m.bias,) if bias else ()):
        p.data = torch.randn(p.shape, generator=g, device="cuda")
    return m, g


def _signs(m):
    b = m.weight.contiguous().view(torch.uint8)
    return 1.0 - 2.0 * ((b[:, :, None] >> torch.arange(8, device=b.device, dtype=torch.uint8)) & 1).reshape(b.shape[0], -1).double()


def _check(m, x, seed=0):
    a = (x * m.input_factor).double()
    u64 = (a @ _signs(m).T) * m.weight_scale.double()
    y = m(x)
    ln, m.layernorm = m.layernorm, nn.Identity()
    u = m(x)                                             # no LayerNorm, no bias
    m.layernorm = ln
    bound = 4 * 2.0 ** -24 * a.shape[-1] ** 0.5 * a.norm(dim=-1, keepdim=True) * m.weight_scale.abs().double() + 2.0 ** -22 * u64.abs()
    assert ((u.double() - u64).abs() <= bound).all(), float(((u.double() - u64).abs() / bound).max())
    c = u64 - u64.mean(-1, keepdim=True)
    rstd = 1 / (c.square().mean(-1, keepdim=True) + 1e-5).sqrt()
    y64 = c * rstd + (0 if m.bias is None else m.bias.double())
    # the row's own errors (its mean's too), scaled by 1 / std, and the normalisation's few roundings
    b_y = 2 * rstd * bound.amax(-1, keepdim=True) + 2.0 ** -20 * (1 + y64.abs())
    assert ((y.double() - y64).abs() <= b_y).all(), float(((y.double() - y64).abs() / b_y).max())


# every token block (16, 32, 64, 128; 64 where 128 pads more), one row over and under, whole rounds with and without a split rest
@pytest.mark.parametrize("T", [1, 2, 16, 17, 32, 33, 64, 65, 128, 129, 256, 300])
@pytest.mark.parametrize("K,N", [(4096, 6016), (4064, 9000), (2816, 9000)])
def test_rows_against_64_bits(T, K, N):
    m, g = _layer(K, N, T + K, False)
    _check(m, torch.randn(T, K, generator=g, device="cuda"))


# both numberings of the tiles: the token blocks first up to 8 blocks of 128 rows, beyond it where all tiles run at once on small parts (264 -> 4100), else the columns;
# with and without whole rounds, a split rest in both
@pytest.mark.parametrize("T", [1024, 1025, 1409, 2100])
@pytest.mark.parametrize("K,N", [(264, 4100), (512, 9000), (256, 16388)])
def test_many_token_blocks_against_64_bits(T, K, N):
    m, g = _layer(K, N, T + N, False)
    _check(m, torch.randn(T, K, generator=g, device="cuda"))


# K in and out of whole quads of 256 columns, N at and off the 128-column blocks, other pitches (odd ones with columns left over), wide rows (row pass of
# its own beyond 16384); at the largest T all of them take the matrix cores, whole quads with an odd pitch the general kernel
@pytest.mark.parametrize("K,N,pitch", [(8, 4372, 0), (248, 1004, 0), (264, 2052, 0), (1376, 4100, 0), (512, 128, 16), (512, 128, 3), (1000, 3004, 3), (520, 12292, 1),
                                       (256, 16384, 0), (256, 16388, 0), (13824, 5120, 0)])
@pytest.mark.parametrize("T", [3, 70, 1030])
def test_columns_against_64_bits(T, K, N, pitch):
    m, g = _layer(K, N, K + N, True, pitch)
    _check(m, torch.randn(T, K, generator=g, device="cuda"))


@pytest.mark.parametrize("T", [731, 1500])
def test_whole_tiles_and_split_rest(T):
    m, g = _layer(4096, 11008, T, False)
    x = torch.randn(T, 4096, generator=g, device="cuda")
    x[:, ::512] *= 64
    _check(m, x)


def test_magnitudes_and_non_finite():
    """Wide ranges inside a row are summed exactly as far as float32 carries them; infinities and NaN reach what they reach in float32."""
    m, g = _layer(1024, 256, 3, False)
    x = torch.randn(140, 1024, generator=g, device="cuda") * torch.exp2(torch.randint(-30, 30, (140, 1024), generator=g, device="cuda").float())
    x[7] *= 1e-20
    x[8] *= 1e6           # (2^30 1e6 squared, times a hundred of them: the LayerNorm's sum of squares stays below float32's 3.4e38)
    _check(m, x)
    m.layernorm = nn.Identity()
    m.weight_scale.data.fill_(1.0)
    m.input_factor.data.fill_(1.0)
    x = torch.randn(140, 1024, generator=g, device="cuda")
    x[3, 5], x[4, 6], x[5, 7], x[6, 8] = float("inf"), float("-inf"), float("nan"), 3.0e38
    u, s = m(x), _signs(m)
    assert torch.equal(u[3], s[:, 5].float() * float("inf")) and torch.equal(u[4], -s[:, 6].float() * float("inf"))
    assert u[5].isnan().all() and torch.equal(u[6], s[:, 8].float() * x[6, 8])
    keep = [i for i in range(140) if i not in (3, 4, 5, 6)]
    assert torch.isfinite(u[keep]).all()


@pytest.mark.parametrize("T,K,N", [(11000, 8200, 132), (22500, 4096, 260), (48, 1900000, 20)])
def test_portions_of_bounded_scratch(T, K, N):
    """Scratch memory does not grow with the rows beyond 512 MB of parts; portions of rows, the last one shorter and split otherwise, are the same layer."""
    from onebit_amd import _lib
    ws = lambda t: _lib.load().onebit_linear_workspace_bytes(t, K, N, _lib.ONEBIT_F32)
    rest = 40 * 2 ** 20 + N * (K + 256) // 8             # sums of split K, packed rows with columns left over
    assert T * K * 6 > 2 ** 29 and 0 < ws(T) <= 2 ** 29 + rest and ws(20 * T) <= 2 ** 29 + rest
    m, g = _layer(K, N, T, True)
    _check(m, torch.randn(T, K, generator=g, device="cuda"))


def test_partial_sums_of_a_k_shard_take_no_scratch(monkeypatch):
    from onebit_amd.sharded import hip_partial, shard_k
    T, K, N = 64, 1024, 1000
    m, g = _layer(K, N, 4, False)
    x = torch.randn(T, K, generator=g, device="cuda")
    parts, empty, asked = [], torch.empty, []

    def count(*a, dtype=None, **k):
        if dtype == torch.uint8:
            asked.append(a)
        return empty(*a, dtype=dtype, **k)
    monkeypatch.setattr(torch, "empty", count)
    for r in range(2):
        sh = shard_k(m.weight.data, m.input_factor.data, m.weight_scale.data, None, r, 2)
        parts.append(hip_partial(sh, x[:, sh.k0:sh.k1]))
    assert not asked
    z = (x * m.input_factor).double() @ _signs(m).T
    assert float((sum(parts).double() - z).norm() / z.norm()) < 1e-6


def test_without_memory_for_scratch(monkeypatch):
    """No room for the scratch memory: the general kernel, which needs none, as before there was any."""
    T, K, N = 70, 1376, 4100
    m, g = _layer(K, N, 2, True)
    x = torch.randn(T, K, generator=g, device="cuda")
    y, empty = m(x), torch.empty

    def full(*a, dtype=None, **k):
        if dtype == torch.uint8:
            raise torch.OutOfMemoryError("full")
        return empty(*a, dtype=dtype, **k)
    monkeypatch.setattr(torch, "empty", full)
    np.testing.assert_allclose(m(x).cpu().numpy(), y.cpu().numpy(), rtol=0, atol=2e-5)


def test_workspace_of_the_promised_alignment():
    """16 bytes, as the header promises: the same kernels (bit for bit) as with the module's."""
    from onebit_amd import _lib
    from onebit_amd.bitnet import _stream_ptr
    for T, K, N in ((64, 1024, 1000), (20, 1376, 4100)):
        m, g = _layer(K, N, 1, True)
        x = torch.randn(T, K, generator=g, device="cuda")
        y, n = torch.empty(T, N, device="cuda"), _lib.load().onebit_linear_workspace_bytes(T, K, N, _lib.ONEBIT_F32)
        ws = torch.empty(n + 16, dtype=torch.uint8, device="cuda")
        assert _lib.load().onebit_linear_forward(m.weight.data_ptr(), m.weight.stride(0), x.data_ptr(), m.input_factor.data_ptr(), m.weight_scale.data_ptr(),
                                                 m.bias.data_ptr(), y.data_ptr(), None, ws.data_ptr() + 16, n, T, K, N, _lib.ONEBIT_F32, 1e-5, 0,
                                                 _stream_ptr(x.device)) == 0
        assert torch.equal(y, m(x))


def test_small_workspace_keeps_the_general_path():
    """A caller without the workspace is served as before, by the same numbers up to the order of additions."""
    from onebit_amd import _lib
    from onebit_amd.bitnet import _stream_ptr
    T, K, N = 64, 1024, 1000
    m, g = _layer(K, N, 1, False)
    x = torch.randn(T, K, generator=g, device="cuda")
    y = torch.empty(T, N, device="cuda")
    assert _lib.load().onebit_linear_workspace_bytes(T, K, N, _lib.ONEBIT_F32) > 0
    rc = _lib.load().onebit_linear_forward(m.weight.data_ptr(), m.weight.stride(0), x.data_ptr(), m.input_factor.data_ptr(), m.weight_scale.data_ptr(), None,
                                           y.data_ptr(), None, None, 0, T, K, N, _lib.ONEBIT_F32, 1e-5, 0, _stream_ptr(x.device))
    assert rc == 0
    np.testing.assert_allclose(y.cpu().numpy(), m(x).cpu().numpy(), rtol=0, atol=2e-5)
