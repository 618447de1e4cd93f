"""The float16 train-mode layer (csrc/ob_train16.h) against the same formulas in 64 bits, at the edges of its 16- and 32-element tiles, 128-row and
128- / 256-column blocks (64 to 256 x 256 where they are more than the CUs: all three products at 4100 x 8200 x 8216, one or two each at the sizes after it), with rows
that are not 16-byte aligned.

Bound: every tensor-level result is rounded to float16 (2^-11 relative) once per operation, at most five of them in a row (x h, z, u, gz, ga,
gx); roundings of a sum's addends are independent.  A row or column of a result may therefore be off by about 5 x 2^-11 = 2.4e-3 of its 2-norm at the
very most; 4e-3 is asserted of every single row and column (a lost or doubled tile, row or column shows as 1e-1 and more)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _exact(x, w, h, g, gy):
    x, w, h, g, gy = (t.double() for t in (x, w, h, g, gy))
    s, a = torch.sign(w), x * h
    z = a @ s.T
    u = z * g
    c = u - u.mean(-1, keepdim=True)
    r = 1 / (c.square().mean(-1, keepdim=True) + 1e-5).sqrt()
    y = c * r
    gu = r * (gy - gy.mean(-1, keepdim=True) - y * (gy * y).mean(-1, keepdim=True))
    gz = gu * g
    ga = gz @ s
    return y, ga * h, (gz.T @ a) * (1.001 - torch.tanh(w) ** 2), (gu * z).sum(0), (ga * x).sum(0), gy.sum(0)


def _off(got, ref):
    """The worst row's or column's error, over its norm (or over the typical one, for those that are small by chance)."""
    d, worst = got.detach().double() - ref, 0.0
    if ref.dim() == 1:
        return float(d.norm() / ref.norm())
    for dim in (0, 1):
        n = ref.norm(dim=dim)
        worst = max(worst, float((d.norm(dim=dim) / n.clamp_min(float(n.detach().median()))).max()))
    return worst


def _case(T, K, N, seed, shift=0):
    from onebit_amd.train import BitLinear
    g = torch.Generator(device=DEV).manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    odd = lambda t: torch.cat([t.new_zeros(shift), t.reshape(-1)])[shift:].view(t.shape)      # the same values, `shift` elements off the alignment
    m = BitLinear(K, N, bias=True, device=DEV, dtype=torch.float16)
    m.weight.data = odd((0.3 * rnd(N, K)).half())
    m.weight.data[0, :2] = 0
    m.weight_scale.data = odd((0.05 + 0.1 * torch.rand(N, generator=g, device=DEV)).half())
    m.input_factor.data = odd((0.05 + 0.1 * torch.rand(K, generator=g, device=DEV)).half())
    m.bias.data = odd((0.1 * rnd(N)).half())
    return m, odd(rnd(T, K).half()).requires_grad_(True), odd((0.05 * rnd(T, N)).half())


@pytest.mark.parametrize("T,K,N,shift", [
    (1, 32, 64, 0), (31, 33, 32, 0), (32, 64, 31, 0), (33, 31, 130, 0), (127, 160, 129, 0), (128, 256, 256, 0), (129, 257, 255, 0),
    (200, 1376, 1000, 0), (65, 2050, 1028, 3), (300, 264, 520, 1), (4100, 512, 2056, 0), (1030, 4096, 4160, 0), (96, 1024, 16392, 0),
    (1, 256, 130, 0), (33, 259, 129, 1), (129, 513, 33, 0),                                              # (smaller ones: the forward of two launches)
    (4100, 8200, 8216, 0), (8200, 200, 8216, 0), (8216, 8200, 40, 0), (40, 8216, 8200, 1),              # 256-column blocks, sums of 2-7 steps of 32
    # one operand straight to registers, 64 / 128 / 256 of the other's: last blocks part-filled, sums of 1 to 4 turns of steps and every remainder
    (1300, 4100, 2300, 0), (2056, 2056, 4104, 1), (1930, 2081, 3000, 3), (31, 4104, 4200, 0), (4500, 33, 2500, 0), (4500, 96, 2500, 0), (4500, 130, 2056, 0),
    (4500, 260, 2056, 1), (3000, 4096, 300, 0), (5000, 4096, 33, 0), (1281, 5000, 1500, 0)])
def test_rows_and_columns_against_64_bits(T, K, N, shift):
    m, x, gy = _case(T, K, N, T + K + N, shift)
    y = m(x)
    got = torch.autograd.grad(y, [x, m.weight, m.weight_scale, m.input_factor, m.bias], gy)
    ref = _exact(x.detach(), m.weight.detach(), m.input_factor.detach(), m.weight_scale.detach(), gy)
    assert _off(y - m.bias.detach(), ref[0]) <= 4e-3
    for i, t in enumerate(got):
        assert t.dtype == torch.float16 and _off(t, ref[1 + i]) <= 4e-3, (i, _off(t, ref[1 + i]))
    again = torch.autograd.grad(m(x), [x, m.weight, m.weight_scale, m.input_factor, m.bias], gy)
    assert all(torch.equal(a, b) for a, b in zip(got, again))


def test_forward_without_workspace_is_the_same_layer():
    from onebit_amd import _lib
    from onebit_amd.bitnet import _stream_ptr
    T, K, N = 77, 328, 264
    m, x, _ = _case(T, K, N, 5)
    y, z, st = (torch.empty(s, dtype=d, device=DEV) for s, d in (((T, N), torch.float16), ((T, N), torch.float16), ((T, 2), torch.float32)))
    lib = _lib.load()
    assert lib.onebit_train_forward_workspace_bytes(T, K, N, _lib.ONEBIT_F16) > 0 and lib.onebit_train_forward_workspace_bytes(T, K, N, _lib.ONEBIT_F32) == 0
    p = lambda t: t.detach().data_ptr()
    assert lib.onebit_train_forward(p(x), p(m.weight), p(m.input_factor), p(m.weight_scale), p(m.bias), p(y), p(z), p(st), T, K, N, _lib.ONEBIT_F16, 1e-5,
                                    _stream_ptr(y.device)) == 0
    # (sums in another order: a float16 of z may fall one ulp apart, 2^-11 of it)
    assert _off(y, m(x).detach().double()) <= 2e-3


def test_scratch_memory_is_bounded_and_optional(monkeypatch):
    """The forward's scratch does not grow with the rows beyond 512 MB of them (portions are the same layer); the backward's holds one matrix of the layer
    beside the output's gradient; without memory the forward runs without."""
    from onebit_amd import _lib
    T, K, N = 35000, 8200, 136
    lib = _lib.load()
    fw, bw = lib.onebit_train_forward_workspace_bytes, lib.onebit_train_workspace_bytes
    assert T * K * 2 > 2 ** 29 and fw(T, K, N, _lib.ONEBIT_F16) <= 2 ** 29 + 2 * 160 * 8224 and fw(9 * T, K, N, _lib.ONEBIT_F16) <= 2 ** 29 + 2 * 160 * 8224
    assert bw(4096, 4096, 11008, _lib.ONEBIT_F16) < 1.05 * 2 * 11008 * (4096 + 4096)
    m, x, _ = _case(T, K, N, 3)
    y = m(x.detach())
    s, a = torch.sign(m.weight.detach()).float(), (x.detach() * m.input_factor.detach()).float()
    u = (a @ s.T).half() * m.weight_scale.detach()
    ref = torch.nn.functional.layer_norm(u.double(), (N,)) + m.bias.detach().double()
    assert _off(y, ref) <= 4e-3
    T, K, N = 300, 520, 264
    m, x, gy = _case(T, K, N, 4)
    full, empty = m(x.detach()), torch.empty

    def none_left(*a, dtype=None, **k):
        if dtype == torch.uint8:
            raise torch.OutOfMemoryError("full")
        return empty(*a, dtype=dtype, **k)
    monkeypatch.setattr(torch, "empty", none_left)
    assert _off(m(x.detach()), full.detach().double()) <= 2e-3


def test_small_products_ask_for_no_workspace():
    from onebit_amd import _lib
    ws = lambda *s: _lib.load().onebit_train_forward_workspace_bytes(*s, _lib.ONEBIT_F16)
    assert not any((ws(1, 64, 64), ws(2048, 64, 64), ws(64, 128, 128), ws(4096, 256, 64), ws(1, 255, 4096)))
    assert all((ws(1, 256, 128), ws(1, 512, 32), ws(8192, 128, 128), ws(4096, 4096, 11008)))


def test_sign_and_straight_through_factor_at_special_weights():
    """sign(0) = sign(-0) = 0, NaN has no sign; the factor 1.001 - tanh(w)^2 from tiny to saturated weights, with its float16 roundings."""
    from onebit_amd.train import BitLinear
    K, N, T = 64, 32, 32
    m = BitLinear(K, N, device=DEV, dtype=torch.float16)
    w = torch.tensor([0.0, -0.0, 6e-8, -6e-8, 1e-3, 0.02, -0.3, 1.0, -2.5, 5.0, 60000.0, -60000.0, float("inf"), float("-inf"), 0.5, 4.0], device=DEV).half()
    m.weight.data = w.repeat(N * K // 16).view(N, K)
    x = torch.randn(T, K, generator=torch.Generator(device=DEV).manual_seed(0), device=DEV).half()
    gy = torch.randn(T, N, generator=torch.Generator(device=DEV).manual_seed(1), device=DEV).half()
    m.weight_scale.data = torch.linspace(0.5, 1.5, N, device=DEV).half()
    m.weight.data[::2] *= -1                       # (not every row of sums alike)
    y = m(x)
    gw, = torch.autograd.grad(y, [m.weight], gy)
    t = torch.tanh(m.weight.detach())
    # (1.001 as a float16, 1.0009766, as the layer has always had it: what is left of a saturated weight's factor is 2^-10)
    factor = (torch.tensor(1.001).half().float().to(DEV) - (t ** 2).float()).half().double()
    gs = _exact(x, m.weight.detach().nan_to_num(), m.input_factor.detach(), m.weight_scale.detach(), gy)
    z = (x.double() @ torch.sign(m.weight.detach().double()).T)
    u = z * m.weight_scale.detach().double()
    c = u - u.mean(-1, keepdim=True)
    r = 1 / (c.square().mean(-1, keepdim=True) + 1e-5).sqrt()
    gu = r * (gy.double() - gy.double().mean(-1, keepdim=True) - c * r * (gy.double() * c * r).mean(-1, keepdim=True))
    ref = ((gu * m.weight_scale.detach().double()).T @ x.double()) * factor
    # one float16 ulp of the factor near 1 (2^-11), the roundings of gz and of the products
    assert ((gw.double() - ref).abs() <= 4e-3 * ref.abs() + 4e-3 * ref.abs().mean() * factor).all()
    assert _off(y, gs[0]) <= 4e-3


@pytest.mark.parametrize("T,K,N,shift", [(1, 4096, 256, 0), (64, 4096, 1000, 0), (128, 2081, 4100, 1), (129, 8200, 260, 0), (257, 1030, 2050, 3), (600, 4096, 1030, 0),
                                         (100, 530, 8216, 0)])
def test_products_in_slices_of_their_steps(T, K, N, shift):
    """Few output tiles and a long sum (csrc/onebit_train.hip, ob_train_plan): ragged slices, rows and columns, 128 x 128 and 128 x 256 tiles."""
    from onebit_amd import _lib
    up = lambda n: -(-n // 32) * 32
    lib, f16 = _lib.load(), _lib.ONEBIT_F16
    sliced = (lib.onebit_train_forward_workspace_bytes(T, K, N, f16) > 2 * up(K) * (up(T) + up(N)),
              lib.onebit_train_workspace_bytes(T, K, N, f16) > 2 * (max(up(T) * up(K), up(K) * up(N)) + up(T) * up(N)) + 4 * T * K)
    assert any(sliced)
    test_rows_and_columns_against_64_bits(T, K, N, shift)
