"""The float32 train-mode layer on bf16 matrix products (csrc/ob_train32.h) against the same sums in 64 bits: edges of tiles, rows and columns that are no multiples
of anything, every form of the products, the smallest shapes."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _case(T, K, N, seed, gscale=1.0):
    from onebit_amd.train import BitLinear
    g = torch.Generator(device=DEV).manual_seed(seed)
    m = BitLinear(K, N, bias=True, device=DEV, dtype=torch.float32)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    with torch.no_grad():
        m.weight.copy_(0.02 * r(N, K))
        m.weight[0, :3] = 0.0
        m.weight_scale.copy_(0.1 * r(N)), m.input_factor.copy_(0.1 * r(K)), m.bias.copy_(r(N))
    x = r(T, K)
    x[:, ::512] *= 8
    return m, x.requires_grad_(True), gscale * r(T, N)


def _exact(m, x, gy):
    w, g, h, x, gy = (t.detach().double() for t in (m.weight, m.weight_scale, m.input_factor, x, gy))
    s, a = torch.sign(w), x * h
    z = a @ s.T
    u = z * g
    c = u - u.mean(-1, keepdim=True)
    r = 1 / (c.square().mean(-1, keepdim=True) + 1e-5).sqrt()
    y = c * r
    gu = r * (gy - gy.mean(-1, keepdim=True) - y * (gy * y).mean(-1, keepdim=True))
    gz = gu * g
    ga = gz @ s
    return y + m.bias.detach().double(), ga * h, (gz.T @ a) * (1.001 - torch.tanh(w) ** 2), (gu * z).sum(0), (ga * x).sum(0), gy.sum(0)


# Norms of the differences: a sum of n float32 terms is off by 2^-24 sqrt(n) / 4 of the terms' norm and less (32 at a time are added for one rounding), n is 13824
# at most here, and a handful of element-wise roundings precede and follow it; a gradient's terms partly cancel (the LayerNorm takes the mean out), a factor of 4.
def _check(got, want, n):
    for name, a, b in zip(("y", "x", "weight", "weight_scale", "input_factor", "bias"), got, want):
        off = float((a.detach().double() - b).norm() / b.norm().clamp_min(1e-300))
        assert off <= 2.0 ** -22 * (4 + n ** 0.5 / 4), (name, off)


@pytest.mark.parametrize("T,K,N", [(5, 24, 8), (33, 1000, 1000), (64, 1024, 1000), (97, 1027, 1030), (257, 1376, 4100), (300, 2080, 516),      # few tiles
                                   (129, 13824, 128), (1100, 4096, 2050), (2100, 2049, 3070)])                                              # 128 x 256, 256 x 256 tiles, odd widths
def test_layer_and_gradients_against_64_bits(T, K, N):
    m, x, gy = _case(T, K, N, T + K)
    y = m(x)
    got = (y, *torch.autograd.grad(y, [x, m.weight, m.weight_scale, m.input_factor, m.bias], gy))
    _check(got, _exact(m, x, gy), max(T, K, N))
    y = m(x)
    again = (y, *torch.autograd.grad(y, [x, m.weight, m.weight_scale, m.input_factor, m.bias], gy))
    assert all(torch.equal(a, b) for a, b in zip(got, again))


def test_gradients_of_any_magnitude():
    """The parts are exact from 2^-110 on: gradients of 1e-20 and 1e20 are as close as those of 1."""
    for scale in (1e-20, 1e20):
        m, x, gy = _case(130, 1024, 1000, 7, scale)
        y = m(x)
        _check((y, *torch.autograd.grad(y, [x, m.weight, m.weight_scale, m.input_factor, m.bias], gy)), _exact(m, x, gy), 1024)


def test_forward_without_workspace_and_special_values(monkeypatch):
    """Without memory the forward takes the kernel that needs none; an infinite activation makes its row NaN and no other; NaN weights have no sign."""
    T, K, N = 200, 1024, 1000
    m, x, _ = _case(T, K, N, 9)
    full, empty = m(x.detach()).detach(), torch.empty

    def none_left(*a, dtype=None, **k):
        if dtype == torch.uint8:
            raise torch.OutOfMemoryError("full")
        return empty(*a, dtype=dtype, **k)
    with monkeypatch.context() as p:
        p.setattr(torch, "empty", none_left)
        # (z of the float32 instruction: K / 4 roundings)
        assert float((m(x.detach()).detach() - full).norm() / full.norm()) <= 2.0 ** -22 * (4 + K ** 0.5)
    xs = x.detach().clone()
    xs[17, 5] = float("inf")
    with torch.no_grad():
        m.weight[3, 7] = float("nan")
    y = m(xs).detach()
    assert torch.isnan(y[17]).all() and torch.isfinite(y[:17]).all() and torch.isfinite(y[18:]).all()
    with torch.no_grad():
        m.weight[3, 7] = 0.0
    assert torch.equal(m(x.detach())[:17], y[:17])


def test_workspaces_are_bounded():
    from onebit_amd import _lib
    lib, f32 = _lib.load(), _lib.ONEBIT_F32
    fw, bw = lib.onebit_train_forward_workspace_bytes, lib.onebit_train_workspace_bytes
    assert fw(60, 1024, 1000, f32) == 0 and fw(64, 1024, 1000, f32) > 0
    assert fw(400000, 4096, 1000, f32) <= 2 ** 29 + 2 * 1024 * 4096 and fw(4096, 4096, 4096, f32) == (6 + 2) * 4096 * 4096
    assert bw(4096, 4096, 11008, f32) < 1.05 * 6 * 4096 * (4096 + 11008)


@pytest.mark.parametrize("T,K,N", [(64, 4096, 1000), (128, 2081, 4100), (129, 8200, 260), (257, 1030, 2050), (600, 4096, 1030), (100, 530, 8216)])
def test_products_in_slices_of_their_steps(T, K, N):
    """Few output tiles and a long sum (csrc/onebit_train.hip, ob_train_plan): every slice walks all pairs of parts."""
    test_layer_and_gradients_against_64_bits(T, K, N)


def _backward(T, K, N, dtype, nbytes, seed=5):
    """Gradients of the layer of _case(T, K, N, seed) in `dtype` through the C entry with `nbytes` of workspace, between two rows of 7s."""
    from onebit_amd import _lib
    lib, code = _lib.load(), _lib.ONEBIT_F32 if dtype == torch.float32 else _lib.ONEBIT_F16
    m, x, gy = _case(T, K, N, seed)
    w, h, g, x, gy = (t.detach().to(dtype).contiguous() for t in (m.weight, m.input_factor, m.weight_scale, x, gy))
    z, y, stats = torch.empty(T, N, dtype=dtype, device=DEV), torch.empty(T, N, dtype=dtype, device=DEV), torch.empty(T, 2, device=DEV)
    fw = torch.empty(max(1, lib.onebit_train_forward_workspace_bytes(T, K, N, code)), dtype=torch.uint8, device=DEV)
    out = [torch.empty(s, dtype=dtype, device=DEV) for s in ((T, K), (N, K), (K,), (N,), (N,))]
    ws = torch.full((nbytes + 512,), 7, dtype=torch.uint8, device=DEV)
    p, s = (lambda t: t.data_ptr()), torch.cuda.current_stream().cuda_stream
    _lib.check(lib.onebit_train_forward_ws(p(x), p(w), p(h), p(g), None, p(y), p(z), p(stats), p(fw), fw.numel(), T, K, N, code, 1e-5, s), "forward")
    _lib.check(lib.onebit_train_backward(p(gy), p(x), p(w), p(h), p(g), p(z), p(stats), *(p(o) for o in (out[0], out[1], out[2], out[3], out[4])),
                                         p(ws) + 256, nbytes, T, K, N, code, s), "backward")
    assert (ws[:256] == 7).all() and (ws[256 + nbytes:] == 7).all()
    gx, gw, gh, gg, gb = (o.float() for o in out)
    return m, x, gy, (gx, gw, gg, gh, gb)


# (the sums of the float32 instruction: a rounding every four terms)
@pytest.mark.parametrize("T,K,N", [(5, 24, 8), (33, 1000, 1000), (97, 1027, 1030), (257, 1376, 4100), (64, 4096, 1000), (1100, 516, 2050)])
def test_backward_with_the_least_workspace(T, K, N):
    from onebit_amd import _lib
    lib = _lib.load()
    need, least = (f(T, K, N, _lib.ONEBIT_F32) for f in (lib.onebit_train_workspace_bytes, lib.onebit_train_least_workspace_bytes))
    assert least < need and least <= 4 * T * (K + N) + 8 * T + 128 * max(2 * N, K) + 1024
    m, x, gy, got = _backward(T, K, N, torch.float32, least)
    n = max(T, K, N)
    for name, a, b in zip(("x", "weight", "weight_scale", "input_factor", "bias"), got, _exact(m, x, gy)[1:]):
        off = float((a.double() - b).norm() / b.norm().clamp_min(1e-300))
        assert off <= 2.0 ** -22 * (4 + n ** 0.5), (name, off)
    assert lib.onebit_train_backward(*[256] * 13, least - 1, T, K, N, _lib.ONEBIT_F32, None) == -5


# few rows, whose products run in slices given the room: one slice in what is left without it
@pytest.mark.parametrize("T,K,N", [(64, 1000, 4096), (129, 260, 8200)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_backward_without_room_for_slices(T, K, N, dtype):
    from onebit_amd import _lib
    lib, code = _lib.load(), _lib.ONEBIT_F32 if dtype == torch.float32 else _lib.ONEBIT_F16
    need = lib.onebit_train_workspace_bytes(T, K, N, code)
    one = lib.onebit_train_least_workspace_bytes(T, K, N, code) if dtype == torch.float16 else need - 1
    assert one < need
    full, less = _backward(T, K, N, dtype, need)[3], _backward(T, K, N, dtype, one)[3]
    for a, b in zip(full, less):
        # sums in another order; float16: and the roundings of ga to it
        assert float((a - b).norm() / b.norm()) <= (2.0 ** -22 * (4 + max(T, K, N) ** 0.5) if dtype == torch.float32 else 2.0 ** -9)


def test_backward_without_memory_takes_the_least_workspace(monkeypatch):
    T, K, N = 97, 1027, 1030
    from onebit_amd import _lib
    least = _lib.load().onebit_train_least_workspace_bytes(T, K, N, _lib.ONEBIT_F32)
    m, x, gy = _case(T, K, N, 6)
    y, empty = m(x), torch.empty

    def little_left(*a, dtype=None, **k):
        if dtype == torch.uint8 and a[0] > least:
            raise torch.OutOfMemoryError("full")
        return empty(*a, dtype=dtype, **k)
    monkeypatch.setattr(torch, "empty", little_left)
    got = torch.autograd.grad(y, [x, m.weight, m.weight_scale, m.input_factor, m.bias], gy)
    for a, b in zip(got, _exact(m, x, gy)[1:]):
        assert float((a.double() - b).norm() / b.norm()) <= 2.0 ** -22 * (4 + K ** 0.5)


# the straight-through factor alone: the gradient over that of a layer of the same signs whose weights' factor is 1.001f
@pytest.mark.parametrize("lo,hi,rms,most", [(0, 0.02, 5.8e-8, 1.1e-7), (0.1, 0.25, 5.0e-8, 1.1e-7), (0.25, 0.5, 5.2e-8, 1.3e-7), (0.5, 0.8, 6.7e-8, 2.1e-7), (0.8, 1.0, 7.5e-8, 2.2e-7),
                                            (1.0, 2.5, 8.2e-8, 2.4e-7), (2.5, 9.0, 9.1e-8, 2.6e-7)])
def test_straight_through_factor_against_64_bits(lo, hi, rms, most):
    """Errors of 1.001f - tanhf(w)^2 (root mean square, largest) are the bounds, and either gradient's rounding (half an ulp at most, 0.42 in the mean square)."""
    from onebit_amd.train import BitLinear
    T, K, N = 64, 1024, 1000
    g = torch.Generator(device=DEV).manual_seed(3)
    w = lo + (hi - lo) * torch.rand(N, K, generator=g, device=DEV)
    x, gy = torch.randn(T, K, generator=g, device=DEV), torch.randn(T, N, generator=g, device=DEV)
    out = []
    for latent in (w, torch.full_like(w, 1e-30)):                      # the same signs: the same gz and a
        m = BitLinear(K, N, device=DEV, dtype=torch.float32)
        with torch.no_grad():
            m.weight.copy_(latent), m.weight_scale.fill_(1.0), m.input_factor.fill_(1.0)
        out.append(torch.autograd.grad(m(x), m.weight, gy)[0].double())
    base = out[1] / float(torch.tensor(1.001, dtype=torch.float32))
    keep = base.abs() > 1e-3 * base.abs().mean()
    f = (1.001 - torch.tanh(w.double()) ** 2)[keep]
    off, room = (out[0] / base)[keep] - f, 2.0 ** -24 * f
    assert float((off.abs() - 2 * room).max()) <= most, float((off.abs() - 2 * room).max())
    assert float(off.square().mean().sqrt()) <= (rms ** 2 + 2 * float((0.45 * room).square().mean())) ** 0.5, float(off.square().mean().sqrt())
