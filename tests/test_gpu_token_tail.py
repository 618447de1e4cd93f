"""One token through ``BitLinearInf`` in one launch (ob_decode.h, TAIL) against the two launches that a captured call still takes: the same bits at the edges of its
tiles, of its 2048-element rounds and of its widths, on many streams and threads at once, and behind each other on one."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _layer(K, N, seed, bias=False):
    from onebit_amd import BitLinearInf
    g = torch.Generator(device=DEV).manual_seed(seed)
    m = BitLinearInf(K, N, bias=bias, device=DEV, dtype=torch.float16)
    m.weight.data = torch.randint(0, 256, (N, K // 8), generator=g, device=DEV, dtype=torch.uint8).view(torch.int8)
    m.input_factor.data = (0.05 + 0.1 * torch.rand(K, generator=g, device=DEV)).half()
    m.weight_scale.data = (0.05 + 0.1 * torch.rand(N, generator=g, device=DEV)).half()
    if bias:
        m.bias.data = torch.randn(N, generator=g, device=DEV).half()
    return m, torch.randn(1, K, generator=g, device=DEV).half()


def _captured(m, x):
    m(x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.no_grad(), torch.cuda.graph(graph):
        y = m(x)
    graph.replay()
    torch.cuda.synchronize()
    return y


@pytest.mark.parametrize("K", [128, 512, 4096, 5120, 8192, 11008, 16384])
@pytest.mark.parametrize("N", [8, 24, 1000, 2048, 2056, 4096, 11008, 16384])
def test_one_launch_equals_two(K, N):
    for bias in (False, True):
        m, x = _layer(K, N, K + N, bias)
        ref = _captured(m, x)
        for _ in range(9):                                            # (slots of tickets, taken in turn)
            assert torch.equal(m(x), ref)
        x[0, K // 2] = float("nan")                                   # ... and the NaN of the whole row
        assert bool(torch.isnan(m(x)).all())


def test_streams_beside_each_other():
    """Calls of different layers in flight on many streams, eager and replayed ones on the same stream."""
    layers = [_layer(K, N, i, bool(i & 1)) for i, (K, N) in enumerate([(4096, 4096), (4096, 11008), (11008, 4096), (512, 16), (2048, 5632)])]
    refs = [_captured(m, x) for m, x in layers]
    streams = [torch.cuda.Stream() for _ in range(40)]
    out = []
    for r in range(6):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                m, x = layers[(i + r) % 5]
                out.append(((i + r) % 5, m(x)))
    torch.cuda.synchronize()
    assert all(torch.equal(y, refs[i]) for i, y in out)
    graph, (m, x) = torch.cuda.CUDAGraph(), layers[0]
    with torch.no_grad(), torch.cuda.graph(graph):
        yg = m(x)
    for _ in range(4):
        yg.zero_()
        graph.replay()
        y = m(x)
        graph.replay()
        assert torch.equal(y, refs[0]) and torch.equal(yg, refs[0])


def test_threads_of_one_stream_and_of_their_own():
    layers = [_layer(4096, n, n) for n in (4096, 11008, 1024, 64)]
    refs, bad = [_captured(m, x) for m, x in layers], []

    def work(i, stream):
        m, x = layers[i]
        with torch.cuda.stream(stream):
            ys = [m(x) for _ in range(200)]
        stream.synchronize()
        bad.extend(1 for y in ys if not torch.equal(y, refs[i]))

    for streams in ([torch.cuda.current_stream()] * 4, [torch.cuda.Stream() for _ in range(4)]):
        torch.cuda.synchronize()
        ts = [threading.Thread(target=work, args=(i, s)) for i, s in enumerate(streams)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
    assert not bad


# workgroups that draw from one counter (32 at most), one more, a last group of one and of all, and where groups grow (512 workgroups, 528, 1024)
@pytest.mark.parametrize("K,N", [(512, 512), (512, 528), (4096, 16 * 48), (4096, 16 * 49), (4096, 4080), (8192, 16384), (11008, 16 * 513), (11008, 16 * 528), (16384, 16384)])
def test_groups_of_tickets(K, N):
    m, x = _layer(K, N, K + N)
    ref = _captured(m, x)
    ys = [m(x) for _ in range(70)]                                    # (every slot, both of its sets)
    torch.cuda.synchronize()
    assert all(torch.equal(y, ref) for y in ys)


def _launches(f):
    """Kernels that ``f`` launches."""
    from torch.profiler import ProfilerActivity, profile
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        f()
        torch.cuda.synchronize()
    return sum(e.count for e in prof.key_averages() if "ob_" in e.key)


def test_one_launch_on_the_fiftieth_stream():
    """What a call took is given back when it ends, whatever becomes of its stream."""
    import ctypes
    hip, streams = ctypes.CDLL("libamdhip64.so"), []
    m, x = _layer(4096, 4096, 1)
    ref = _captured(m, x)
    assert _launches(lambda: m(x)) == 1
    for i in range(50):
        h = ctypes.c_void_p()
        assert hip.hipStreamCreateWithFlags(ctypes.byref(h), 1) == 0              # (non-blocking)
        streams.append(h)
        with torch.cuda.stream(torch.cuda.ExternalStream(h.value)):
            y = m(x)
            if i == 49:
                assert _launches(lambda: m(x)) == 1
        torch.cuda.synchronize()
        assert torch.equal(y, ref)
    for h in streams:
        assert hip.hipStreamDestroy(h) == 0


def test_far_ahead_of_the_device():
    """More calls waiting on a stream than there are slots, and calls on another stream beside them: all right, and the slots are back afterwards."""
    layers = [_layer(K, N, i, bool(i & 1)) for i, (K, N) in enumerate([(4096, 4096), (8192, 16384), (16384, 16384), (512, 16), (4096, 520)])]
    refs = [_captured(m, x) for m, x in layers]
    other = torch.cuda.Stream()
    for _ in range(3):
        torch.cuda._sleep(20_000_000)
        out = []
        for i in range(90):
            m, x = layers[i % 5]
            out.append((i % 5, m(x)))
        with torch.cuda.stream(other):
            for i in range(90):
                m, x = layers[i % 5]
                out.append((i % 5, m(x)))
        torch.cuda.synchronize()
        assert all(torch.equal(y, refs[i]) for i, y in out)
    assert [_launches(lambda: m(x)) for m, x in layers] == [1] * 5
