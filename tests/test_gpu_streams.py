"""Order between streams: weights re-tiled, forwards, graph replays and split workspaces (run on an MI355X).

Races are provoked by holding one stream up with a long kernel (``torch.cuda._sleep``) while the others go on,
and every result is compared with the same call made alone.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

HOLD = 200_000_000  # cycles of a held stream: 0.1 to 2 s


@pytest.fixture(scope="module")
def cuda(gpu):
    if not torch.cuda.is_available():
        pytest.skip("torch sees no GPU")
    return torch.device("cuda:0")


def module(d_in, d_out, **kw):
    import metal_kans as mk
    np.random.seed(0)
    return mk.TorchMetalKANLinear(d_in, d_out, **kw).to("cuda")


def scale(m, s):
    with torch.no_grad():
        for p in m.parameters():
            p.mul_(s)


def alone(m, x):
    torch.cuda.synchronize()
    y = m(x).clone()
    torch.cuda.synchronize()
    return y


def hip_runtime():
    """The HIP runtime that this process uses."""
    with open("/proc/self/maps") as f:
        paths = {line.split()[-1] for line in f if "libamdhip64" in line}
    assert len(paths) == 1, paths
    return ctypes.CDLL(paths.pop())


def test_destroyed_stream_is_drained(cuda):
    """A stream's handle is taken for the stream: hipStreamDestroy returns when the stream's work is done, so a
    handle that comes back for another stream finds nothing of the old one still running."""
    hip = hip_runtime()
    h = ctypes.c_void_p()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(h), 1) == 0
    done = torch.cuda.Event()
    with torch.cuda.stream(torch.cuda.ExternalStream(h.value)):
        torch.cuda._sleep(HOLD)
        done.record()
    assert not done.query()
    assert hip.hipStreamDestroy(h) == 0
    assert done.query()


def test_retiling_behind_another_streams_forward_keeps_the_host_free(cuda):
    """Weights changed and re-tiled on one stream while a forward of the old ones still waits on another: the
    forward reads the old tiles, and the call that re-tiles does not wait for it on the host."""
    m = module(512, 768, degree=6)
    x = torch.rand(512, 512, device=cuda) * 2 - 1
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.no_grad():
        old = alone(m, x)
        scale(m, 2.0)
        new = alone(m, x)
        scale(m, 0.5)
        torch.cuda.synchronize()
        with torch.cuda.stream(a):
            m(x)
        with torch.cuda.stream(b):
            torch.cuda._sleep(HOLD)
            yb = m(x)
            held = torch.cuda.Event()
            held.record()
        with torch.cuda.stream(a):
            scale(m, 2.0)
            ya = m(x)
        assert not held.query()
    torch.cuda.synchronize()
    assert torch.equal(yb, old) and torch.equal(ya, new)


def test_host_load_behind_a_queued_retiling(cuda):
    """Weights re-tiled on a held stream, then other weights loaded from host arrays: the later load stays."""
    m = module(96, 80, degree=5)
    layer = m.metal_layer
    xh = (np.random.default_rng(0).random((64, 96)) * 2 - 1).astype(np.float32)
    x = torch.from_numpy(xh).to(cuda)
    want = layer(xh)                         # the layer's own arrays
    side = torch.cuda.Stream()
    with torch.no_grad():
        scale(m, 2.0)                        # the module's parameters
        doubled = alone(m, x)
        scale(m, 1.0)                        # (a new version of the same values)
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            torch.cuda._sleep(HOLD)
            y = m(x)                         # its re-tiling waits on the held stream
    first = layer(xh)
    torch.cuda.synchronize()
    assert torch.equal(y, doubled)
    np.testing.assert_array_equal(first, want)
    np.testing.assert_array_equal(layer(xh), want)   # nothing loaded again


def load_on(lib, m, stream, s):
    """The module's weights times s into its layer, on `stream`; returns the arrays, which the load reads."""
    import metal_kans as mk
    ws = [(p.detach() * s).contiguous() for p in (m.weight, m.base_weight, m.bias_param)]
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        torch.cuda._sleep(HOLD)
    mk.device.check(lib.kans_layer_load_weights_stream(m.metal_layer._engine().handle, *[w.data_ptr() for w in ws],
                                                       stream.cuda_stream), "kans_layer_load_weights_stream")
    return ws


@pytest.mark.parametrize("kind", ["chain", "gated"])
def test_graph_replays_follow_a_load_on_another_stream(gpu, cuda, kind):
    """A chain's and a dense gated block's graph, built before, replayed while a load of new weights is still
    queued on a held stream: the result is the new weights'."""
    import metal_kans as mk
    lib = gpu
    dims = ((24, 40), (40, 16)) if kind == "chain" else ((24, 40), (24, 40), (40, 24))
    ms = [module(a, b, degree=4) for a, b in dims]
    with torch.no_grad():
        for m in ms:
            m(torch.zeros(1, m.in_features, device=cuda))   # the handles
    torch.cuda.synchronize()
    handles = [m.metal_layer._engine().handle for m in ms]
    obj = ctypes.c_void_p()
    if kind == "chain":
        arr = (ctypes.c_void_p * 2)(*[h.value for h in handles])
        mk.device.check(lib.kans_chain_create(arr, 2, ctypes.byref(obj)), "kans_chain_create")
        call = lambda x, y: lib.kans_chain_forward_host(obj, x.ctypes.data, y.ctypes.data, len(x))  # noqa: E731
    else:
        mk.device.check(lib.kans_gated_dense_create(*handles, ctypes.byref(obj)), "kans_gated_dense_create")
        call = lambda x, y: lib.kans_gated_dense_forward_host(obj, x.ctypes.data, 0, y.ctypes.data, len(x))  # noqa: E731
    x = (np.random.default_rng(1).random((32, 24)) * 2 - 1).astype(np.float32)

    def forward():
        y = np.empty((32, dims[-1][1]), np.float32)
        mk.device.check(call(x, y), kind)
        return y
    try:
        old = forward()
        side = torch.cuda.Stream()
        keep = load_on(lib, ms[0], side, 0.5)
        new = forward()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(forward(), new)
        assert not np.array_equal(old, new)
        keep += load_on(lib, ms[0], side, 1.0)
        np.testing.assert_array_equal(forward(), old)
    finally:
        torch.cuda.synchronize()
        (lib.kans_chain_destroy if kind == "chain" else lib.kans_gated_dense_destroy)(obj)


def test_forward_without_memory_for_its_splits(cuda):
    """Partial sums larger than the device (550 GB): the forward runs unsplit, with the unsplit forward's bits."""
    m = module(4096, 2048, degree=2, bias=False, use_base=False).half()
    eng = m.metal_layer._engine()
    x = torch.rand(262144, 4096, device=cuda, dtype=torch.float16) * 2 - 1
    with torch.no_grad():
        eng.set_tiling(0, 0, 1)
        want = m(x)
        eng.set_tiling(0, 0, 256)
        assert torch.equal(m(x), want)
        eng.set_tiling(0, 0, 0)
        small = m(x[:64])
    assert torch.isfinite(small).all()


def splits_of(lib, m, B):
    wm, nb, splits = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    assert lib.kans_layer_describe(m.metal_layer._engine().handle, B, ctypes.byref(wm), ctypes.byref(nb),
                                   ctypes.byref(splits)) == 0
    return splits.value


@pytest.mark.parametrize("basis,dtype", [("rbf", torch.float16), ("cheby", torch.float32)])
def test_split_forwards_of_one_layer_on_several_streams(gpu, cuda, basis, dtype):
    """Unordered forwards of a layer whose features are split, on more streams than workspaces are kept for:
    each has partial sums of its own."""
    m = module(1024, 1024, basis=basis, degree=8).to(dtype)
    B, streams = 2048, [torch.cuda.Stream() for _ in range(12)]
    with torch.no_grad():
        xs = [(torch.rand(B, 1024, device=cuda) * 2 - 1).to(dtype) for _ in streams]
        want = [alone(m, x) for x in xs]
        assert splits_of(gpu, m, B) > 1
        for pair in (streams[:2], streams):
            outs = []
            for _ in range(8 if len(pair) == 2 else 1):
                for s, x in zip(pair, xs):
                    with torch.cuda.stream(s):
                        outs.append(m(x))
            torch.cuda.synchronize()
            assert all(torch.equal(y, want[n % len(pair)]) for n, y in enumerate(outs))


def test_captured_split_forward_keeps_its_workspace(gpu, cuda):
    """A forward with split features in a graph: its replays give the eager bits after larger eager forwards (whose
    workspace has grown since) and beside others; the graphs captured once the layer's captured workspaces are
    used up (256 MB) run unsplit."""
    m = module(1024, 1024, basis="rbf", degree=4).half()
    B = 2048
    side, other = torch.cuda.Stream(), torch.cuda.Stream()

    def inputs(n):
        return (torch.rand(n, 1024, device=cuda) * 2 - 1).half()
    with torch.no_grad(), torch.cuda.stream(side):
        x = inputs(B)
        m(x)
        assert splits_of(gpu, m, B) > 1
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            y = m(x)
        big = inputs(3 * B)
        with torch.cuda.stream(other):
            m(big)
        m(big)
        for n in range(4):
            x.copy_(inputs(B))
            side.synchronize()
            graph.replay()
            with torch.cuda.stream(other):
                beside = m(big)
            side.synchronize()
            got = y.clone()
            assert torch.equal(got, m(x)), n
            torch.cuda.synchronize()
            assert torch.equal(beside, m(big)), n
        part = splits_of(gpu, m, B) * B * 1024 * 4
        graphs = []
        for _ in range(256_000_000 // part + 2):
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=side):
                yg = m(x)
            graphs.append((g, yg))
        want = m(x)
        for g, _ in graphs:
            g.replay()
        side.synchronize()
        assert torch.equal(graphs[0][1], want)
        # The same products summed in another order: 1024 * 5 / 16 = 320 matrix steps, each of which rounds a sum of
        # at most S = sum |w| (basis values and SiLU(x) are at most 1 here) to fp32, on either side; then one unit in
        # the last place of fp16.
        S = sum(p.double().abs().reshape(1024, -1).sum(1) for p in m.parameters())
        err = (graphs[-1][1].double() - want.double()).abs()
        assert (err <= 2 * 320 * 2.0 ** -24 * S + 2.0 ** -10 * want.double().abs()).all()


@pytest.mark.parametrize("fmt", ["int4", "ternary"])
def test_split_quantized_prefill_on_several_streams_and_captured(gpu, cuda, fmt):
    """A quantized layer's prefill with split features: unordered on two streams, and captured before the
    workspace of the eager calls grows."""
    from test_gpu_qprefill import make_qlayer
    import metal_kans as mk
    h, _ = make_qlayer(gpu, fmt, 1024, 520, 4, True, True, 3)
    B = 300

    def forward(x, stream):
        with torch.cuda.stream(stream):
            y = torch.empty((x.shape[0], 520), device=cuda)
        mk.device.check(gpu.kans_qlayer_forward(h, x.data_ptr(), 0, 1024, y.data_ptr(), 0, 520, x.shape[0],
                                                stream.cuda_stream), "kans_qlayer_forward")
        return y
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    try:
        xs = [torch.rand(B, 1024, device=cuda) * 2 - 1 for _ in range(2)]
        torch.cuda.synchronize()
        want = []
        for x in xs:
            want.append(forward(x, a))
            a.synchronize()
        outs = [forward(x, s) for _ in range(8) for x, s in zip(xs, (a, b))]
        torch.cuda.synchronize()
        assert all(torch.equal(y, want[n % 2]) for n, y in enumerate(outs))
        graph = torch.cuda.CUDAGraph()
        x = xs[0].clone()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=a):
            y = forward(x, a)
        big = torch.rand(8 * B, 1024, device=cuda)
        torch.cuda.synchronize()
        forward(big, a)
        for n in range(4):
            x.copy_(xs[n % 2])
            torch.cuda.synchronize()
            forward(big, b)
            with torch.cuda.stream(a):
                graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, want[n % 2]), n
    finally:
        torch.cuda.synchronize()
        gpu.kans_qlayer_destroy(h)


def test_per_thread_stream(gpu, cuda):
    """hipStreamPerThread, one handle for a stream of each thread: no workspace is kept for it (split forwards and
    backwards run unsplit) and weights loaded on it are waited for."""
    import metal_kans as mk
    per_thread = ctypes.c_void_p(2)
    m = module(512, 512, degree=5)
    x, g = torch.rand(256, 512, device=cuda) * 2 - 1, torch.randn(256, 512, device=cuda)
    with torch.no_grad():
        y1 = alone(m, x)
        scale(m, 2.0)
        want = alone(m, x)
        torch.cuda.synchronize()
    assert splits_of(gpu, m, 256) > 1
    h = m.metal_layer._engine().handle
    xr = x.clone().requires_grad_(True)
    m(xr).backward(g)
    grads = [t.grad for t in (*m.parameters(), xr)]
    ws = [p.detach() for p in (m.weight, m.base_weight, m.bias_param)]
    y, outs = torch.empty_like(want), [torch.empty_like(t) for t in grads]
    torch.cuda.synchronize()
    hip = hip_runtime()
    for s in (0.5, 1.0):
        half = [(w * s).contiguous() for w in ws]
        torch.cuda.synchronize()
        mk.device.check(gpu.kans_layer_load_weights_stream(h, *[w.data_ptr() for w in half], per_thread), "load")
        mk.device.check(gpu.kans_layer_forward_ex(h, x.data_ptr(), 0, 512, y.data_ptr(), 0, 512, 256, per_thread), "forward")
        assert hip.hipStreamSynchronize(per_thread) == 0
        ref = y1 if s == 0.5 else want
        # other order of 512 * 5 fp32 sums
        assert (y - ref).abs().max() <= 1e-5 * ref.abs().max()
    mk.device.check(gpu.kans_cheby_backward(g.data_ptr(), x.data_ptr(), ws[0].data_ptr(), ws[1].data_ptr(),
                                            *[t.data_ptr() for t in outs], 256, 512, 512, 5, 1, 1, per_thread), "backward")
    assert hip.hipStreamSynchronize(per_thread) == 0
    for a, b in zip(outs, grads):
        assert (a - b).abs().max() <= 1e-5 * b.abs().max()
    assert gpu.kans_stream_keep(per_thread) < 0


def test_parameters_given_back_while_their_retiling_is_queued(cuda):
    """Parameters replaced right after a forward on a held stream: their memory is not reused before the re-tiling
    has read it."""
    m = module(512, 640, degree=4, use_base=False, bias=False)
    x = torch.rand(128, 512, device=cuda) * 2 - 1
    side = torch.cuda.Stream()
    with torch.no_grad():
        want = alone(m, x)
        for fill in (float("nan"), 0.0):
            m.weight = torch.nn.Parameter(m.weight.detach().clone())   # another version of the same values
            torch.cuda.synchronize()
            with torch.cuda.stream(side):
                torch.cuda._sleep(HOLD)
                y = m(x)
            kept = m.weight.detach().cpu()
            shape = m.weight.shape
            m.weight = None
            reuse = [torch.full(shape, fill, device=cuda) for _ in range(3)]
            torch.cuda.synchronize()
            assert torch.equal(y, want)
            del reuse
            m.weight = torch.nn.Parameter(kept.to(cuda))


def test_capture_while_a_load_is_queued(gpu, cuda):
    """Weights loaded on a held stream that is then captured: the captured forward waits for them (its replay runs on
    another stream at once), and a first forward on a third stream meanwhile neither fails nor breaks the capture."""
    import metal_kans as mk
    m = module(64, 72, degree=4)
    side, other, third = (torch.cuda.Stream() for _ in range(3))
    x = torch.rand(96, 64, device=cuda) * 2 - 1
    y3 = torch.empty(96, 72, device=cuda)
    with torch.no_grad():
        for third_first in (False, True):
            old = alone(m, x)
            scale(m, 2.0)
            torch.cuda.synchronize()
            with torch.cuda.stream(side):
                torch.cuda._sleep(HOLD)
                m(x)                          # the load waits on the held stream
                graph = torch.cuda.CUDAGraph()
                graph.capture_begin()
                if third_first:
                    mk.device.check(gpu.kans_layer_forward_ex(m.metal_layer._engine().handle, x.data_ptr(), 0, 64,
                                                              y3.data_ptr(), 0, 72, 96, third.cuda_stream), "forward")
                y = m(x)
                graph.capture_end()
            with torch.cuda.stream(other):
                graph.replay()
                got = y.clone()
            torch.cuda.synchronize()
            want = alone(m, x)
            assert torch.equal(got, want) and not torch.equal(got, old)
            assert not third_first or torch.equal(y3, want)


def test_load_while_a_readers_stream_is_captured(gpu, cuda):
    """A load behind a forward whose stream is captured by then: the old forward keeps its weights, the capture
    survives."""
    import metal_kans as mk
    m = module(512, 512, degree=5)
    x = torch.rand(256, 512, device=cuda) * 2 - 1
    side, other = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.no_grad():
        old = alone(m, x)
        scale(m, 2.0)
        new = alone(m, x)
        scale(m, 0.5)
        torch.cuda.synchronize()
        doubled = [(p.detach() * 2.0).contiguous() for p in (m.weight, m.base_weight, m.bias_param)]
        with torch.cuda.stream(other):
            m(x)                              # the old weights, loaded
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            torch.cuda._sleep(HOLD)
            y = m(x)                          # reads the old tiles, held
            z = torch.zeros(8, device=cuda)
            graph = torch.cuda.CUDAGraph()
            graph.capture_begin()
            mk.device.check(gpu.kans_layer_load_weights_stream(m.metal_layer._engine().handle,
                                                               *[w.data_ptr() for w in doubled], other.cuda_stream), "load")
            z.add_(1.0)
            graph.capture_end()
        torch.cuda.synchronize()
        assert torch.equal(y, old)
        graph.replay()
        torch.cuda.synchronize()
        y2 = torch.empty_like(new)
        mk.device.check(gpu.kans_layer_forward_ex(m.metal_layer._engine().handle, x.data_ptr(), 0, 512, y2.data_ptr(), 0,
                                                  512, 256, other.cuda_stream), "forward")
        torch.cuda.synchronize()
        assert torch.equal(y2, new) and z[0].item() == 1.0
