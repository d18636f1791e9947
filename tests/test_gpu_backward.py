"""GPU parity of the fused Chebyshev backward (run on an MI355X).

Oracle: ``oracle.kan_oracle.cheby_backward`` in float64 (pinned in tests/test_oracle.py against
finite differences, the closed form of T'_k and brute-force loops).  Bar: fp32, max|g - g_ref| /
max|g_ref| <= 1e-4 for every gradient.  Also re-runs the reference's own backward tests:
test_optimizations.py:59-100 (fused vs unfused entry point) and test_training.py:20-71 (finite
differences through the layer API).
"""
import ctypes

import numpy as np
import pytest

from oracle import kan_oracle as O

pytestmark = pytest.mark.gpu


def run_host(lib, fn, dY, X, W, Wb, has_bias):
    B, D_in = X.shape
    D_out = dY.shape[1]
    K = W.shape[1] // D_in
    dW = np.full_like(W, np.nan)
    dWb = np.full_like(Wb, np.nan) if Wb is not None else None
    db = np.full(D_out, np.nan, np.float32) if has_bias else None
    dX = np.full_like(X, np.nan)
    ptr = lambda a: a.ctypes.data if a is not None else None  # noqa: E731
    rc = fn(ptr(dY), ptr(X), ptr(W), ptr(Wb), ptr(dW), ptr(dWb), ptr(db), ptr(dX), B, D_in, D_out, K,
            int(Wb is not None), int(has_bias))
    assert rc == 0, lib.kans_last_error()
    return dW, dWb, db, dX


def case(seed, B, D_in, D_out, K, base, bias, x_lo=-1.3, x_hi=1.3):
    rng = np.random.default_rng(seed)
    X = rng.uniform(x_lo, x_hi, (B, D_in)).astype(np.float32)
    W = rng.normal(0, 1 / np.sqrt(D_in * K), (D_out, D_in * K)).astype(np.float32)
    Wb = rng.normal(0, 1 / np.sqrt(D_in), (D_out, D_in)).astype(np.float32) if base else None
    dY = rng.normal(0, 1, (B, D_out)).astype(np.float32)
    return dY, X, W, Wb


def check(got, ref, tol=1e-4):
    for g, r, name in zip(got, ref, ("dW", "dW_base", "dbias", "dX")):
        if r is None:
            assert g is None
            continue
        e = O.rel_err(g, r)
        assert np.isfinite(g).all(), name
        assert e <= tol, f"{name}: rel err {e:.2e}"


SHAPES = [(1, 3, 5), (37, 24, 70), (130, 33, 64), (300, 16, 9)]


@pytest.mark.parametrize("K", [1, 2, 4, 9, 16, 32])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("base,bias", [(True, True), (False, False), (True, False)])
def test_backward_matches_oracle(gpu, K, shape, base, bias):
    B, D_in, D_out = shape
    dY, X, W, Wb = case(K * 100 + B, B, D_in, D_out, K, base, bias)
    got = run_host(gpu, gpu.metal_kan_cheby_backward_fused, dY, X, W, Wb, bias)
    check(got, O.cheby_backward(dY, X, W, Wb, bias))


def test_backward_device_entry_larger_shape(gpu):
    """kans_cheby_backward on device buffers at 2048 x 512 -> 256, K = 9 (base, bias)."""
    lib = gpu
    B, D_in, D_out, K = 2048, 512, 256, 9
    dY, X, W, Wb = case(77, B, D_in, D_out, K, True, True)
    ref = O.cheby_backward(dY, X, W, Wb, True)
    bufs = {}
    try:
        for name, a in (("dY", dY), ("X", X), ("W", W), ("Wb", Wb)):
            p = ctypes.c_void_p()
            assert lib.kans_dev_malloc(ctypes.byref(p), a.nbytes) == 0
            assert lib.kans_memcpy_h2d(p, a.ctypes.data, a.nbytes) == 0
            bufs[name] = p
        outs = {"dW": np.empty_like(W), "dWb": np.empty_like(Wb), "db": np.empty(D_out, np.float32),
                "dX": np.empty_like(X)}
        for name, a in outs.items():
            p = ctypes.c_void_p()
            assert lib.kans_dev_malloc(ctypes.byref(p), a.nbytes) == 0
            bufs[name] = p
        assert lib.kans_cheby_backward(bufs["dY"], bufs["X"], bufs["W"], bufs["Wb"], bufs["dW"], bufs["dWb"],
                                       bufs["db"], bufs["dX"], B, D_in, D_out, K, 1, 1, None) == 0, \
            lib.kans_last_error()
        assert lib.kans_synchronize() == 0
        for name, a in outs.items():
            assert lib.kans_memcpy_d2h(a.ctypes.data, bufs[name], a.nbytes) == 0
        check((outs["dW"], outs["dWb"], outs["db"], outs["dX"]), ref)
    finally:
        for p in bufs.values():
            lib.kans_dev_free(p)


def test_backward_rejects_bad_arguments(gpu):
    lib = gpu
    dY, X, W, Wb = case(1, 4, 3, 2, 4, True, True)
    z = np.zeros(64, np.float32)
    p = z.ctypes.data
    assert lib.metal_kan_cheby_backward_fused(p, p, p, None, p, None, None, p, 4, 3, 2, 4, 1, 0) < 0  # base, no W_base
    assert lib.metal_kan_cheby_backward_fused(p, p, p, p, p, p, None, p, 4, 3, 2, 4, 1, 1) < 0  # bias, no dbias
    assert lib.metal_kan_cheby_backward_fused(p, p, p, p, p, p, p, p, 0, 3, 2, 4, 1, 1) < 0     # B = 0
    assert lib.metal_kan_cheby_backward_fused(p, p, p, p, p, p, p, p, 4, 3, 2, 33, 1, 1) < 0    # K > 32


def test_reference_fused_vs_unfused(gpu):
    """test_optimizations.py:59-100: both entry points, B=32, 16 -> 8, degree 4, base and bias."""
    lib = gpu
    B, D_in, D_out, degree = 32, 16, 8, 4
    np.random.seed(123)
    dY = np.random.randn(B, D_out).astype(np.float32)
    X = np.random.uniform(-0.9, 0.9, (B, D_in)).astype(np.float32)
    W = np.random.randn(D_out, D_in * degree).astype(np.float32)
    Wb = np.random.randn(D_out, D_in).astype(np.float32)
    a = run_host(lib, lib.metal_kan_cheby_backward, dY, X, W, Wb, True)
    b = run_host(lib, lib.metal_kan_cheby_backward_fused, dY, X, W, Wb, True)
    assert np.max(np.abs(a[0] - b[0])) < 1e-4
    assert np.max(np.abs(a[3] - b[3])) < 1e-4
    assert np.max(np.abs(a[2] - b[2])) < 1e-5
    check(b, O.cheby_backward(dY, X, W, Wb, True))


def test_reference_layer_gradient_numerical_check(gpu):
    """test_training.py:20-71: ChebyKAN(3 -> 2, degree 4) dX and dW against central differences of
    the GPU forward (eps 1e-4, relative error < 1e-3), then zero_grad."""
    import metal_kans as mk
    np.random.seed(42)
    B, D_in, D_out, deg = 4, 3, 2, 4
    layer = mk.ChebyKAN(D_in, D_out, degree=deg, bias=True, use_base=True)
    X = np.random.uniform(-0.8, 0.8, (B, D_in)).astype(np.float32)
    dY = np.random.randn(B, D_out).astype(np.float32)
    layer(X)
    dX = layer.backward(dY)
    eps = 1e-4
    dX_num = np.zeros_like(X)
    for i in range(B):
        for j in range(D_in):
            Xp, Xm = X.copy(), X.copy()
            Xp[i, j] += eps
            Xm[i, j] -= eps
            dX_num[i, j] = (np.sum(layer(Xp) * dY) - np.sum(layer(Xm) * dY)) / (2 * eps)
    rel = np.linalg.norm(dX - dX_num) / (np.linalg.norm(dX) + np.linalg.norm(dX_num) + 1e-7)
    assert rel < 1e-3
    layer(X)
    layer.backward(dY)
    gW = layer.grad_w_cheby.copy()
    dW_num = np.zeros_like(layer.w_cheby)
    for i in range(layer.w_cheby.shape[0]):
        for j in range(layer.w_cheby.shape[1]):
            w0 = layer.w_cheby[i, j]
            layer.w_cheby[i, j] = w0 + eps
            lp = np.sum(layer(X) * dY)
            layer.w_cheby[i, j] = w0 - eps
            lm = np.sum(layer(X) * dY)
            layer.w_cheby[i, j] = w0
            dW_num[i, j] = (lp - lm) / (2 * eps)
    rel = np.linalg.norm(gW - dW_num) / (np.linalg.norm(gW) + np.linalg.norm(dW_num) + 1e-7)
    assert rel < 1e-3
    assert layer.grad_bias.shape == (D_out,) and layer.grad_w_base.shape == (D_out, D_in)
    layer.zero_grad()
    assert not layer.grad_w_cheby.any() and not layer.grad_bias.any()


def test_layer_backward_shapes_and_dtypes(gpu):
    """Layer API: 3-D input, no base / bias, and a half layer differentiated in fp32."""
    import metal_kans as mk
    np.random.seed(7)
    layer = mk.ChebyKAN(24, 10, degree=5, bias=False, use_base=False)
    x = np.random.uniform(-1.2, 1.2, (2, 7, 24)).astype(np.float32)
    y = layer(x)
    dY = np.random.randn(*y.shape).astype(np.float32)
    dX = layer.backward(dY)
    assert dX.shape == x.shape
    assert layer.grad_w_base.shape == (1,) and layer.grad_bias.shape == (1,)
    ref = O.cheby_backward(dY.reshape(14, 10), x.reshape(14, 24), layer.w_cheby, None, False)
    assert O.rel_err(layer.grad_w_cheby, ref[0]) <= 1e-4
    assert O.rel_err(dX.reshape(14, 24), ref[3]) <= 1e-4

    h = mk.ChebyKAN(16, 8, degree=4).half()
    xh = np.random.uniform(-1, 1, (9, 16)).astype(np.float16)
    h(xh)
    dYh = np.random.randn(9, 8).astype(np.float32)
    dXh = h.backward(dYh)
    ref = O.cheby_backward(dYh, xh.astype(np.float32), h.w_cheby.astype(np.float32),
                           h.w_base.astype(np.float32), True)
    assert O.rel_err(dXh, ref[3]) <= 1e-4 and O.rel_err(h.grad_w_cheby, ref[0]) <= 1e-4


# Edges of the backward kernels' tiles: 32-row tiles in workgroups of 128 (NS = K - 1 + base > 5 slots) or 256
# rows, 64 features, 16-deep steps; slot counts 1..10 and several groups of them; grids that split the
# contraction and (the last two) grids that fill the chip without; odd widths (no 16-byte rows of dY).
EDGES = [(1, 1, 1, 2, 0), (16, 64, 256, 3, 0), (17, 65, 257, 4, 1), (33, 63, 129, 6, 0), (128, 32, 128, 7, 0),
         (129, 96, 127, 7, 1), (250, 31, 31, 8, 1), (64, 64, 64, 9, 1), (40, 33, 48, 11, 0), (40, 70, 50, 12, 1),
         (48, 20, 36, 22, 1), (31, 40, 20, 32, 1), (40, 2048, 2050, 2, 0), (2050, 2048, 20, 2, 0)]


@pytest.mark.parametrize("B,D_in,D_out,K,base", EDGES)
def test_backward_tile_edges(gpu, B, D_in, D_out, K, base):
    dY, X, W, Wb = case(B + K, B, D_in, D_out, K, bool(base), True)
    got = run_host(gpu, gpu.metal_kan_cheby_backward_fused, dY, X, W, Wb, True)
    # fp32 sums of at most 2050 terms: 2^-24 * sqrt(2050) = 3e-6 of the largest gradient
    check(got, O.cheby_backward(dY, X, W, Wb, True), 1e-5)


def test_backward_wide_range_and_infinities(gpu):
    """Operands of 1e-30 .. 1e30 keep fp32 accuracy (their bf16 terms have fp32's exponent range), and an
    infinite upstream gradient makes exactly the gradients it enters non-finite."""
    B, D_in, D_out, K = 48, 40, 30, 5
    dY, X, W, Wb = case(3, B, D_in, D_out, K, True, True)
    scale = np.float32(10.0) ** np.linspace(-30, 30, B).astype(np.float32)
    dY *= scale[:, None]
    dX = run_host(gpu, gpu.metal_kan_cheby_backward_fused, dY, X, W, Wb, True)[3]
    ref = O.cheby_backward(dY, X, W, Wb, True)[3]
    for b in range(B):   # every row at its own scale
        assert O.rel_err(dX[b], ref[b]) <= 1e-5, b
    dY, X, W, Wb = case(4, B, D_in, D_out, K, True, True)
    dY[7, 11] = np.inf
    dW, dWb, db, dX = run_host(gpu, gpu.metal_kan_cheby_backward_fused, dY, X, W, Wb, True)
    for g in (dW, dWb):
        assert np.isfinite(np.delete(g, 11, 0)).all()
    # one infinite term in each sum: inf times the sign of T_k(x) (SiLU(x)), as in one fp32 sum
    np.testing.assert_array_equal(dWb[11], np.sign(X[7]) * np.inf)
    np.testing.assert_array_equal(dW[11].reshape(D_in, K)[:, 1], np.sign(np.clip(X[7], -1, 1)) * np.inf)
    assert db[11] == np.inf and np.isfinite(np.delete(db, 11)).all()
    assert not np.isfinite(dX[7][np.abs(X[7]) <= 1]).any() and np.isfinite(np.delete(dX, 7, 0)).all()


def test_backward_streams_and_capture(gpu):
    """Calls that share the partial-sum workspace from two streams, and a call recorded into a graph (which
    gets no workspace), give the gradients of a call alone."""
    torch = pytest.importorskip("torch")
    from metal_kans import device
    B, D_in, D_out, K = 512, 64, 96, 5
    arrs = [case(20 + n, B, D_in, D_out, K, True, True) for n in range(2)]
    dev = [[torch.from_numpy(a).cuda() for a in c] for c in arrs]
    outs = [[torch.zeros(s, device="cuda") for s in ((D_out, D_in * K), (D_out, D_in), (D_out,), (B, D_in))]
            for _ in range(2)]

    def call(n, stream):
        p = [t.data_ptr() for t in dev[n] + outs[n]]
        device.check(gpu.kans_cheby_backward(*p, B, D_in, D_out, K, 1, 1, stream.cuda_stream), "backward")

    refs = [O.cheby_backward(*c, True) for c in arrs]
    s = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    for _ in range(4):
        call(0, s[0])
        call(1, s[1])
    torch.cuda.synchronize()
    for n in range(2):
        check([t.cpu().numpy() for t in outs[n]], refs[n], 1e-5)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s[0]):
        call(0, s[0])
    for _ in range(3):
        for t in outs[0]:
            t.zero_()
        call(1, s[1])
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        check([t.cpu().numpy() for t in outs[0]], refs[0], 1e-5)


def test_backward_wide_output(gpu):
    """More outputs than 32-bit offsets over the 256 rows of a dX tile reach (2^32 / 1024), two row blocks."""
    B, D_in, D_out, K = 33, 1, (1 << 22) + 3, 2
    dY, X, W, Wb = case(9, B, D_in, D_out, K, False, True)
    got = run_host(gpu, gpu.metal_kan_cheby_backward_fused, dY, X, W, Wb, True)
    # T_0 = 1, T_1 = x; dX = dY W[:, 1] where |x| <= 1
    t = np.clip(X[:, 0].astype(np.float64), -1, 1)
    db = dY.sum(0, dtype=np.float64)
    dW = np.stack([db, t @ dY], 1)
    dX = (dY.astype(np.float64) @ W[:, 1].astype(np.float64))[:, None] * (np.abs(X) <= 1)
    check(got[:3], (dW, None, db), 1e-5)
    # dX adds 64 partial sums of 4096 steps, six products each: as many roundings of half a unit (2^-24), which add
    # like a random walk, four deviations
    assert O.rel_err(got[3], dX) <= 4 * np.sqrt(6 * 4096) * 2.0 ** -24


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("B,D_in,D_out,K,base", [e for e in EDGES if e[3] - 1 + e[4] <= 10] + [(40, 33, 48, 10, 1)])
def test_backward_16bit_arrays(gpu, dtype, B, D_in, D_out, K, base):
    """kans_cheby_backward_ex on 16-bit arrays: the gradients of those values, each rounded once."""
    torch = pytest.importorskip("torch")
    dt = getattr(torch, dtype)
    dev = [None if a is None else torch.from_numpy(a).cuda().to(dt) for a in case(B + K, B, D_in, D_out, K, bool(base), True)]
    outs = [torch.empty(s, device="cuda", dtype=dt) if s else None
            for s in ((D_out, D_in * K), (D_out, D_in) if base else None, (D_out,), (B, D_in))]
    torch.cuda.synchronize()
    assert gpu.kans_cheby_backward_ex({"float16": 1, "bfloat16": 2}[dtype],
                                      *(t.data_ptr() if t is not None else None for t in dev + outs),
                                      B, D_in, D_out, K, base, 1, None) == 0, gpu.kans_last_error()
    assert gpu.kans_synchronize() == 0
    ref = O.cheby_backward(*(None if t is None else t.float().cpu().numpy() for t in dev), True)
    # half a unit in the last place of a 16-bit result, beside the fp32 sums' 1e-5 of the largest gradient
    half_ulp = 2.0 ** (-11 if dtype == "float16" else -8)
    for got, r, name in zip(outs, ref, ("dW", "dW_base", "dbias", "dX")):
        if got is None:
            continue
        g = got.double().cpu().numpy()
        bound = half_ulp * np.abs(r) + 1e-5 * np.abs(r).max() + 2.0 ** -24
        assert (np.abs(g - r) <= bound).all(), f"{name}: {np.max(np.abs(g - r) / bound):.3f} of the bound"


def test_backward_16bit_infinities_and_limits(gpu):
    """An infinite 16-bit upstream gradient makes exactly the gradients it enters non-finite; slot counts that
    the 16-bit kernels don't take and unknown types are refused."""
    torch = pytest.importorskip("torch")
    B, D_in, D_out, K = 48, 40, 30, 5
    for code, dt in ((1, torch.float16), (2, torch.bfloat16)):
        dev = [torch.from_numpy(a).cuda().to(dt) for a in case(4, B, D_in, D_out, K, True, True)]
        dev[0][7, 11] = float("inf")
        outs = [torch.empty(s, device="cuda", dtype=dt) for s in ((D_out, D_in * K), (D_out, D_in), (D_out,), (B, D_in))]
        ptrs = [t.data_ptr() for t in dev + outs]
        torch.cuda.synchronize()
        assert gpu.kans_cheby_backward_ex(code, *ptrs, B, D_in, D_out, K, 1, 1, None) == 0
        assert gpu.kans_synchronize() == 0
        dW, dWb, db, dX = (t.float().cpu().numpy() for t in outs)
        x = dev[1][7].float().cpu().numpy()
        assert np.isfinite(np.delete(dW, 11, 0)).all() and np.isfinite(np.delete(dWb, 11, 0)).all()
        np.testing.assert_array_equal(dWb[11], np.sign(x) * np.inf)
        np.testing.assert_array_equal(dW[11].reshape(D_in, K)[:, 1], np.sign(x) * np.inf)
        assert db[11] == np.inf and np.isfinite(np.delete(db, 11)).all()
        assert not np.isfinite(dX[7][np.abs(x) <= 1]).any() and np.isfinite(np.delete(dX, 7, 0)).all()
        assert gpu.kans_cheby_backward_ex(code, *ptrs, B, D_in, D_out, 11, 1, 1, None) < 0
        assert gpu.kans_cheby_backward_ex(code, *ptrs, B, D_in, D_out, 1, 0, 1, None) < 0
    assert gpu.kans_cheby_backward_ex(7, *ptrs, B, D_in, D_out, K, 1, 1, None) < 0


def test_backward_largest_values_and_products_of_infinities(gpu):
    """Gradients of the largest finite size stay finite, and an infinite gradient times an infinite weight or
    activation is an infinity of the right sign."""
    B, D_in, D_out, K = 40, 36, 34, 5
    dY, X, W, Wb = case(5, B, D_in, D_out, K, True, True, -0.9, 0.9)
    big = np.float32(np.finfo(np.float32).max)
    W *= np.float32(0.01)
    Wb *= np.float32(0.01)
    dY[:] = 0
    dY[np.arange(34), np.arange(34)] = big * np.where(np.arange(34) % 2, 1, -1).astype(np.float32)
    got = run_host(gpu, gpu.metal_kan_cheby_backward_fused, dY, X, W, Wb, True)
    ref = O.cheby_backward(dY, X, W, Wb, True)
    for g, r in zip(got, ref):   # one product in each sum, of fp32 factors (T'_k and SiLU' of a few roundings)
        assert np.isfinite(g).all()
        assert (np.abs(g - r) <= 2.0 ** -20 * np.abs(r) + 2.0 ** -22 * np.abs(r).max()).all()
    dY, X, W, Wb = case(6, B, D_in, D_out, K, True, True, -0.9, 0.9)
    dY[7, 11], X[7, 2], Wb[11, 4] = -np.inf, np.inf, np.inf
    dW, dWb, db, dX = run_host(gpu, gpu.metal_kan_cheby_backward_fused, dY, X, W, Wb, True)
    assert dWb[11, 2] == -np.inf              # -inf * SiLU(inf)
    assert dX[7, 4] == -np.inf or np.isnan(dX[7, 4])
    keep = np.delete(np.arange(D_out), 11)
    assert np.isfinite(dWb[np.ix_(keep, np.delete(np.arange(D_in), 2))]).all()
    np.testing.assert_array_equal(dWb[keep, 2], np.sign(dY[7, keep]) * np.inf)


@pytest.mark.parametrize("D_in,D_out,K,base", [(1, (1 << 25) + 5, 2, False),      # rows of dY
                                               ((1 << 24) + 3, 2, 5, True),       # rows of W
                                               ((1 << 24) + 3, 1, 20, True)])     # and more workgroups than a launch takes
def test_backward_rows_beyond_32_bit_offsets(gpu, D_in, D_out, K, base):
    """Shapes whose rows the dX kernel's 32-bit lane offsets do not reach over."""
    B = 2
    rng = np.random.default_rng(D_out)
    X = rng.uniform(-1.2, 1.2, (B, D_in)).astype(np.float32)
    W = (rng.random((D_out, D_in * K), dtype=np.float32) - 0.5) / np.float32(K)
    Wb = rng.random((D_out, D_in), dtype=np.float32) - 0.5 if base else None
    dY = (rng.random((B, D_out), dtype=np.float32) - 0.5)
    dW, dWb, db, dX = run_host(gpu, gpu.metal_kan_cheby_backward_fused, dY, X, W, Wb, True)
    x, g = X.astype(np.float64), dY.astype(np.float64)
    t, inside = np.clip(x, -1, 1), np.abs(X) <= 1
    # the largest sum here has 2^25 terms of both signs: 32768 partial steps, a random walk of half units (2^-24)
    tol = 1e-5 if D_out < 1 << 20 else 4 * np.sqrt(6 * D_out / 64 / 16) * 2.0 ** -24

    def close(got, want, name):
        assert np.abs(got - want).max() <= tol * max(np.abs(want).max(), 1e-3), name
    close(db, g.sum(0), "dbias")
    T, D = [np.ones_like(t), t], [np.zeros_like(x), np.ones_like(x)]
    dx = np.zeros_like(x)
    W3, dW3 = W.reshape(D_out, D_in, K), dW.reshape(D_out, D_in, K)
    for k in range(K):
        if k >= 2:
            T = [T[1], 2 * t * T[1] - T[0]]
            D = [D[1], 2 * T[0] + 2 * t * D[1] - D[0]]
        Tk, Dk = (T[k], D[k]) if k < 2 else (T[1], D[1])
        close(dW3[:, :, k], g.T @ Tk, f"dW {k}")
        if k:
            dx += (g @ W3[:, :, k].astype(np.float64)) * Dk * inside
    if base:
        sg = 1 / (1 + np.exp(-x))
        close(dWb, g.T @ (x * sg), "dW_base")
        dx += (g @ Wb.astype(np.float64)) * sg * (1 + x * (1 - sg))
    close(dX, dx, "dX")
