"""Products and convolutions with results of a few 32 x 32 tiles, whose reductions are dealt to wavefronts and workgroups."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    import nhtest
    return nhtest.Hip()


def _check(got, a, b, k):
    """a [M,K], b [N,K] in 64 bits: at most one rounding per product and a few for the shares and the epilogue"""
    bound = (k + 40) * 2.0 ** -24 * (a.abs() @ b.abs().T)
    excess = ((got.double() - a @ b.T).abs() - bound).max().item()
    assert excess <= 0, excess


# one row, a tile edge and one beside it, 4 and 8 wavefronts, 1 to 16 slices, even and odd numbers of them and of the groups of a share,
# K that ends in each quad of a group
SHAPES = [(1, 1, 128), (1, 1000, 1280), (31, 33, 132), (32, 32, 384), (33, 65, 252), (49, 160, 960), (37, 512, 2048), (50, 101, 644),
          (5, 7, 8196), (784, 32, 192), (1024, 256, 256), (37, 512, 400), (50, 1024, 512), (33, 480, 768), (100, 512, 1100), (64, 64, 1304)]
BATCHES = [(8, 33, 65, 132), (4, 60, 100, 256), (3, 1, 50, 388), (200, 7, 31, 128)]
CONVOLUTIONS = [(1, 7, 7, 512, 512, 3, 1, False), (1, 14, 14, 256, 256, 3, 1, True), (1, 28, 28, 256, 512, 1, 2, False),
                (2, 5, 3, 80, 36, 5, 2, True), (1, 2, 50, 256, 250, 3, 1, True), (3, 9, 11, 16, 48, 3, 1, False), (1, 30, 30, 48, 48, 3, 1, True)]
STEPS = [(132, 5), (260, 33)]  # ( hidden, batch )
# ( batch, height, width, channels, filters, filter size, padding )
GRADIENTS = [(1, 7, 7, 256, 256, 3, 1), (2, 9, 11, 80, 48, 5, 2), (1, 5, 6, 33, 512, 3, 0), (1, 30, 29, 48, 32, 3, 1)]


@pytest.fixture(scope="module")
def launched():
    import nhtest
    calls = [("nt", 1, m, n, k, n + 3) for m, n, k in SHAPES] + [("nt", b, m, n, k, n) for b, m, n, k in BATCHES]
    calls += [("conv", n, h, w, cin, cout, f, f // 2, stride) for n, h, w, cin, cout, f, stride, _ in CONVOLUTIONS]
    calls += [("conv_backward",) + c + (1,) for c in GRADIENTS] + [("lstm", 2, batch, 24, hidden) for hidden, batch in STEPS]
    return dict(zip(calls, nhtest.kernel_names(calls)))


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_products(hip, launched, m, n, k):
    assert launched["nt", 1, m, n, k, n + 3] == ["smallProductKernel<0, %d>" % (8 if k > 240 else 4)]
    torch = hip.torch
    g = torch.Generator(device=hip.dev).manual_seed(m + n + k)
    pitch = n + 3
    a = torch.randn(m, k, generator=g, device=hip.dev)
    b = torch.randn(n, k, generator=g, device=hip.dev)
    c = torch.full((m, pitch), 7.0, device=hip.dev)
    first = None
    for _ in range(3):  # ( the arrival counters are back at zero behind every launch )
        hip.call("nhMultiplyMatrixByTransposedMatrix", hip.p(a), m, k, k, hip.p(b), n, k, hip.p(c), pitch, c.numel())
        _check(c[:, :n], a.double(), b.double(), k)
        assert (c[:, n:] == 7.0).all()
        assert first is None or torch.equal(first, c)
        first = c.clone()


@pytest.mark.parametrize("batch,m,n,k", BATCHES)
def test_batches(hip, launched, batch, m, n, k):
    assert launched["nt", batch, m, n, k, n] == ["smallProductKernel<0, %d>" % (8 if k > 240 else 4)]
    torch = hip.torch
    g = torch.Generator(device=hip.dev).manual_seed(batch)
    a = torch.randn(batch, m, k, generator=g, device=hip.dev)
    b = torch.randn(batch, n, k, generator=g, device=hip.dev)
    c = torch.full((batch, m, n), 7.0, device=hip.dev)
    hip.call("nhBatchMultiplyMatrixByTransposedMatrix", batch, hip.p(a), m, k, hip.p(b), n, hip.p(c), c.numel())
    for i in range(batch):
        _check(c[i], a[i].double(), b[i].double(), k)


@pytest.mark.parametrize("hidden,batch", STEPS)
def test_products_added_to_the_result(hip, launched, hidden, batch):
    """The steps of an LSTM whose width no other path takes: gates += h * W^T."""
    assert "smallProductKernel<0, %d>" % (8 if hidden > 240 else 4) in launched["lstm", 2, batch, 24, hidden]
    import numpy as np
    from nhtest import Cpu, assert_close
    g = np.random.default_rng(hidden)

    def values(*shape):
        return g.uniform(-0.1, 0.1, shape).astype(np.float32)

    args = (values(4 * hidden, 24), values(4 * hidden), values(4 * hidden, hidden), values(4 * hidden), g.uniform(-1, 1, (6, batch, 24)).astype(np.float32))
    for reverse in (False, True):
        for got, want in zip(hip.lstm(*args, reverse=reverse), Cpu("orc").lstm(*args, reverse=reverse)):
            assert_close(got, want, "lstm, %d units" % hidden)


def test_residual(hip):
    """The down convolution of a gated block over one small image: free term, and the residual added behind it."""
    import numpy as np
    from nhtest import Cpu, assert_close
    g = np.random.default_rng(7)
    for n, h, w, c, cout in ((1, 7, 7, 480, 80), (1, 9, 5, 132, 33)):
        x = g.uniform(-1, 1, (n, h, w, c)).astype(np.float32)
        gate = g.uniform(0, 1, (n, c)).astype(np.float32)
        res = g.uniform(-1, 1, (n, h, w, cout)).astype(np.float32)
        down = (g.normal(0, 0.1, (cout, c)).astype(np.float32), g.uniform(-1, 1, cout).astype(np.float32))
        assert_close(hip.mobilenetv3_post_se(x, gate, res, "hswish", 0.0, down), Cpu("orc").mobilenetv3_post_se(x, gate, res, "hswish", 0.0, down),
                     "down convolution %s" % ((n, h, w, c, cout),))


@pytest.mark.parametrize("n,h,w,cin,cout,f,pad", GRADIENTS)
def test_gradients_by_the_input(hip, launched, n, h, w, cin, cout, f, pad):
    assert "smallProductKernel<6, %d>" % (8 if f * f * cout > 240 else 4) in launched["conv_backward", n, h, w, cin, cout, f, pad, 1]
    torch = hip.torch
    g = torch.Generator(device=hip.dev).manual_seed(n * h * w)
    d = hip.conv_desc(n, h, w, cin, cout, f, f, pad, pad, 1, 1)
    grad = torch.randn(n, d.resultHeight, d.resultWidth, cout, generator=g, device=hip.dev)
    filt = torch.randn(cout, f, f, cin, generator=g, device=hip.dev)
    free = torch.randn(cin, generator=g, device=hip.dev)
    x = torch.empty(n * h * w, cin, device=hip.dev)
    size = ctypes.c_size_t(0)
    hip.na.check(hip.lib.nhBlobConvolutionBackwardWorkspaceSize(ctypes.byref(d), ctypes.byref(size)))
    work = torch.empty(size.value // 4 + 1, device=hip.dev)
    hip.call("nhBlobConvolutionBackward", ctypes.byref(d), hip.p(grad), hip.p(filt), hip.p(free), hip.p(x), hip.p(work), size)
    # a convolution of the gradient, padded by what the window hangs over, with the filter turned round
    over = f - 1 - pad
    p = torch.nn.functional.pad(grad.double(), (0, 0, over, over, over, over)).unfold(1, f, 1).unfold(2, f, 1)
    a = p.permute(0, 1, 2, 4, 5, 3).reshape(n * h * w, f * f * cout)
    b = filt.double().flip(1, 2).permute(3, 1, 2, 0).reshape(cin, f * f * cout)
    one = torch.ones(a.shape[0], 1, device=hip.dev, dtype=torch.float64)
    _check(x, torch.cat([a, one], 1), torch.cat([b, free.double()[:, None]], 1), f * f * cout)


@pytest.mark.parametrize("n,h,w,cin,cout,f,stride,relu", CONVOLUTIONS)
def test_convolutions(hip, launched, n, h, w, cin, cout, f, stride, relu):
    assert launched["conv", n, h, w, cin, cout, f, f // 2, stride] == ["smallProductKernel<6, %d>" % (8 if f * f * cin > 240 else 4)]
    torch = hip.torch
    pad = f // 2
    g = torch.Generator(device=hip.dev).manual_seed(n * h * w)
    x = torch.randn(n, h, w, cin, generator=g, device=hip.dev)
    filt = torch.randn(cout, f, f, cin, generator=g, device=hip.dev)
    bias = torch.randn(cout, generator=g, device=hip.dev)
    d = hip.conv_desc(n, h, w, cin, cout, f, f, pad, pad, stride, stride)
    y = torch.empty(n * d.resultHeight * d.resultWidth, cout, device=hip.dev)
    p = torch.nn.functional.pad(x.double(), (0, 0, pad, pad, pad, pad)).unfold(1, f, stride).unfold(2, f, stride)
    a = p.permute(0, 1, 2, 4, 5, 3).reshape(-1, f * f * cin)
    a = torch.cat([a, torch.ones(a.shape[0], 1, device=hip.dev, dtype=torch.float64)], 1)
    b = torch.cat([filt.double().reshape(cout, -1), bias.double()[:, None]], 1)
    hip.call("nhBlobConvolutionWithActivation", ctypes.byref(d), hip.p(x), hip.p(filt), hip.p(bias), 1 if relu else 0, 0.0, hip.p(y))
    if relu:
        bound = (f * f * cin + 40) * 2.0 ** -24 * (a.abs() @ b.abs().T)
        assert ((y.double() - (a @ b.T).clamp(min=0)).abs() <= bound).all()
    else:
        _check(y, a, b, f * f * cin)


def test_slices_under_capture(hip):
    """A recorded launch has no scratch to meet in: it takes another way, and every replay gives the eager result."""
    torch = hip.torch
    a, b = torch.randn(37, 2048, device=hip.dev), torch.randn(512, 2048, device=hip.dev)
    c = torch.empty(37, 512, device=hip.dev)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()

    def call():
        hip.call("nhMultiplyMatrixByTransposedMatrix", hip.p(a), 37, 2048, 2048, hip.p(b), 512, 2048, hip.p(c), 512, c.numel())

    with torch.cuda.stream(side):
        call()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=side):
            call()
    for _ in range(3):
        a.normal_()
        c.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        _check(c, a.double(), b.double(), 2048)
