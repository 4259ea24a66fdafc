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


# one row, a tile edge and one beside it, 4 and 8 wavefronts, 1 to 16 slices, K that ends in each quad of a group
SHAPES = [(1, 1, 128), (1, 1000, 1280), (31, 33, 132), (32, 32, 384), (33, 65, 252), (49, 160, 960), (37, 512, 2048), (50, 101, 644),
          (5, 7, 8196), (784, 32, 192), (1024, 256, 256)]


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_products(hip, m, n, k):
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


@pytest.mark.parametrize("n,h,w,cin,cout,f,stride,relu", [(1, 7, 7, 512, 512, 3, 1, False), (1, 14, 14, 256, 256, 3, 1, True), (1, 28, 28, 256, 512, 1, 2, False),
                                                         (2, 5, 3, 80, 36, 5, 2, True), (1, 2, 50, 256, 250, 3, 1, True), (3, 9, 11, 16, 48, 3, 1, False)])
def test_convolutions(hip, n, h, w, cin, cout, f, stride, relu):
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
