"""Products and convolutions of a few more workgroups than all compute units hold eight of: six at once up to twelve to a unit."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    import nhtest
    return nhtest.Hip()


def _check(got, a, b, bias, k):
    """a [M,K], b [N,K] in 64 bits: at most one rounding per product and a few for the slices and the epilogue"""
    bound = (k + 40) * 2.0 ** -24 * (a.abs() @ b.abs().T + bias.abs())
    excess = ((got.double() - (a @ b.T + bias)).abs() - bound).max().item()
    assert excess <= 0, excess


# 64 x 64 tiles: 2048, 2052, 3072 and 3076 of them, and 2504 of four steps of 16
@pytest.mark.parametrize("m,n,k", [(32768, 256, 100), (32769, 256, 100), (49152, 256, 68), (49153, 256, 68), (20011, 509, 52)])
def test_products(hip, m, n, k):
    torch = hip.torch
    g = torch.Generator(device=hip.dev).manual_seed(m)
    a, b = torch.randn(m, k, generator=g, device=hip.dev), torch.randn(n, k, generator=g, device=hip.dev)
    c = torch.full((m + 1, n), 7.0, device=hip.dev)
    hip.call("nhMultiplyMatrixByTransposedMatrix", hip.p(a), m, k, k, hip.p(b), n, k, hip.p(c), n, m * n)
    _check(c[:m], a.double(), b.double(), torch.zeros(n, device=hip.dev, dtype=torch.float64), k)
    assert (c[m] == 7.0).all()


# 2352 workgroups of three slices that meet, 2338 of one slice with ragged last tiles
@pytest.mark.parametrize("n,h,w,cin,cout", [(64, 14, 14, 256, 256), (13, 71, 81, 16, 70)])
@pytest.mark.parametrize("residual", [False, True])
def test_convolutions(hip, n, h, w, cin, cout, residual):
    torch = hip.torch
    g = torch.Generator(device=hip.dev).manual_seed(h)
    x, filt = torch.randn(n, h, w, cin, generator=g, device=hip.dev), torch.randn(cout, 3, 3, cin, generator=g, device=hip.dev)
    bias, other = torch.randn(cout, generator=g, device=hip.dev), torch.randn(n * h * w, cout, generator=g, device=hip.dev)
    d = hip.conv_desc(n, h, w, cin, cout, 3, 3, 1, 1, 1, 1)
    y = torch.empty(n * h * w, cout, device=hip.dev)
    stream = ctypes.c_void_p()
    hip.na.check(hip.lib.nhStreamCreate(ctypes.byref(stream)))
    try:
        hip.na.check(hip.lib.nhStreamDeferSmallOps(stream, 1))
        torch.cuda.synchronize()
        hip.na.check(hip.lib.nhBlobConvolution(stream, ctypes.byref(d), hip.p(x), hip.p(filt), hip.p(bias), hip.p(y)))
        if residual:  # ( one launch with the convolution, a kernel of its own )
            hip.na.check(hip.lib.nhVectorAdd(stream, hip.p(y), hip.p(other), hip.p(y), y.numel()))
        hip.na.check(hip.lib.nhStreamSynchronize(stream))
    finally:
        hip.na.check(hip.lib.nhStreamDestroy(stream))
    p = torch.nn.functional.pad(x.double(), (0, 0, 1, 1, 1, 1)).unfold(1, 3, 1).unfold(2, 3, 1)
    a = p.permute(0, 1, 2, 4, 5, 3).reshape(-1, 9 * cin)
    _check(y, a, filt.double().reshape(cout, -1), bias.double() + (other.double() if residual else 0), 9 * cin)
