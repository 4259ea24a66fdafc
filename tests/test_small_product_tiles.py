"""The tiles that products of a few hundred workgroups are cut into: 16 x 16, 16 x 32 and 32 x 32, with and without slices."""
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


# one group of 16 k, a group that ends in each of its quads, shares below, at, one above and twice the groups in flight (4 and 6) with 4 and
# 8 wavefronts, a wavefront without a share; results one beside the edges of each tile, few tiles (16 x 16) to many (32 x 32)
@pytest.mark.parametrize("m,n,k", [
    (1, 1, 16), (17, 33, 20), (16, 16, 36), (15, 47, 48), (33, 31, 64), (31, 65, 100), (96, 512, 240), (97, 513, 256), (37, 2048, 516), (200, 640, 772),
    (784, 144, 24), (785, 193, 32), (257, 700, 900), (37, 513, 1028), (16, 160, 1536), (17, 96, 1664), (49, 512, 3072)])
def test_edges(hip, m, n, k):
    torch = hip.torch
    g = torch.Generator(device=hip.dev).manual_seed(m + n + k)
    pitch = n + 1
    a = torch.randn(m, k + 4, generator=g, device=hip.dev)  # ( what lies behind a row's K values must not count )
    b = torch.randn(n, k + 8, generator=g, device=hip.dev)
    a[:, k:] = float("nan")
    b[:, k:] = float("nan")
    c = torch.full((m, pitch), 7.0, device=hip.dev)
    hip.call("nhMultiplyMatrixByTransposedMatrix", hip.p(a), m, k, k + 4, hip.p(b), n, k + 8, hip.p(c), pitch, c.numel())
    _check(c[:, :n], a[:, :k].double(), b[:, :k].double(), k)
    assert (c[:, n:] == 7.0).all()


@pytest.mark.parametrize("n,h,w,cin,cout,f,stride", [(1, 7, 7, 512, 512, 3, 1), (1, 14, 14, 256, 256, 3, 1), (1, 56, 56, 64, 64, 3, 1), (2, 9, 7, 16, 20, 1, 2)])
def test_meeting_in_the_fixed_array(hip, n, h, w, cin, cout, f, stride):
    """The convolution that allocates nothing takes the same tiles and slices: the same bits."""
    torch = hip.torch
    g = torch.Generator(device=hip.dev).manual_seed(h)
    x = torch.randn(n, h, w, cin, generator=g, device=hip.dev)
    filt = torch.randn(cout, f, f, cin, generator=g, device=hip.dev)
    bias = torch.randn(cout, generator=g, device=hip.dev)
    d = hip.conv_desc(n, h, w, cin, cout, f, f, f // 2, f // 2, stride, stride)
    results = []
    for name in ("nhBlobConvolution", "nhBlobConvolutionNoAlloc"):
        y = torch.empty(n * d.resultHeight * d.resultWidth, cout, device=hip.dev)
        hip.call(name, ctypes.byref(d), hip.p(x), hip.p(filt), hip.p(bias), hip.p(y))
        results.append(y)
    assert torch.equal(*results)
    pad = f // 2
    p = torch.nn.functional.pad(x.double(), (0, 0, pad, pad, pad, pad)).unfold(1, f, stride).unfold(2, f, stride)
    a = p.permute(0, 1, 2, 4, 5, 3).reshape(-1, f * f * cin)
    one = torch.ones(a.shape[0], 1, device=hip.dev, dtype=torch.float64)
    _check(results[0], torch.cat([a, one], 1), torch.cat([filt.double().reshape(cout, -1), bias.double()[:, None]], 1), f * f * cin)
