"""Products for which the kernels of gemm_mfma.hip have shapes of their own, each asked for by the kernel's name, against 64 bits:
results beyond 32-bit offsets, and tiles whose reduction is cut into two halves inside one workgroup."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    import nhtest
    return nhtest.Hip()


def _check(got, a, b, k, free=None, relu=False):
    """a [M,K], b [N,K] in 64 bits: one rounding for every product, all of them one way at worst; in the 2-norm the partial sums grow as
    a random walk ( each rounding 2^-24 / sqrt( 3 ) of one )."""
    want = a @ b.T
    bound = (k + 8) * 2.0 ** -24 * (a.abs() @ b.abs().T)
    if free is not None:
        want = want + free
        bound = bound + (k + 8) * 2.0 ** -24 * free.abs()
    if relu:
        want = want.clamp(min=0)
    error = got.double() - want
    assert (error.abs() <= bound).all()
    assert (error.norm() / want.norm()).item() < 2.0 ** -24 * (k / 6) ** 0.5


# just more than 2^31 bytes; the last tile row and column partly empty, a reduction that ends in a step and one that does not
LARGE = [(32811, 16400, 128), (32800, 16411, 132), (600003, 897, 264)]
HALVES = [(3596, 329, 864), (9755, 203, 1248), (450, 1692, 540), (243, 3642, 508)]
# ( batch, height, width, channels, filters, filter size, padding, stride )
HALVES_OF_CONVOLUTIONS = [(9, 47, 53, 64, 64, 3, 1, 1), (32, 32, 32, 64, 64, 3, 1, 1)]


@pytest.fixture(scope="module")
def launched():
    import nhtest
    calls = [("nt", 1, m, n, k, n) for m, n, k in LARGE + HALVES] + [("conv",) + c for c in HALVES_OF_CONVOLUTIONS]
    return dict(zip((c[1:] for c in calls), nhtest.kernel_names(calls)))


@pytest.mark.parametrize("m,n,k", LARGE)
def test_results_beyond_32_bit_offsets(hip, launched, m, n, k):
    torch = hip.torch
    assert m * n * 4 > 2 ** 31
    assert launched[1, m, n, k, n] == ["longProductKernel<%s>" % ("false" if k % 16 == 0 else "true")]
    g = torch.Generator(device=hip.dev).manual_seed(m)
    a = torch.randn(m, k, generator=g, device=hip.dev)
    b = torch.randn(n, k, generator=g, device=hip.dev)
    free = torch.randn(n, generator=g, device=hip.dev)
    c = torch.full((m, n), 7.0, device=hip.dev)
    hip.call("nhMultiplyMatrixByTransposedMatrix", hip.p(a), m, k, k, hip.p(b), n, k, hip.p(c), n, c.numel())
    rows = (m + 7) // 8
    for i in range(0, m, rows):
        _check(c[i:i + rows], a[i:i + rows].double(), b.double(), k)
    # ( the same behind a pointwise convolution with its free term and its ReLU )
    hip.call("nhPointwiseConvolutionWithActivation", hip.p(a), m, k, hip.p(b), hip.p(free), n, 1, 0.0, hip.p(c))
    for i in range(0, m, rows):
        _check(c[i:i + rows], a[i:i + rows].double(), b.double(), k, free.double(), relu=True)


@pytest.mark.parametrize("m,n,k", HALVES)
def test_halves_of_the_reduction(hip, launched, m, n, k):
    torch = hip.torch
    assert launched[1, m, n, k, n] == ["matMulKernel<64, 64, 2, 2, 0, 0, true, 2>"]
    g = torch.Generator(device=hip.dev).manual_seed(m)
    a = torch.randn(m, k, generator=g, device=hip.dev)
    b = torch.randn(n, k, generator=g, device=hip.dev)
    c = torch.full((m, n), 7.0, device=hip.dev)
    hip.call("nhMultiplyMatrixByTransposedMatrix", hip.p(a), m, k, k, hip.p(b), n, k, hip.p(c), n, c.numel())
    _check(c, a.double(), b.double(), k)


@pytest.mark.parametrize("n,h,w,cin,cout,f,pad,stride", HALVES_OF_CONVOLUTIONS)
def test_halves_of_a_convolution(hip, launched, n, h, w, cin, cout, f, pad, stride):
    torch = hip.torch
    assert launched[n, h, w, cin, cout, f, pad, stride] == ["matMulKernel<64, 64, 2, 2, 6, 0, true, 2>"]
    g = torch.Generator(device=hip.dev).manual_seed(n)
    x = torch.randn(n, h, w, cin, generator=g, device=hip.dev)
    filt = torch.randn(cout, f, f, cin, generator=g, device=hip.dev)
    free = torch.randn(cout, generator=g, device=hip.dev)
    d = hip.conv_desc(n, h, w, cin, cout, f, f, pad, pad, stride, stride)
    y = torch.empty(n * d.resultHeight * d.resultWidth, cout, device=hip.dev)
    hip.call("nhBlobConvolution", ctypes.byref(d), hip.p(x), hip.p(filt), hip.p(free), hip.p(y))
    p = torch.nn.functional.pad(x.double(), (0, 0, pad, pad, pad, pad)).unfold(1, f, stride).unfold(2, f, stride)
    _check(y, p.permute(0, 1, 2, 4, 5, 3).reshape(-1, f * f * cin), filt.double().reshape(cout, -1), f * f * cin, free.double())
