"""Products that run on the bf16 matrix instructions with operands split in three, and convolutions of such sizes, which do not,
against 64 bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    import nhtest
    return nhtest.Hip()


def _check(got, a, b, k, chunk=128, norm=2.5e-7):
    """a [M,K], b [N,K] in 64 bits. Every result within what its roundings can add up to at worst: twelve for each 16 k of a chunk of up
    to 128 k, each up to 2^-23 of a partial sum ( the instruction does not round to nearest ), one for every chunk, and a few for the
    products of parts that are left out and the epilogue. And all of them, in the 2-norm, within 2.5e-7: 1.2e-7 to 1.8e-7 is
    measured, 3.5e-6 is what it would be without the lowest parts."""
    want = a @ b.T
    bound = (2 * 12 * min(k, chunk) / 16 + k / 64 + 8) * 2.0 ** -24 * (a.abs() @ b.abs().T)
    excess = ((got.double() - want).abs() - bound).max().item()
    assert excess <= 0, excess
    assert ((got.double() - want).norm() / want.norm()).item() < norm


# Each tile shape, with and without a last step of the reduction that is not whole. The last tile row and column partly and all but
# empty, K that ends in each quad of a step.
WHOLE, RAGGED = "false", "true"
TILES_256x128, TILES_128x128, TILES_128x64 = "4, 2, 2, 2, 2", "2, 4, 2, 1, 2", "2, 2, 2, 1, 3"
PRODUCTS = [(8192, 2048, 512, TILES_256x128, WHOLE), (8199, 1921, 528, TILES_256x128, WHOLE), (4097, 1025, 1004, TILES_256x128, RAGGED),
            (8065, 513, 264, TILES_256x128, RAGGED),
            (8192, 512, 512, TILES_128x128, WHOLE), (8192, 512, 2064, TILES_128x128, WHOLE), (1921, 1790, 176, TILES_128x128, WHOLE),
            (8129, 511, 516, TILES_128x128, RAGGED), (8001, 509, 2044, TILES_128x128, RAGGED),
            (1792, 1024, 512, TILES_128x64, WHOLE), (41001, 257, 208, TILES_128x64, WHOLE), (128, 32768, 128, TILES_128x64, WHOLE),
            (20000, 192, 392, TILES_128x64, RAGGED), (8192, 2048, 136, TILES_128x64, RAGGED), (2817, 2042, 132, TILES_128x64, RAGGED)]


@pytest.fixture(scope="module")
def launched():
    import nhtest
    return nhtest.kernel_names([["nt", 1, m, n, k, n] for m, n, k, _, _ in PRODUCTS])


@pytest.mark.parametrize("index", range(len(PRODUCTS)), ids=lambda i: "%dx%dx%d" % PRODUCTS[i][:3])
def test_products(hip, launched, index):
    m, n, k, tiles, ragged = PRODUCTS[index]
    assert launched[index] == ["splitProductKernel<%s, %s>" % (tiles, ragged)]
    torch = hip.torch
    g = torch.Generator(device=hip.dev).manual_seed(m + n + k)
    a = torch.randn(m, k, generator=g, device=hip.dev)
    b = torch.randn(n, k, generator=g, device=hip.dev)
    c = torch.full((m, n), 7.0, device=hip.dev)
    hip.call("nhMultiplyMatrixByTransposedMatrix", hip.p(a), m, k, k, hip.p(b), n, k, hip.p(c), n, c.numel())
    _check(c, a.double(), b.double(), k)


@pytest.mark.parametrize("pitch_a,pitch_b,pitch_c", [(4, 8, 1), (8, 4, 3), (0, 0, 64)])
def test_rows_with_gaps(hip, pitch_a, pitch_b, pitch_c):
    torch = hip.torch
    m, n, k = 8129, 511, 516
    g = torch.Generator(device=hip.dev).manual_seed(pitch_c)
    a = torch.randn(m, k + pitch_a, generator=g, device=hip.dev)
    b = torch.randn(n, k + pitch_b, generator=g, device=hip.dev)
    c = torch.full((m, n + pitch_c), 7.0, device=hip.dev)
    hip.call("nhMultiplyMatrixByTransposedMatrix", hip.p(a), m, k, k + pitch_a, hip.p(b), n, k + pitch_b, hip.p(c), n + pitch_c, c.numel())
    _check(c[:, :n], a[:, :k].double(), b[:, :k].double(), k)
    assert (c[:, n:] == 7.0).all()


def test_batch(hip):
    torch = hip.torch
    batch, m, n, k = 3, 2049, 1020, 264
    g = torch.Generator(device=hip.dev).manual_seed(3)
    a = torch.randn(batch, m, k, generator=g, device=hip.dev)
    b = torch.randn(batch, n, k, generator=g, device=hip.dev)
    c = torch.empty(batch, m, n, device=hip.dev)
    import nhtest
    assert nhtest.kernel_names([["nt", batch, m, n, k, n]])[0][0].startswith("splitProductKernel")
    hip.call("nhBatchMultiplyMatrixByTransposedMatrix", batch, hip.p(a), m, k, hip.p(b), n, hip.p(c), c.numel())
    for i in range(batch):
        _check(c[i], a[i].double(), b[i].double(), k)


def test_errors_lean_to_neither_side(hip):
    """The mean error of many sums: the instruction's own roundings lean to minus infinity by 3e-8 to 1e-7 of the results'
    size. Errors of 1.7e-7 each that lean nowhere have a mean of 1.7e-7 / sqrt( 4 M ) = 8e-11 over independent results; rows and
    columns share operands, so the mean is as of some 512 values: 8e-9, four times that is the bar."""
    torch = hip.torch
    m, n, k = 8192, 512, 1152
    g = torch.Generator(device=hip.dev).manual_seed(9)
    a = torch.rand(m, k, generator=g, device=hip.dev)
    b = torch.randn(n, k, generator=g, device=hip.dev) * 0.05
    c = torch.empty(m, n, device=hip.dev)
    hip.call("nhMultiplyMatrixByTransposedMatrix", hip.p(a), m, k, k, hip.p(b), n, k, hip.p(c), n, c.numel())
    want = a.double() @ b.double().T
    size = want.pow(2).mean().sqrt()
    error = (c.double() - want) / size
    assert error.pow(2).mean().sqrt().item() < 2.5e-7
    assert abs(error.mean().item()) < 3.2e-8


def _patches(torch, x, fh, fw, pad, stride):
    x = torch.nn.functional.pad(x, (0, 0, pad, pad, pad, pad))
    p = x.unfold(1, fh, stride).unfold(2, fw, stride)  # n, ho, wo, c, fh, fw
    return p.permute(0, 1, 2, 4, 5, 3).reshape(-1, fh * fw * x.shape[3])


# odd image sizes, windows over every edge, a filter other than 3x3, stride 2, a last tile row that is partly empty
CONVOLUTIONS = [(65, 33, 31, 128, 256, 3, 1, 1), (33, 59, 61, 144, 130, 3, 1, 1), (64, 65, 63, 128, 256, 3, 1, 2), (33, 41, 37, 80, 96, 5, 2, 1),
                (61, 73, 77, 64, 64, 3, 1, 1), (9, 3, 700, 256, 256, 3, 1, 1), (16, 30, 30, 512, 512, 3, 1, 1)]


@pytest.mark.parametrize("n,h,w,cin,cout,f,pad,stride", CONVOLUTIONS)
def test_convolutions(hip, n, h, w, cin, cout, f, pad, stride):
    torch = hip.torch
    g = torch.Generator(device=hip.dev).manual_seed(n * h * w)
    x = torch.randn(n, h, w, cin, generator=g, device=hip.dev)
    filt = torch.randn(cout, f, f, cin, generator=g, device=hip.dev)
    bias = torch.randn(cout, generator=g, device=hip.dev)
    d = hip.conv_desc(n, h, w, cin, cout, f, f, pad, pad, stride, stride)
    y = torch.empty(n * d.resultHeight * d.resultWidth, cout, device=hip.dev)
    import ctypes
    hip.call("nhBlobConvolution", ctypes.byref(d), hip.p(x), hip.p(filt), hip.p(bias), hip.p(y))
    a = _patches(torch, x.double(), f, f, pad, stride)
    one = torch.ones(a.shape[0], 1, device=hip.dev, dtype=torch.float64)
    a, b = torch.cat([a, one], 1), torch.cat([filt.double().reshape(cout, -1), bias.double()[:, None]], 1)
    # one rounding for every product: at worst all of them add up, in the 2-norm the partial sums grow as a random walk
    want = a @ b.T
    k = f * f * cin
    assert ((y.double() - want).abs() <= (k + 8) * 2.0 ** -24 * (a.abs() @ b.abs().T)).all()
    assert ((y.double() - want).norm() / want.norm()).item() < 2.0 ** -24 * (k / 6) ** 0.5


def test_a_convolution_rounds_alike_at_every_batch(hip):
    """The ReLU behind a convolution decides by a value's sign: what is computed of an image does not change with the images beside
    it. ( The last tiles of a launch may be cut into slices of the reduction: the images in front of them, to the bit. )"""
    torch = hip.torch
    import ctypes
    g = torch.Generator(device=hip.dev).manual_seed(6)
    x = torch.rand(70, 56, 56, 64, generator=g, device=hip.dev)
    filt = torch.randn(64, 3, 3, 64, generator=g, device=hip.dev) * 0.06
    bias = torch.randn(64, generator=g, device=hip.dev) * 0.01
    results = []
    for batch in (64, 70):  # 14.8 and 16.2 GFLOP
        d = hip.conv_desc(batch, 56, 56, 64, 64, 3, 3, 1, 1, 1, 1)
        y = torch.empty(batch, 56, 56, 64, device=hip.dev)
        hip.call("nhBlobConvolution", ctypes.byref(d), hip.p(x), hip.p(filt), hip.p(bias), hip.p(y))
        results.append(y)
    assert torch.equal(results[0][:52], results[1][:52])


def test_values_without_finite_parts(hip):
    """Infinity, NaN, values that round to infinity in bf16, a product that overflows, values whose parts are too small:
    what the fp32 instructions give, and the rows beside them untouched."""
    torch = hip.torch
    m, n, k = 8192, 512, 512
    g = torch.Generator(device=hip.dev).manual_seed(5)
    a = torch.randn(m, k, generator=g, device=hip.dev)
    b = torch.randn(n, k, generator=g, device=hip.dev)
    big = float(np.finfo(np.float32).max)
    a[5, 7] = float("inf")
    a[200, 0] = float("nan")
    a[1000, :] = 0.0
    a[1000, 3] = big
    b[:, 3] = torch.where(b[:, 3].abs() < 1, b[:, 3], 0.5)
    b[17, :] = 1.0
    a[3000, :] = a[3000, :] * 1e-34
    a[5000, :] = 1e38
    a[8191, 511] = -float("inf")
    b[100, 7] = 0.0
    c = torch.empty(m, n, device=hip.dev)
    hip.call("nhMultiplyMatrixByTransposedMatrix", hip.p(a), m, k, k, hip.p(b), n, k, hip.p(c), n, c.numel())
    want = a.double() @ b.double().T
    special = [5, 200, 5000, 8191]
    plain = torch.ones(m, dtype=torch.bool, device=hip.dev)
    plain[special] = False
    plain[3000] = False
    _check(c[plain], a[plain].double(), b.double(), k)
    # ( one in 1e4 of these values is denormal and counts as zero, 1.2e-4 of the others' size at most: 1.2e-6 in the 2-norm at worst )
    _check(c[3000:3001] * 2.0 ** 100, a[3000:3001].double() * 2.0 ** 100, b.double(), k, norm=1.5e-6)
    for row in (5, 200, 8191):
        assert torch.equal(c[row].isnan(), want[row].isnan()), row
        assert torch.equal(c[row].isinf(), want[row].isinf()), row
        assert torch.equal(c[row][c[row].isinf()].double(), want[row][want[row].isinf()]), row
    # sums of 512 values up to 3e38: those far beyond the range are infinite, with their sign ( or NaN where partial sums of
    # both signs left it ), none that stays well inside its running range may be anything but close
    over = want[5000].abs() > 4 * big
    assert not torch.isfinite(c[5000][over]).any()
    assert c[5000, 17] == float("inf")


# ( a product for each of the three tile shapes; no sums next to the smallest normal number, where 2^-126 is lost to any kernel )
@pytest.mark.parametrize("m,n,k", [(8192, 2048, 512), (8192, 512, 1024), (2048, 1024, 516)])
@pytest.mark.parametrize("of_a,of_b", [(-104, 60), (-116, 60), (60, -116), (-125, 100), (-110, 10), (-50, -50), (110, -60), (-90, 103), (45, 45)])
def test_small_values_with_large_partners(hip, m, n, k, of_a, of_b):
    """Normal values whose lower parts would lie under the smallest normal number, against partners that bring the products back
    into the middle of the range; small products of both; values and sums that overflow times the factors of the split. In the 2-norm k products that are added one by one, the partial sums growing as a random walk, are
    off by 2^-24 sqrt( k / 6 ) ( each rounding 2^-24 / sqrt( 3 ) of a partial sum )."""
    torch = hip.torch
    g = torch.Generator(device=hip.dev).manual_seed(m + k)

    def values(rows, power):
        v = torch.rand(rows, k, generator=g, device=hip.dev, dtype=torch.float64) + 1
        sign = torch.randint(0, 2, (rows, k), generator=g, device=hip.dev, dtype=torch.float64) * 2 - 1
        return (v * sign * 2.0 ** power).float()

    a, b = values(m, of_a), values(n, of_b)
    c = torch.empty(m, n, device=hip.dev)
    hip.call("nhMultiplyMatrixByTransposedMatrix", hip.p(a), m, k, k, hip.p(b), n, k, hip.p(c), n, c.numel())
    want = a.double() @ b.double().T
    assert ((c.double() - want).norm() / want.norm()).item() < 2.0 ** -24 * (k / 6) ** 0.5


@pytest.mark.parametrize("m,n,k", [(8192, 2048, 512), (8192, 512, 1024), (2048, 1024, 516)])
def test_one_small_value(hip, m, n, k):
    """One such value in a row of A, one in a row of B, by itself in its row: the results are its products, rounded once."""
    torch = hip.torch
    g = torch.Generator(device=hip.dev).manual_seed(k)
    a = torch.randn(m, k, generator=g, device=hip.dev)
    b = torch.randn(n, k, generator=g, device=hip.dev)
    for one, other, row, at in ((a, b, m - 3, k - 1), (b, a, n // 2, 5)):
        one[row] = 0.0
        one[row, at] = 1.2345678 * 2.0 ** -118
        other[:, at] = torch.rand(other.shape[0], generator=g, device=hip.dev) * 2.0 ** 80
        other[m - 3 if other is a else n // 2, at] = 0.0
    c = torch.empty(m, n, device=hip.dev)
    hip.call("nhMultiplyMatrixByTransposedMatrix", hip.p(a), m, k, k, hip.p(b), n, k, hip.p(c), n, c.numel())
    want = a.double() @ b.double().T
    for got, right in ((c[m - 3], want[m - 3]), (c[:, n // 2], want[:, n // 2])):
        assert ((got.double() - right).abs() <= 2.0 ** -23 * right.abs()).all()
    rest = torch.ones(m, n, dtype=torch.bool, device=hip.dev)
    rest[m - 3] = False
    rest[:, n // 2] = False
    bound = (2 * 12 * 128 / 16 + k / 64 + 8) * 2.0 ** -24 * (a.double().abs() @ b.double().abs().T)  # ( as in _check )
    assert ((c.double() - want).abs() <= bound)[rest].all()


# steps of 16 k: 17 and 18 ( four chunks of four or six steps ), 25, 40, 72 ( ten ), 129
@pytest.mark.parametrize("m,n,k", [(8192, 2048, 264), (8192, 512, 288), (8192, 512, 392), (8192, 512, 640), (8192, 512, 1152), (8192, 512, 2064)])
def test_chunks_of_either_sign_are_as_many(hip, m, n, k):
    """One chunk of the reduction more with one sign than with the other leaves its lean in the results: 3e-9 to 5e-9 of their
    size, all of them measured. With as many of either sign two steps at most are left over, where the chunks have 6 or more to a sign: a
    third of that, 1.6e-9. ( Errors of 1.7e-7 that are independent from result to result add 1.7e-7 / sqrt( m n ) = 8e-11. )"""
    torch = hip.torch
    g = torch.Generator(device=hip.dev).manual_seed(k)
    a = torch.rand(m, k, generator=g, device=hip.dev)
    b = torch.randn(n, k, generator=g, device=hip.dev) * 0.05
    c = torch.empty(m, n, device=hip.dev)
    hip.call("nhMultiplyMatrixByTransposedMatrix", hip.p(a), m, k, k, hip.p(b), n, k, hip.p(c), n, c.numel())
    want = a.double() @ b.double().T
    error = (c.double() - want) / want.pow(2).mean().sqrt()
    assert error.pow(2).mean().sqrt().item() < 2.5e-7
    assert abs(error.mean().item()) < 1.7e-9
