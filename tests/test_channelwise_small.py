"""3x3 depthwise convolutions of a few wavefronts per compute unit: one, two and four pixels to a thread."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    import nhtest
    return nhtest.Hip()


# results of 2^16, 2^17 and 2^18 quads of channels at most, and just beyond; widths that are no multiple of a thread's pixels; images smaller
# than the window
@pytest.mark.parametrize("n,h,w,c,stride,pad", [
    (1, 1, 1, 4, 1, 1), (2, 2, 3, 8, 2, 1), (1, 7, 7, 960, 1, 1), (3, 15, 13, 20, 2, 1), (1, 9, 9, 12, 1, 0), (1, 64, 64, 64, 1, 1), (1, 64, 65, 64, 1, 1),
    (1, 128, 65, 64, 2, 1), (2, 64, 63, 64, 1, 1), (2, 64, 65, 64, 1, 1), (4, 64, 63, 64, 1, 1), (4, 64, 65, 64, 1, 1), (2, 128, 127, 64, 2, 1), (2, 130, 129, 64, 2, 1)])
def test_against_64_bits(hip, n, h, w, c, stride, pad):
    torch = hip.torch
    g = torch.Generator(device=hip.dev).manual_seed(h * w + c)

    def blob(*shape):
        return torch.randn(shape, generator=g, device=hip.dev)

    x, f, bias = blob(n, h, w, c), blob(3, 3, c), blob(c)
    d = hip.na.ConvDesc(n, h, w, c, c, 3, 3, pad, pad, stride, stride, 1, 1, 0, 0)
    hip.na.check(hip.lib.nhInitBlobChannelwiseConvolution(ctypes.byref(d)))
    shape = (n, d.resultHeight, d.resultWidth, c)

    def conv(image, taps, free):
        padded = torch.nn.functional.pad(image.double(), (0, 0, pad, pad, pad, pad)).unfold(1, 3, stride).unfold(2, 3, stride)
        terms = padded * taps.double().permute(2, 0, 1)
        return terms.sum((-1, -2)) + free.double(), terms.abs().sum((-1, -2)) + free.double().abs()

    want, size = conv(x, f, bias)
    bound = 12 * 2.0 ** -24 * size + 1e-30
    y = torch.full((want.numel() + 4,), 7.0, device=hip.dev)
    hip.call("nhBlobChannelwiseConvolution", ctypes.byref(d), hip.p(x), hip.p(f), hip.p(bias), hip.p(y))
    got = y[:-4].view(shape)
    assert ((got.double() - want).abs() <= bound).all()
    assert (y[-4:] == 7.0).all()
    # the ReLU with a threshold in device memory, as a launch of its own and in this one
    top = torch.full((1,), 0.5, device=hip.dev)
    stream = ctypes.c_void_p()
    hip.na.check(hip.lib.nhStreamCreate(ctypes.byref(stream)))
    hip.na.check(hip.lib.nhStreamDeferSmallOps(stream, 1))
    z = torch.empty(shape, device=hip.dev)
    torch.cuda.synchronize()
    hip.na.check(hip.lib.nhBlobChannelwiseConvolution(stream, ctypes.byref(d), hip.p(x), hip.p(f), None, hip.p(z)))
    hip.na.check(hip.lib.nhVectorReLU(stream, hip.p(z), hip.p(z), z.numel(), hip.p(top)))
    hip.na.check(hip.lib.nhStreamSynchronize(stream))
    hip.na.check(hip.lib.nhStreamDestroy(stream))
    want, size = conv(x, f, torch.zeros_like(bias))
    assert ((z.double() - want.clamp(0, 0.5)).abs() <= 12 * 2.0 ** -24 * size + 1e-30).all()
    if stride == 1 and pad == 1:  # the gradient by the input: the taps turned round
        back = torch.empty_like(x)
        hip.call("nhBlobChannelwiseConvolutionBackward", ctypes.byref(d), hip.p(x), hip.p(f), hip.p(back))
        want, size = conv(x, f.flip(0, 1), torch.zeros_like(bias))
        assert ((back.double() - want).abs() <= 12 * 2.0 ** -24 * size + 1e-30).all()
