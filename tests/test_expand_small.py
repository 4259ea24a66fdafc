"""Inverted residual blocks of a few images: expansion and depthwise convolution in one launch."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu

NONE, RELU, HSWISH = 0, 1, 2


@pytest.fixture(scope="module")
def hip():
    import nhtest
    return nhtest.Hip()


def _act(torch, v, kind, top):
    if kind == RELU:
        return v.clamp(0, top) if top > 0 else v.clamp(min=0)
    return v * (v + 3).clamp(0, 6) / 6 if kind == HSWISH else v


# input channels in each count of 16 that the kernel is built for and between, ending inside a group; rows of a workgroup that do not divide the
# image, images of one row or column, more images than one; pixels that are no multiple of 16; both strides, no free terms
@pytest.mark.parametrize("n,h,w,cin,e,cout,stride,residual,act,free", [
    (1, 112, 112, 16, 96, 24, 2, False, (RELU, 6.0), True), (1, 56, 56, 24, 144, 24, 1, True, (RELU, 6.0), True), (2, 28, 28, 32, 192, 32, 1, True, (RELU, 6.0), True),
    (1, 14, 14, 64, 384, 96, 1, False, (RELU, 0.0), True), (1, 14, 13, 96, 576, 160, 2, False, (RELU, 6.0), False), (2, 7, 7, 160, 960, 320, 1, False, (HSWISH, 0.0), True),
    (1, 1, 1, 4, 16, 8, 1, False, (RELU, 6.0), True), (3, 1, 37, 20, 32, 12, 2, False, (NONE, 0.0), True), (2, 41, 1, 36, 48, 16, 1, False, (RELU, 6.0), True),
    (1, 11, 30, 68, 16, 68, 1, True, (HSWISH, 0.0), False), (5, 9, 10, 100, 80, 24, 2, False, (RELU, 6.0), True), (1, 2, 3, 12, 64, 12, 1, True, (RELU, 1.0), True)])
def test_blocks(hip, n, h, w, cin, e, cout, stride, residual, act, free):
    torch = hip.torch
    g = torch.Generator(device=hip.dev).manual_seed(h * w + cin)

    def blob(*shape):
        return torch.randn(shape, generator=g, device=hip.dev)

    x, we, wd, wo = blob(n, h, w, cin), blob(e, cin) * cin ** -0.5, blob(3, 3, e) / 3, blob(cout, e) * e ** -0.5
    be, bd, bo = (blob(e), blob(e), blob(cout)) if free else (None, None, None)
    d = hip.na.SeparableBlockDesc(n, h, w, cin, e, cout, stride, 1 if residual else 0, act[0], act[1], act[0], act[1])
    size = ctypes.c_size_t(0)
    hip.na.check(hip.lib.nhMobileNetV2BlockWorkspaceSize(ctypes.byref(d), ctypes.byref(size)))
    # ( what the kernel does not write must not count: the work space starts as NaN )
    work = torch.full((size.value // 4 + 1,), float("nan"), device=hip.dev)
    ho, wo_ = (h + stride - 1) // stride, (w + stride - 1) // stride
    y = torch.full((n, ho, wo_, cout), 7.0, device=hip.dev)

    def p(t):
        return hip.p(t) if t is not None else None

    hip.call("nhMobileNetV2Block", ctypes.byref(d), p(x), p(we), p(be), p(wd), p(bd), p(wo), p(bo), p(y), p(work), size)

    def add(v, b):
        return v + b.double() if b is not None else v

    z = _act(torch, add(x.double() @ we.double().T, be), *act)
    windows = torch.nn.functional.pad(z, (0, 0, 1, 1, 1, 1)).unfold(1, 3, stride).unfold(2, 3, stride)
    z = _act(torch, add((windows * wd.double().permute(2, 0, 1)).sum((-1, -2)), bd), *act)
    want = add(z @ wo.double().T, bo) + (x.double() if residual else 0)
    # all values are of the size of one: a sum of k products is off by no more than k + 2 roundings of the sum of their sizes, each
    # stage hands on what the one in front of it was off by
    error = (cin + 4) * cin ** 0.5 + 14 * 3 + (e + 4) * e ** 0.5
    assert (y.double() - want).abs().max() <= error * 2.0 ** -24 * 4
    assert (y.double() - want).norm() <= 3e-6 * want.norm()
