"""A convolution, the sum over its result and the ReLU over the sum as one launch on a stream that puts calls aside: the bits of
the three launches, whatever follows or lies in between."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def streams():
    from test_small_ops_chain import Streams
    s = Streams()
    yield s
    s.close()


# every kernel that a convolution may take: few tiles with and without slices, 64 x 64 tiles, slices that meet, the tail of whole rounds,
# two groups in a workgroup, 128 x 32 tiles, short reductions, products split in three, per-lane taps, channels that are no multiple of 4
SHAPES = [(1, 7, 7, 512, 512, 3, 1), (2, 9, 11, 32, 40, 3, 1), (16, 56, 56, 64, 64, 3, 1), (24, 14, 14, 256, 256, 3, 1), (64, 28, 28, 128, 128, 3, 1),
          (32, 32, 32, 64, 64, 3, 1), (40, 28, 28, 32, 32, 3, 1), (32, 28, 28, 32, 96, 1, 1), (64, 14, 14, 512, 256, 1, 1), (8, 28, 28, 64, 128, 1, 2),
          (16, 30, 30, 20, 36, 3, 1), (2, 15, 13, 3, 33, 3, 1), (64, 64, 64, 3, 64, 7, 2)]


def _arguments(d, x, p, y):
    return [ctypes.byref(d), x, p[0], p[1], y]


@pytest.mark.parametrize("n,h,w,cin,cout,f,stride", SHAPES)
def test_sum_and_relu(streams, n, h, w, cin, cout, f, stride):
    import nhtest
    torch, lib, na = streams.torch, streams.lib, streams.na
    hip = nhtest.Hip()
    g = torch.Generator(device=streams.dev).manual_seed(h * cin)

    def blob(*shape):
        return torch.randn(shape, generator=g, device=streams.dev)

    def p(t):
        return ctypes.c_void_p(t.data_ptr())

    d = hip.conv_desc(n, h, w, cin, cout, f, f, f // 2, f // 2, stride, stride)
    shape = (n, d.resultHeight, d.resultWidth, cout)
    count = int(np.prod(shape))
    x, filt, bias, other = blob(n, h, w, cin), blob(cout, f, f, cin), blob(cout), blob(*shape)
    # the shortcut: a pointwise convolution of another image to a result of the same size
    side, side_filt = blob(n, d.resultHeight, d.resultWidth, 16), blob(cout, 1, 1, 16)
    ds = hip.conv_desc(n, d.resultHeight, d.resultWidth, 16, cout, 1, 1, 0, 0, 1, 1)
    other.view(-1)[::97] = float("nan")
    zero, six = torch.zeros(1, device=streams.dev), torch.full((1,), 6.0, device=streams.dev)

    def conv(y):
        return ("nhBlobConvolution", [ctypes.byref(d), p(x), p(filt), p(bias), p(y)])

    def shortcut(s):
        return ("nhBlobConvolution", [ctypes.byref(ds), p(side), p(side_filt), None, p(s)])

    def add(a, b, into, size=count):
        return ("nhVectorAdd", [p(a), p(b), p(into), size])

    def relu(y, top=zero):
        return ("nhVectorReLU", [p(y), p(y), count, p(top)])

    programs = {
        "sum and relu": lambda y, s: [conv(y), add(y, other, y), relu(y)],
        "the operands exchanged, a clipped relu": lambda y, s: [conv(y), add(other, y, y), relu(y, six)],
        "hswish": lambda y, s: [conv(y), add(y, other, y), ("nhVectorHSwish", [p(y), p(y), count])],
        "the sum alone": lambda y, s: [conv(y), add(y, other, y)],
        "two sums": lambda y, s: [conv(y), add(y, other, y), add(y, other, y), relu(y)],
        "into another blob": lambda y, s: [conv(y), add(y, other, s), relu(s)],
        "onto itself": lambda y, s: [conv(y), add(y, y, y), relu(y)],
        "a part": lambda y, s: [conv(y), add(y, other, y, count - 1), relu(y)],
        "a shortcut": lambda y, s: [conv(y), shortcut(s), add(y, s, y), relu(y)],
        "a shortcut, the sum over its result": lambda y, s: [conv(y), shortcut(s), add(y, s, s), relu(s)],
        "a shortcut and another sum": lambda y, s: [conv(y), shortcut(s), add(y, other, y), relu(y)],
        "a shortcut with its relu": lambda y, s: [conv(y), shortcut(s), relu(s), add(y, s, y), relu(y)],
        "two convolutions": lambda y, s: [conv(y), shortcut(s), relu(y)],
        "the second one over the first one's result": lambda y, s: [conv(y), shortcut(y), add(y, other, y), relu(y)],
        "three convolutions": lambda y, s: [conv(y), shortcut(s), conv(y), add(y, s, y), relu(y)],
    }
    for what, program in programs.items():
        results = []
        for stream in (streams.plain, streams.deferring):
            y, s = torch.full(shape, 7.0, device=streams.dev), torch.full(shape, 8.0, device=streams.dev)
            torch.cuda.synchronize()
            for name, args in program(y, s):
                na.check(getattr(lib, name)(stream, *args))
            na.check(lib.nhStreamSynchronize(stream))
            results.append((y.view(torch.int32), s.view(torch.int32)))
        assert torch.equal(results[0][0], results[1][0]), what
        assert torch.equal(results[0][1], results[1][1]), what


def test_a_result_beyond_32_bit_offsets(streams):
    import nhtest
    torch, lib, na = streams.torch, streams.lib, streams.na
    hip = nhtest.Hip()
    size, cin, cout = 2899, 16, 64  # 2.15 GB
    g = torch.Generator(device=streams.dev).manual_seed(5)
    d = hip.conv_desc(1, size, size, cin, cout, 3, 3, 1, 1, 1, 1)
    count = size * size * cout
    assert count * 4 > 2 ** 31
    x, filt, bias, other = (torch.randn(shape, generator=g, device=streams.dev) for shape in ((1, size, size, cin), (cout, 3, 3, cin), (cout,), (count,)))
    top = torch.full((1,), 6.0, device=streams.dev)

    def p(t):
        return ctypes.c_void_p(t.data_ptr())

    for activation in ([], [("nhVectorReLU", count, p(top))], [("nhVectorHSwish", count)]):
        results = []
        for stream in (streams.plain, streams.deferring):
            y = torch.empty(count, device=streams.dev)
            torch.cuda.synchronize()
            na.check(lib.nhBlobConvolution(stream, ctypes.byref(d), p(x), p(filt), p(bias), p(y)))
            na.check(lib.nhVectorAdd(stream, p(y), p(other), p(y), count))
            for name, *args in activation:
                na.check(getattr(lib, name)(stream, p(y), p(y), *args))
            na.check(lib.nhStreamSynchronize(stream))
            results.append(y)
        assert torch.equal(results[0].view(torch.int32), results[1].view(torch.int32))
        del results, y
