"""Transpositions of a few thousand values, by themselves and several by one launch on a stream that puts calls aside."""
import numpy as np
import pytest

from test_small_ops_chain import ARENA, at, same_bits, streams  # noqa: F401 ( a fixture )

pytestmark = pytest.mark.gpu


def _call(source, result, b, h, m, w, c):
    return ("nhTransposeMatrix", [b, at(source), h, m, w, c, at(result), b * h * m * w * c])


# four channels to a thread and one, off the 16-byte boundaries, plain matrices, a middle dimension, as many values as are taken and more, none
# to be exchanged
@pytest.mark.parametrize("b,h,m,w,c,shift", [(1, 37, 1, 8, 64, 0), (1, 37, 1, 512, 1, 0), (2, 8, 1, 37, 64, 0), (3, 5, 7, 11, 3, 0), (2, 3, 4, 5, 8, 1), (1, 256, 1, 256, 1, 0), (1, 257, 1, 256, 1, 0),
                                             (4, 1, 1, 9, 12, 0), (4, 1, 3, 9, 12, 0), (1, 2, 1, 2, 1, 0), (1, 64, 1, 16, 64, 0), (1, 64, 1, 16, 65, 0)])
def test_one(streams, b, h, m, w, c, shift):  # noqa: F811
    start = np.random.default_rng(h * w).uniform(-1, 1, ARENA).astype(np.float32)
    n = b * h * m * w * c
    want = start.copy()
    want[200000 + shift:200000 + shift + n] = start[shift:shift + n].reshape(b, h, m, w, c).transpose(0, 3, 2, 1, 4).reshape(-1)
    for stream in (streams.plain, streams.deferring):
        assert same_bits(streams.run(stream, [_call(shift, 200000 + shift, b, h, m, w, c)], start), want)


def test_several(streams):  # noqa: F811
    start = np.random.default_rng(3).uniform(-1, 1, ARENA).astype(np.float32)
    n = 37 * 512
    x = [i * 20000 for i in range(12)]
    cells = lambda i, o: _call(x[i], x[o], 1, 37, 1, 8, 64)  # noqa: E731
    plain = lambda i, o: _call(x[i], x[o], 1, 37, 1, 512, 1)  # noqa: E731
    large = _call(0, 262144, 1, 260, 1, 256, 1)
    other = ("nhVectorAbs", [at(x[5]), at(x[5]), n])
    for what, program in {
            "three": [cells(0, 5), plain(1, 6), cells(2, 7)], "six": [cells(0, 5), plain(1, 6), cells(2, 7), plain(3, 8), cells(4, 9), plain(0, 10)],
            "one reads what another wrote": [cells(0, 5), plain(5, 6), cells(6, 7)], "one writes what another reads": [cells(0, 5), plain(1, 0), cells(2, 7)],
            "two write one place": [cells(0, 5), plain(1, 5)], "one writes half of what another reads": [cells(1, 5), _call(x[0], x[1] + 512, 1, 37, 1, 8, 64), cells(2, 7)],
            "a large one in between": [cells(0, 5), large, plain(1, 6)], "a call over a result in between": [cells(0, 5), other, plain(5, 6)],
            "a call behind them": [cells(0, 5), plain(1, 6), other], "a copy in between": [cells(0, 5), _call(x[1], x[6], 1, 1, 1, 37, 512), plain(2, 7)]}.items():
        assert same_bits(streams.run(streams.plain, program, start), streams.run(streams.deferring, program, start)), what
