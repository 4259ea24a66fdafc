"""The calls of a normalisation layer, and the sum in front of them, as one pass on a stream that puts calls aside: the bits of the separate
launches, whatever is missing, lies in between or overlaps."""
import numpy as np
import pytest

from test_small_ops_chain import ARENA, at, same_bits, streams  # noqa: F401 ( a fixture )

pytestmark = pytest.mark.gpu

SCALARS = ARENA - 16  # 1 / width, epsilon


def _layout(rows, width, shift=0):
    size = (rows * width + 3) // 4 * 4
    names = ("a", "b", "m", "sq", "y", "z")
    where = {name: i * size + shift for i, name in enumerate(names)}
    end = len(names) * size + 8
    where.update(mean=end, dev=end + rows + 4, scale=(end + 2 * rows + 12) // 4 * 4 + shift)
    where["bias"] = where["scale"] + (width + 3) // 4 * 4
    assert where["bias"] + width < SCALARS
    return where


def _calls(w, rows, width, add=True, out="y"):
    p = {k: at(v) for k, v in w.items()}
    inv, eps, n = at(SCALARS), at(SCALARS + 1), rows * width
    calls = [("nhVectorAdd", [p["a"], p["b"], p["m"], n])] if add else []
    return calls + [
        ("nhSumMatrixColumns", [p["mean"], p["m"], rows, width]),
        ("nhVectorNegMultiply", [p["mean"], p["mean"], rows, inv]),
        ("nhAddVectorToMatrixColumns", [p["m"], p["sq"], rows, width, p["mean"]]),
        ("nhVectorEltwiseMultiply", [p["sq"], p["sq"], p["sq"], n]),
        ("nhSumMatrixColumns", [p["dev"], p["sq"], rows, width]),
        ("nhVectorMultiply", [p["dev"], p["dev"], rows, inv]),
        ("nhVectorAddValue", [p["dev"], p["dev"], rows, eps]),
        ("nhVectorSqrt", [p["dev"], p["dev"], rows]),
        ("nhVectorInv", [p["dev"], p["dev"], rows]),
        ("nhAddVectorToMatrixColumns", [p["m"], p["y"], rows, width, p["mean"]]),
        ("nhMultiplyDiagMatrixByMatrix", [p["dev"], rows, p["y"], width, p["y"], n]),
        ("nhBatchMultiplyMatrixByDiagMatrix", [1, p["y"], rows, width, 0, p["scale"], 0, p[out], n]),
        ("nhAddVectorToMatrixRows", [1, p[out], p[out], rows, width, p["bias"]])]


def _start(seed, rows, width):
    start = np.random.default_rng(seed).uniform(-1, 1, ARENA).astype(np.float32)
    start[SCALARS], start[SCALARS + 1] = 1.0 / width, 1e-5
    return start


def _compare(streams, program, start, what):  # noqa: F811
    plain, deferred = (streams.run(s, program, start) for s in (streams.plain, streams.deferring))
    assert same_bits(plain, deferred), what


# one row, rows that do not fill a workgroup; widths below, at and beside a wavefront's quads, the widest, one too wide, one that is no multiple of four
@pytest.mark.parametrize("rows,width", [(1, 4), (37, 512), (5, 256), (6, 260), (130, 128), (3, 1024), (33, 1028), (9, 2048), (7, 2052), (11, 30), (150, 516)])
def test_whole_layers(streams, rows, width):  # noqa: F811
    start = _start(rows + width, rows, width)
    for shift in (0, 1):
        w = _layout(rows, width, shift)
        for add in (True, False):
            for out in ("y", "z"):
                program = _calls(w, rows, width, add, out)
                _compare(streams, program, start, (shift, add, out))
                _compare(streams, program + program, start, "twice")
    w = _layout(rows, width)
    out = streams.run(streams.deferring, _calls(w, rows, width), start)
    get = lambda name, shape: start[w[name]:w[name] + int(np.prod(shape))].astype(np.float64).reshape(shape)  # noqa: E731
    x = get("a", (rows, width)) + get("b", (rows, width))
    x -= x.mean(1, keepdims=True)
    want = x / np.sqrt((x * x).mean(1, keepdims=True) + 1e-5) * get("scale", (width,)) + get("bias", (width,))
    got = out[w["y"]:w["y"] + rows * width].reshape(rows, width)
    assert np.allclose(got, want, rtol=1e-4, atol=1e-5)


def test_parts_and_calls_in_between(streams):  # noqa: F811
    rows, width = 37, 512
    start = _start(1, rows, width)
    w = _layout(rows, width)
    calls = _calls(w, rows, width)
    n = rows * width
    others = [("nhVectorAbs", [at(w["z"]), at(w["z"]), n]), ("nhVectorAbs", [at(w["mean"]), at(w["mean"]), rows]), ("nhVectorNeg", [at(w["m"]), at(w["m"]), n]),
              ("nhAddVectorToMatrixColumns", [at(w["m"]), at(w["z"]), rows, width, at(w["mean"])]), ("nhSumMatrixColumns", [at(w["mean"]), at(w["sq"]), rows, width]),
              ("nhVectorFill", [at(w["dev"]), 2.0, rows]), ("nhVectorNeg", [at(SCALARS), at(SCALARS), 1])]
    for k in range(len(calls) + 1):
        _compare(streams, calls[:k], start, "the first %d calls" % k)
        _compare(streams, calls[k:], start, "all but the first %d calls" % k)
        for i, other in enumerate(others):
            _compare(streams, calls[:k] + [other] + calls[k:], start, "call %d behind the first %d" % (i, k))
    for k in range(len(calls)):
        _compare(streams, calls[:k] + calls[k + 1:], start, "without call %d" % k)


def test_blobs_that_overlap(streams):  # noqa: F811
    rows, width = 37, 512
    start = _start(2, rows, width)
    n = rows * width
    for what, changes in {
            "the sum over a summand": {"m": ("a", 0)}, "the sum over the other one": {"m": ("b", 0)},
            "the squares over the sum": {"sq": ("m", 0)}, "the result over the sum": {"y": ("m", 0)}, "the result over the squares": {"y": ("sq", 0)},
            "the result over a summand": {"y": ("a", 0)}, "the mean and the deviation in one place": {"dev": ("mean", 0)},
            "the deviation among the means": {"dev": ("mean", 4)}, "the scale in the squares": {"scale": ("sq", 8)}, "the free term in the squares": {"bias": ("sq", n - 512)}}.items():
        w = _layout(rows, width)
        for name, (other, shift) in changes.items():
            w[name] = w[other] + shift
        for add in (True, False):
            _compare(streams, _calls(w, rows, width, add), start, (what, add))
