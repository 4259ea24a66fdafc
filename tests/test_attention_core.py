"""The core of an attention layer as one launch on a stream that puts calls aside: products, factor, softmax, weighted sum, exchange of heads
and rows, against 64 bits, and the separate launches for everything that is not that sequence."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def streams():
    from test_small_ops_chain import Streams
    s = Streams()
    yield s
    s.close()


class Layer:
    def __init__(self, streams, images, heads, rows, columns, k, d, seed=0):
        self.s, self.torch = streams, streams.torch
        self.images, self.heads, self.m, self.n, self.k, self.d = images, heads, rows, columns, k, d
        self.b = images * heads
        g = self.torch.Generator(device=streams.dev).manual_seed(seed + rows * columns)
        draw = lambda *shape: self.torch.randn(shape, generator=g, device=streams.dev)  # noqa: E731
        # ( each blob ends where its storage ends, behind NaN of its neighbours: what is read beside it shows )
        self.q, self.kt, self.v = draw(self.b, rows, k), draw(self.b, k, columns), draw(self.b, columns, d)
        self.factor = self.torch.full((1,), 0.125, device=streams.dev)
        self.blobs = {name: self.torch.full((size + 16,), 7.0, device=streams.dev) for name, size in (
            ("scores", self.b * rows * columns), ("weights", self.b * rows * columns), ("context", self.b * rows * d), ("out", self.b * rows * d), ("other", self.b * rows * columns))}

    def calls(self):
        p = {name: t.data_ptr() for name, t in self.blobs.items()}
        q, kt, v, f = (t.data_ptr() for t in (self.q, self.kt, self.v, self.factor))
        b, m, n, k, d = self.b, self.m, self.n, self.k, self.d
        return p, [("nhBatchMultiplyMatrixByMatrix", [b, q, m, k, kt, n, p["scores"], b * m * n]), ("nhVectorMultiply", [p["scores"], p["scores"], b * m * n, f]),
                   ("nhMatrixSoftmaxByRows", [p["scores"], b * m, n, p["weights"]]), ("nhBatchMultiplyMatrixByMatrix", [b, p["weights"], m, n, v, d, p["context"], b * m * d]),
                   ("nhTransposeMatrix", [self.images, p["context"], self.heads, 1, m, d, p["out"], b * m * d])]

    def run(self, stream, program):
        for t in self.blobs.values():
            t.fill_(7.0)
        self.torch.cuda.synchronize()
        for name, args in program:
            self.s.na.check(getattr(self.s.lib, name)(stream, *[ctypes.c_void_p(a) if isinstance(a, int) and a > 1 << 32 else a for a in args]))
        self.s.na.check(self.s.lib.nhStreamSynchronize(stream))
        return {name: t.clone() for name, t in self.blobs.items()}


# one row and one column; rows and columns beside 16, at and beside each run of 64 columns, the most columns; head sizes of fewer groups than
# wavefronts; queries and keys of different lengths; many heads, few
@pytest.mark.parametrize("images,heads,rows,columns,k,d", [
    (1, 8, 37, 37, 64, 64), (1, 1, 1, 1, 16, 1), (2, 3, 16, 17, 32, 33), (1, 2, 33, 64, 64, 64), (1, 4, 15, 65, 48, 64), (3, 2, 47, 128, 64, 16), (1, 2, 20, 129, 64, 64),
    (2, 2, 31, 256, 64, 64), (1, 3, 18, 257, 32, 50), (1, 2, 100, 512, 64, 64), (1, 2, 9, 511, 16, 64), (16, 8, 64, 64, 64, 64)])
def test_against_64_bits(streams, images, heads, rows, columns, k, d):
    layer = Layer(streams, images, heads, rows, columns, k, d)
    torch = streams.torch
    got = layer.run(streams.deferring, layer.calls()[1])
    scores = layer.q.double() @ layer.kt.double().contiguous() * 0.125
    weights = torch.softmax(scores, -1)
    context = weights @ layer.v.double()
    out = context.view(images, heads, rows, d).transpose(1, 2).reshape(-1)
    # a score is a sum of k products of values of the size of one; an error e of a score is one of 2 e, relatively, of a weight
    error = (k + 4) * 2.0 ** -24 * 0.125 * (layer.q.double().abs() @ layer.kt.double().abs().contiguous())
    assert ((got["scores"][:-16].view_as(scores).double() - scores).abs() <= error).all()
    relative = 2 * error.amax(-1, keepdim=True) + (columns + 40) * 2.0 ** -23
    assert ((got["weights"][:-16].view_as(weights).double() - weights).abs() <= relative * weights + 1e-37).all()
    bound = (relative + (columns + 4) * 2.0 ** -24) * (weights @ layer.v.double().abs()) + 1e-37
    assert ((got["context"][:-16].view_as(context).double() - context).abs() <= bound).all()
    assert torch.equal(got["out"][:-16], got["context"][:-16].view(images, heads, rows, d).transpose(1, 2).reshape(-1))
    assert all((t[-16:] == 7.0).all() for t in got.values())
    assert torch.allclose(out, got["out"][:-16].double(), rtol=1e-4, atol=1e-5)


def test_masked_and_infinite_scores(streams):
    """A column of scores of minus infinity, a row of nothing else, a NaN: what the separate calls give."""
    layer = Layer(streams, 1, 4, 20, 70, 64, 64)
    layer.kt[1, 0, 3] = float("-inf")
    layer.q[1, :, 0].abs_()
    layer.q[1, 2, 0] = 0.0  # ( minus infinity times zero: a row with a NaN )
    layer.kt[2, 5, :] = float("inf")
    layer.v[3, 7, :] = float("nan")
    plain, deferred = (layer.run(s, layer.calls()[1]) for s in (streams.plain, streams.deferring))
    for name in plain:
        assert streams.torch.allclose(plain[name], deferred[name], rtol=1e-4, atol=1e-5, equal_nan=True), name


def test_other_sequences(streams):
    layer = Layer(streams, 2, 4, 37, 53, 64, 64)
    # ( scores of the size of two, factor or not, whose 64 products have a sum of sizes of 10: off by no more than 68 * 2^-24 * 10 = 4e-5, and a
    # weight, relatively, by twice that )
    layer.kt *= 0.25
    layer.factor.fill_(0.5)
    p, calls = layer.calls()
    b, m, n, d = layer.b, layer.m, layer.n, layer.d
    count = b * m * n
    f = layer.factor.data_ptr()
    others = [("nhVectorAbs", [p["other"], p["other"], count]), ("nhVectorMultiply", [p["scores"], p["scores"], count, f]), ("nhVectorNeg", [p["weights"], p["weights"], count]),
              ("nhVectorNeg", [p["scores"], p["scores"], count]), ("nhMatrixSoftmaxByRows", [p["scores"], b * m, n, p["other"]]), ("nhVectorAdd", [p["context"], p["out"], p["out"], b * m * d]),
              ("nhTransposeMatrix", [b, p["context"], m, 1, d, 1, p["out"], b * m * d]), ("nhTransposeMatrix", [1, p["context"], b, 1, m, d, p["out"], b * m * d])]
    programs = {}
    for i in range(len(calls) + 1):
        programs["the first %d" % i] = calls[:i]
        programs["without call %d" % i] = calls[:i] + calls[i + 1:]
        for j, other in enumerate(others):
            programs["call %d behind the first %d" % (j, i)] = calls[:i] + [other] + calls[i:]
    name, args = calls[3]
    programs["softmax in place"] = calls[:2] + [("nhMatrixSoftmaxByRows", [p["scores"], b * m, n, p["scores"]]), (name, [b, p["scores"]] + args[2:])]
    programs["a part of the weights"] = calls[:3] + [(name, [b - 1] + args[1:])] + calls[4:]
    programs["other rows"] = calls[:3] + [(name, [b * m, p["weights"], 1, n, args[4], 1, p["context"], b * m])]
    programs["the result over the scores"] = calls[:3] + [(name, args[:6] + [p["scores"], args[7]])]
    programs["the result over the weights' front"] = calls[:3] + [calls[3], ("nhTransposeMatrix", [2, p["context"], 4, 1, m, d, p["weights"], b * m * d])]
    for what, program in programs.items():
        plain, deferred = (layer.run(s, program) for s in (streams.plain, streams.deferring))
        for blob in plain:
            assert streams.torch.allclose(plain[blob], deferred[blob], rtol=1e-4, atol=1e-5, equal_nan=True), (what, blob)


# as many strips as a launch has workgroups for, and one more, which goes out as separate launches: fewer than 2^32 threads to a launch
@pytest.mark.parametrize("batch", [(1 << 24) - 1, 1 << 24])
def test_the_most_workgroups(streams, batch):
    torch = streams.torch
    layer = Layer(streams, batch, 1, 1, 4, 16, 1)
    got = layer.run(streams.deferring, layer.calls()[1])
    at = torch.cat([torch.arange(1000, device=streams.dev), torch.arange(batch - 1000, batch, device=streams.dev)])
    scores = layer.q[at].double() @ layer.kt[at].double().contiguous() * 0.125
    weights = torch.softmax(scores, -1)
    context = weights @ layer.v[at].double()
    # ( 16 products of normal values, their sum of sizes below 100, times 0.125: 20 * 2^-24 * 12.5; weights below one, twice that relatively )
    for name, want in (("scores", scores), ("weights", weights), ("context", context), ("out", context)):
        found = got[name][:batch * want[0].numel()].view(batch, -1)[at].double()
        assert torch.allclose(found, want.reshape(found.shape), rtol=0, atol=1e-4), name
        assert not (got[name][:batch * want[0].numel()] == 7.0).any() and (got[name][batch * want[0].numel():] == 7.0).all()
