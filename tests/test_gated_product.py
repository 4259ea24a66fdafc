"""A fully connected layer and the GELU over its result as one launch on a stream that puts calls aside: the bits of the launches, whatever
follows, lies in between or overlaps."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def streams():
    from test_small_ops_chain import Streams
    s = Streams()
    yield s
    s.close()


# few tiles with and without slices, one row, columns beside a tile; products split in three in each shape of tile, a last row of tiles that
# hangs over; the tiles that take no GELU along; off the 16-byte boundaries
@pytest.mark.parametrize("m,n,k,shift", [(37, 2048, 512, 0), (1, 33, 16, 0), (50, 512, 2048, 0), (300, 96, 640, 0), (8192, 512, 512, 0), (8100, 2048, 512, 0), (2200, 640, 768, 0),
                                         (1000, 1500, 64, 0), (20000, 64, 64, 0), (37, 64, 62, 0), (40, 128, 256, 1)])
def test_gelu(streams, m, n, k, shift):
    torch, lib, na = streams.torch, streams.lib, streams.na
    g = torch.Generator(device=streams.dev).manual_seed(m + n)
    draw = lambda *shape: torch.randn(shape, generator=g, device=streams.dev)  # noqa: E731
    a, b, bias, factor = draw(m * k + 4), draw(n * k + 4) * k ** -0.5, draw(n), torch.full((1,), 1.702, device=streams.dev)
    if m >= 16384:
        bias.zero_()  # ( the kernel for short reductions begins its sums with the free term instead of ending them with it )
    count = m * n
    p = {"a": a.data_ptr() + 4 * shift, "b": b.data_ptr() + 4 * shift, "bias": bias.data_ptr(), "factor": factor.data_ptr()}
    blobs = {name: torch.empty(count + 4, device=streams.dev) for name in ("x", "t", "o")}
    p.update((name, t.data_ptr() + 4 * shift) for name, t in blobs.items())
    product = ("nhMultiplyMatrixByTransposedMatrix", ["a", m, k, k, "b", n, k, "x", n, count])
    free = ("nhAddVectorToMatrixRows", [1, "x", "x", m, n, "bias"])

    def gelu(t="t", out="x", x="x"):
        return [("nhVectorMultiply", [x, t, count, "factor"]), ("nhVectorSigmoid", [t, t, count]), ("nhVectorEltwiseMultiply", [x, t, out, count])]

    layer = [product, free] + gelu()
    programs = {"layer": layer, "the factors exchanged": layer[:4] + [("nhVectorEltwiseMultiply", ["t", "x", "x", count])], "into another blob": [product, free] + gelu(out="o"),
                "into the gates": [product, free] + gelu(out="t"), "no free term": [product] + gelu(), "two free terms": [product, free, free] + gelu(),
                "gates over the result": [product, free, ("nhVectorMultiply", ["x", "x", count, "factor"])], "a sum behind it": layer + [("nhVectorAdd", ["x", "t", "o", count])],
                "another product in between": [product, free, product, free] + gelu(), "a call in between": layer[:3] + [("nhVectorAbs", ["o", "o", count])] + layer[3:],
                "a call over the result in between": layer[:3] + [("nhVectorAbs", ["x", "x", count])] + layer[3:],
                "a part": layer[:2] + [("nhVectorMultiply", ["x", "t", count - 1, "factor"])] + layer[3:], "tanh": layer[:3] + [("nhVectorTanh", ["t", "t", count])] + layer[4:],
                "twice": layer + layer, "sums of rows": [product, free, ("nhSumMatrixColumns", ["o", "x", m, n])],
                "the factor in the gates": layer[:2] + [("nhVectorMultiply", ["x", "t", count, "t"])]}
    programs.update(("the first %d calls" % i, layer[:i]) for i in range(1, 5))
    for what, program in programs.items():
        results = []
        for stream in (streams.plain, streams.deferring):
            for name, t in blobs.items():
                t.fill_(0.25)
            torch.cuda.synchronize()
            for name, args in program:
                na.check(getattr(lib, name)(stream, *[ctypes.c_void_p(p[v]) if isinstance(v, str) else v for v in args]))
            na.check(lib.nhStreamSynchronize(stream))
            results.append({name: t.clone() for name, t in blobs.items()})
        for name in blobs:
            x, y = results[0][name], results[1][name]
            # ( the product's own free term is added to its sums on one stream and to what it stored on the other: the same values )
            assert torch.equal(x.view(torch.int32), y.view(torch.int32)), (what, name)
