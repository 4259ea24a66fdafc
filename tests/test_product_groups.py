"""Fully connected layers over one input as one launch on a stream that puts calls aside: what the separate launches give, whatever
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


# one row, ragged tiles and reductions, as many tiles as are taken and one row more, few tiles whose product alone would be cut into slices, more
# than a group is for
@pytest.mark.parametrize("m,n,k", [(37, 512, 512), (1, 33, 16), (50, 100, 260), (128, 512, 512), (129, 512, 256), (20, 64, 2048), (300, 1000, 64), (37, 51, 62)])
def test_groups(streams, m, n, k):
    torch, lib, na = streams.torch, streams.lib, streams.na
    g = torch.Generator(device=streams.dev).manual_seed(m + n)
    draw = lambda *shape: torch.randn(shape, generator=g, device=streams.dev)  # noqa: E731
    count, size = m * n, max(m * n, n * k, m * k)
    start = {name: draw(size) * (k ** -0.5 if name[0] == "w" else 1.0) for name in ("a", "w0", "w1", "w2", "w3", "c0", "c1", "c2", "c3", "t")}
    start.update(("b%d" % i, draw(n)) for i in range(4))
    start["factor"] = torch.full((1,), 1.702, device=streams.dev)
    blobs = {name: torch.empty_like(t) for name, t in start.items()}

    def product(w, c, a="a", rows=m):
        return ("nhMultiplyMatrixByTransposedMatrix", [a, rows, k, k, w, n, k, c, n, rows * n])

    def free(c, b, rows=m):
        return ("nhAddVectorToMatrixRows", [1, c, c, rows, n, b])

    def layer(i):
        return [product("w%d" % i, "c%d" % i), free("c%d" % i, "b%d" % i)]

    three = layer(0) + layer(1) + layer(2)
    programs = {"three": three, "two": layer(0) + layer(1), "four": three + layer(3), "the last without its free term": three[:5], "the second without": three[:3] + three[4:],
                "one free term for all": [product("w0", "c0"), free("c0", "b0"), product("w1", "c1"), free("c1", "b0"), product("w2", "c2"), free("c2", "b0")],
                "one result": layer(0) + [product("w1", "c0"), free("c0", "b1")], "a result that is the next one's input": layer(0) + [product("w1", "c1", "c0"), free("c1", "b1")],
                "a result over the input": layer(0) + [product("w1", "a"), free("a", "b1")] + layer(2), "a result over the next one's weights": [product("w0", "w1"), free("w1", "b0")] + layer(1),
                "a result over the one before's weights": layer(0) + [product("w1", "w0"), free("w0", "b1")],
                "a result over the free term of the one before": [product("w0", "c0"), free("c0", "t"), product("w1", "t"), free("t", "b1")],
                "a free term that is a result": layer(0) + [product("w1", "c1"), free("c1", "c0")],
                "fewer rows": layer(0) + ([product("w1", "c1", rows=m - 1), free("c1", "b1", m - 1)] if m > 1 else []) + layer(2),
                "a call in between": layer(0) + [("nhVectorAbs", ["t", "t", count])] + layer(1) + layer(2),
                "a call over a result in between": layer(0) + layer(1) + [("nhVectorAbs", ["c0", "c0", count])] + layer(2),
                "a GELU behind them": three + [("nhVectorMultiply", ["c2", "t", count, "factor"]), ("nhVectorSigmoid", ["t", "t", count]), ("nhVectorEltwiseMultiply", ["c2", "t", "c2", count])],
                "twice": three + three}
    for what, program in programs.items():
        results = []
        for stream in (streams.plain, streams.deferring):
            for name, t in blobs.items():
                t.copy_(start[name])
            torch.cuda.synchronize()
            for name, args in program:
                na.check(getattr(lib, name)(stream, *[ctypes.c_void_p(blobs[v].data_ptr()) if isinstance(v, str) else v for v in args]))
            na.check(lib.nhStreamSynchronize(stream))
            results.append({name: t.clone() for name, t in blobs.items()})
        for name in blobs:
            x, y = results[0][name].double(), results[1][name].double()
            # sums of k products of values of the size of one and of k^-1/2, in two orders: off by no more than 2 ( k + 40 ) 2^-24 of k^1/2 ( where one
            # product's result is the next one's input, of k^1/2 of the one and k^1/2 of the other )
            bound = 2 * (k + 40) * 2.0 ** -24 * max(1.0, k ** 0.5) * (max(1.0, k ** 0.5) if "input" in what else 1.0) * 4
            assert (x - y).abs().max() <= bound, (what, name)
    # and against 64 bits
    for i in range(3):
        for name, t in blobs.items():
            t.copy_(start[name])
    torch.cuda.synchronize()
    for name, args in three:
        na.check(getattr(lib, name)(streams.deferring, *[ctypes.c_void_p(blobs[v].data_ptr()) if isinstance(v, str) else v for v in args]))
    na.check(lib.nhStreamSynchronize(streams.deferring))
    a = start["a"][:m * k].view(m, k).double()
    for i in range(3):
        w, b = start["w%d" % i][:n * k].view(n, k).double(), start["b%d" % i].double()
        got = blobs["c%d" % i][:count].view(m, n).double()
        bound = (k + 40) * 2.0 ** -24 * (a.abs() @ w.abs().T + b.abs())
        assert ((got - (a @ w.T + b)).abs() <= bound).all()
        assert torch.equal(blobs["c%d" % i][count:], start["c%d" % i][count:])
