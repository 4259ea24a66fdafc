"""Calls recorded into a graph behind a call that was put aside before: what waited is the graph's first launch, and every recorded call is in the
graph, also those that would have joined it."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu

BATCH, ROWS, DIM = 4, 24, 32  # of the attention core; two images of two heads
M, N, K = 40, 48, 64


def _programs(hip, p):
    conv = hip.conv_desc(2, 9, 11, 32, 40, 3, 3, 1, 1, 1, 1)
    side = hip.conv_desc(2, 9, 11, 16, 40, 1, 1, 0, 0, 1, 1)
    count = 2 * 9 * 11 * 40
    wide = 1 << 19
    product = [("nhMultiplyMatrixByTransposedMatrix", ["a", M, K, K, "b", N, K, "c", N, M * N]), ("nhAddVectorToMatrixRows", [1, "c", "c", M, N, "free"])]
    second = [("nhMultiplyMatrixByTransposedMatrix", ["a", M, K, K, "b2", N, K, "c2", N, M * N]), ("nhAddVectorToMatrixRows", [1, "c2", "c2", M, N, "free"])]
    gelu = [("nhVectorMultiply", ["c", "t", M * N, "factor"]), ("nhVectorSigmoid", ["t", "t", M * N]), ("nhVectorEltwiseMultiply", ["c", "t", "c", M * N])]
    junction = [("nhBlobConvolution", [ctypes.byref(conv), "x", "filter", "free", "y"]), ("nhVectorAdd", ["y", "other", "y", count]), ("nhVectorReLU", ["y", "y", count, "top"])]
    shortcut = [junction[0], ("nhBlobConvolution", [ctypes.byref(side), "x", "filter", None, "z"]), ("nhVectorAdd", ["y", "z", "y", count]), junction[2]]
    scores = BATCH * ROWS * ROWS
    attention = [("nhBatchMultiplyMatrixByMatrix", [BATCH, "q", ROWS, DIM, "k", ROWS, "scores", scores]), ("nhVectorMultiply", ["scores", "scores", scores, "factor"]),
                 ("nhMatrixSoftmaxByRows", ["scores", BATCH * ROWS, ROWS, "weights"]),
                 ("nhBatchMultiplyMatrixByMatrix", [BATCH, "weights", ROWS, ROWS, "v", DIM, "context", BATCH * ROWS * DIM]),
                 ("nhTransposeMatrix", [BATCH // 2, "context", 2, 1, ROWS, DIM, "y", BATCH * ROWS * DIM])]
    turns = [("nhTransposeMatrix", [1, "q", 2 * ROWS, 1, 2, DIM, "t", BATCH * ROWS * DIM]), ("nhTransposeMatrix", [1, "k", 2 * ROWS, 1, 2, DIM, "z", BATCH * ROWS * DIM])]
    small_sum = [("nhVectorAdd", ["a", "b", "c", M * K]), ("nhSumMatrixColumns", ["c2", "c", M, K]), ("nhVectorNegMultiply", ["c2", "c2", M, "factor"])]
    large_sum = [("nhVectorAdd", ["wide", "wide2", "wide3", wide]), ("nhSumMatrixColumns", ["c2", "wide3", 512, wide // 512])]
    square = [("nhAddVectorToMatrixColumns", ["a", "c", M, K, "b"]), ("nhVectorEltwiseMultiply", ["c", "c", "c", M * K]), ("nhSumMatrixColumns", ["c2", "c", M, K])]
    columns = [("nhSumMatrixRows", [2, "c2", "a", M // 2, K]), ("nhVectorMultiply", ["c2", "c2", 2 * K, "factor"])]
    whole = {"product": product + gelu, "two products": product + second, "junction": junction, "shortcut": shortcut, "attention": attention, "transpositions": turns, "sum": small_sum,
             "large sum": large_sum, "squares": square, "columns": columns}
    # ( not with the sum over a shortcut in front: that has launched the shortcut, which is not part of the graph then )
    return {"%s, %d before" % (name, i): (calls[:i], calls[i:]) for name, calls in whole.items() for i in range(1, len(calls)) if (name, i) != ("shortcut", 3)}


def test_recorded_joins():
    import nhtest
    import torch
    hip = nhtest.Hip()
    lib, na = hip.lib, hip.na
    g = torch.Generator(device="cuda:0").manual_seed(3)
    start = {name: torch.randn(1 << 16, generator=g, device="cuda:0") for name in ("a", "b", "b2", "free", "x", "filter", "other", "q", "k", "v")}
    start.update((name, torch.randn(1 << 19, generator=g, device="cuda:0")) for name in ("wide", "wide2"))
    results = {name: torch.empty(1 << 16, device="cuda:0") for name in ("c", "c2", "t", "y", "z", "scores", "weights", "context")}
    results["wide3"] = torch.empty(1 << 19, device="cuda:0")
    blobs = dict(start, **results, factor=torch.full((1,), 0.25, device="cuda:0"), top=torch.full((1,), 6.0, device="cuda:0"))
    blobs["filter"] *= 0.1
    plain, stream = torch.cuda.Stream(), torch.cuda.Stream()

    def clear():
        for t in results.values():
            t.fill_(0.5)
        torch.cuda.synchronize()

    def run(on, calls):
        for name, args in calls:
            na.check(getattr(lib, name)(ctypes.c_void_p(on.cuda_stream), *[ctypes.c_void_p(blobs[v].data_ptr()) if isinstance(v, str) else v for v in args]))

    na.check(lib.nhStreamDeferSmallOps(ctypes.c_void_p(stream.cuda_stream), 1))
    try:
        for what, (before, behind) in _programs(hip, blobs).items():
            clear()
            run(plain, before + behind)
            torch.cuda.synchronize()
            want = {name: t.clone() for name, t in results.items()}
            clear()
            run(stream, before)
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=stream):
                run(stream, behind)
            na.check(lib.nhStreamSynchronize(ctypes.c_void_p(stream.cuda_stream)))
            for replay in range(3):
                clear()
                graph.replay()
                torch.cuda.synchronize()
                for name, t in results.items():
                    # ( sums of up to 288 products in two orders, values of a few units )
                    assert torch.allclose(t, want[name], rtol=1e-4, atol=1e-4), (what, name, replay)
    finally:
        na.check(lib.nhStreamDeferSmallOps(ctypes.c_void_p(stream.cuda_stream), 0))
