"""nhSumMatrixRows over up to a few hundred rows, by itself and waiting for the calls in place over its sums."""
import ctypes

import numpy as np
import pytest

from test_small_ops_chain import ARENA, at, same_bits, streams  # noqa: F401 ( a fixture )

pytestmark = pytest.mark.gpu

RESULT, MATRIX, SCALAR, OTHER = 0, 1 << 16, (1 << 16) - 8, ARENA - 4096


# one row, a lane's first row and one beside it, the last height; columns beside a workgroup's runs of 32 and 8, off the 16-byte boundaries
@pytest.mark.parametrize("batch,height,width,shift", [
    (1, 1, 1, 0), (1, 49, 1280, 0), (3, 49, 512, 0), (2, 31, 33, 0), (2, 32, 36, 0), (5, 33, 7, 0), (1, 255, 132, 0), (2, 255, 9, 1), (1, 49, 512, 1), (4, 0, 12, 0)])
def test_sums(streams, batch, height, width, shift):  # noqa: F811
    g = np.random.default_rng(height * width + shift)
    start = g.uniform(-1, 1, ARENA).astype(np.float32)
    m = MATRIX + shift
    values = start[m:m + batch * height * width].reshape(batch, height, width).astype(np.float64)
    want = values.sum(axis=1)
    bound = (height + 2) * 2.0 ** -24 * np.abs(values).sum(axis=1) + 1e-30
    count = batch * width
    for name, first in (("nhSumMatrixRows", 0.0), ("nhSumMatrixRowsAdd", start[:count].reshape(batch, width).astype(np.float64))):
        out = streams.run(streams.plain, [(name, [batch, at(RESULT), at(m), height, width])], start)
        got = out[:count].reshape(batch, width).astype(np.float64)
        assert (np.abs(got - want - first) <= bound + 2.0 ** -23 * np.abs(first)).all()
        assert same_bits(out[count:], start[count:])
    # the calls that follow: its tail, or a call that is none ( part of the sums, the scalar among them, into another vector, an operand more )
    scale = ("nhVectorMultiply", [at(RESULT), at(RESULT), count, at(SCALAR)])
    tails = [[], [scale], [scale, ("nhVectorAddValue", [at(RESULT), at(RESULT), count, at(SCALAR)]), ("nhVectorSqrt", [at(RESULT), at(RESULT), count])],
             [("nhVectorMultiply", [at(RESULT), at(RESULT), max(1, count - 1), at(SCALAR)])], [("nhVectorMultiply", [at(RESULT), at(RESULT), count, at(RESULT)])],
             [("nhVectorMultiply", [at(RESULT), at(OTHER), min(count, 4000), at(SCALAR)])], [("nhVectorAdd", [at(RESULT), at(MATRIX), at(RESULT), count])], [scale] * 11]
    for tail in tails:
        program = [("nhSumMatrixRows", [batch, at(RESULT), at(m), height, width])] + tail
        assert same_bits(streams.run(streams.plain, program, start), streams.run(streams.deferring, program, start))


# on either side of the line between a thread to a column and rows shared by lanes: 511 and 512 runs of 256 columns ( 127 and 128 where they are read one by
# one ), 31 and 32 rows beyond it; more columns than a launch of 8 or of 32 to a workgroup could have
@pytest.mark.parametrize("batch,height,width,shift", [
    (1, 31, 511 * 256, 0), (1, 31, 512 * 256, 0), (1, 32, 512 * 256, 0), (7, 3, 73 * 256, 0), (8, 3, 64 * 256, 0), (1, 40, 127 * 256 - 1, 0), (1, 40, 127 * 256 + 1, 0), (1, 40, 128 * 256, 1),
    (1, 2, (1 << 27) + 5, 0), (1, 1, (1 << 29) + 4, 0)])
def test_wide_matrices(streams, batch, height, width, shift):  # noqa: F811
    torch, lib, na = streams.torch, streams.lib, streams.na
    g = torch.Generator(device=streams.dev).manual_seed(width)
    values = torch.rand(batch * height * width + shift, generator=g, device=streams.dev)[shift:].view(batch, height, width)
    factor = torch.full((1,), 0.5, device=streams.dev)
    want = sum(values[:, i].double() for i in range(height)) if height < 8 else values.double().sum(dim=1)
    results = []
    for stream in (streams.plain, streams.deferring):
        out = torch.full((batch, width), 7.0, device=streams.dev)
        torch.cuda.synchronize()
        na.check(lib.nhSumMatrixRows(stream, batch, ctypes.c_void_p(out.data_ptr()), ctypes.c_void_p(values.data_ptr()), height, width))
        na.check(lib.nhVectorMultiply(stream, ctypes.c_void_p(out.data_ptr()), ctypes.c_void_p(out.data_ptr()), batch * width, ctypes.c_void_p(factor.data_ptr())))
        na.check(lib.nhStreamSynchronize(stream))
        # ( sums of values between 0 and 1, halved )
        assert ((out.double() - want * 0.5).abs() <= (height + 2) * 2.0 ** -24 * want + 1e-30).all()
        results.append(out)
    assert torch.equal(results[0].view(torch.int32), results[1].view(torch.int32))
