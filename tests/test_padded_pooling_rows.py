"""An image padded with a constant and the 3 x 3 max pooling over it as one launch, for as many rows that a thread walks down several of them with those
that neighbouring windows share kept in registers."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu

LINE = 1 << 21  # rows of four channels up to which a thread takes one


@pytest.fixture(scope="module")
def streams():
    from test_small_ops_chain import Streams
    s = Streams()
    yield s
    s.close()


# beyond the line: each stride, results whose last rows leave a thread fewer than four, windows that overlap by two rows, one and none, borders on
# all sides and on some; on the line and just below it
@pytest.mark.parametrize("n,h,w,c,border,value,stride,beyond", [
    (16, 97, 100, 64, (1, 1, 1, 1), 0.0, 1, True), (64, 97, 103, 64, (1, 1, 1, 1), -100.0, 2, True), (66, 98, 99, 128, (0, 2, 2, 0), 7.5, 3, True),
    (70, 95, 101, 64, (1, 0, 0, 1), 0.25, 2, True), (64, 64, 128, 64, (1, 1, 1, 1), 0.0, 2, False), (64, 64, 64, 32, (1, 1, 1, 1), 0.0, 1, False)])
def test_rows_kept_in_registers(streams, n, h, w, c, border, value, stride, beyond):
    torch, lib, na = streams.torch, streams.lib, streams.na
    left, right, top, bottom = border
    th, tw = h + top + bottom, w + left + right
    pool = na.PoolingDesc(n, th, tw, c, 3, 3, stride, stride, 0, 0)
    na.check(lib.nhInitPooling(ctypes.byref(pool)))
    rh, rw = pool.resultHeight, pool.resultWidth
    assert (n * rw * (c // 4) * rh > LINE) == beyond
    g = torch.Generator(device=streams.dev).manual_seed(h * w)
    image = torch.randn(n, h, w, c, generator=g, device=streams.dev)
    image[0, 0, 0, 0] = image[n - 1, h // 2, w // 2, c - 1] = image[n // 2, h - 1, w - 1, 1] = float("nan")
    src, dst = na.BlobDesc.of(1, n, 1, h, w, 1, c), na.BlobDesc.of(1, n, 1, th, tw, 1, c)

    def p(t):
        return ctypes.c_void_p(t.data_ptr())

    results = []
    for stream in (streams.plain, streams.deferring):
        padded, pooled = torch.full((n, th, tw, c), -7.0, device=streams.dev), torch.full((n, rh, rw, c), -7.0, device=streams.dev)
        torch.cuda.synchronize()
        na.check(lib.nhBlobResizeImage(stream, ctypes.byref(src), p(image), left, right, top, bottom, 0, ctypes.c_float(value), ctypes.byref(dst), p(padded)))
        na.check(lib.nhBlobMaxPooling(stream, ctypes.byref(pool), p(padded), None, p(pooled)))
        na.check(lib.nhStreamSynchronize(stream))
        results.append((padded, pooled))
    for x, y in zip(*results):
        assert torch.equal(x.view(torch.int32), y.view(torch.int32))
    # and against the windows themselves, where no NaN is among them
    padded, pooled = results[1]
    assert torch.equal(padded[:, top:top + h, left:left + w].nan_to_num(9.0), image.nan_to_num(9.0)) and (padded[:, :top] == value).all() and (padded[:, top + h:] == value).all()
    want = torch.nn.functional.max_pool2d(padded.permute(0, 3, 1, 2), 3, stride).permute(0, 2, 3, 1)
    clean = ~want.isnan()
    assert clean.sum() >= want.numel() - 27 and torch.equal(pooled[clean], want[clean])
