"""Calls that wait on a stream that puts calls aside, and the pool that the stream takes its scratch memory from: launched in the order in
which they were asked for, with the operands that they were given, at the pool's limit and with its caches full."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu

MB = 1 << 20


class Pooled:
    """A deferring stream bound to a pool with a limit, and a plain stream without one."""

    def __init__(self, limit):
        import torch
        import neoml_amd
        self.torch, self.na, self.lib = torch, neoml_amd, neoml_amd.load()
        self.pool, self.stream, self.plain = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
        neoml_amd.check(self.lib.nhPoolCreate(ctypes.byref(self.pool), 0, limit))
        for s in (self.stream, self.plain):
            neoml_amd.check(self.lib.nhStreamCreate(ctypes.byref(s)))
        neoml_amd.check(self.lib.nhStreamBindPool(self.stream, self.pool))
        neoml_amd.check(self.lib.nhStreamDeferSmallOps(self.stream, 1))

    def __enter__(self):
        return self

    def __exit__(self, *_):
        for s in (self.stream, self.plain):
            self.na.check(self.lib.nhStreamDestroy(s))
        self.na.check(self.lib.nhPoolDestroy(self.pool))

    def alloc(self, size):
        p = ctypes.c_void_p()
        self.na.check(self.lib.nhPoolHeapAlloc(self.pool, size, ctypes.byref(p)))
        return p

    def free(self, p):
        self.na.check(self.lib.nhPoolHeapFree(self.pool, p))

    def call(self, stream, name, *args):
        self.na.check(getattr(self.lib, name)(stream, *[ctypes.c_void_p(a.data_ptr()) if hasattr(a, "data_ptr") else a for a in args]))

    def draw(self, seed, *shape):
        g = self.torch.Generator(device="cuda:0").manual_seed(seed)
        return self.torch.randn(shape, generator=g, device="cuda:0")


# products whose reduction is cut into slices, by the kernel for few tiles and by the tiles that take no GELU along
@pytest.mark.parametrize("m,n,k", [(8, 64, 8192), (50, 512, 2048), (8, 64, 8190)])
@pytest.mark.parametrize("calls", [3, 4, 5])
def test_calls_behind_a_product_at_the_limit(m, n, k, calls):
    with Pooled(8 * MB) as s:
        torch = s.torch
        cached = [s.alloc(1 * MB) for _ in range(8)]  # all that the limit allows, then back into the caches
        for p in cached:
            s.free(p)
        a, b, bias = s.draw(1, m, k), s.draw(2, n, k) * k ** -0.5, s.draw(3, n)
        factor = torch.full((1,), 1.702, device="cuda:0")
        results = []
        for stream in (s.plain, s.stream):
            x, t = torch.full((m, n), 0.25, device="cuda:0"), torch.full((m, n), 0.25, device="cuda:0")
            torch.cuda.synchronize()
            program = [("nhMultiplyMatrixByTransposedMatrix", a, m, k, k, b, n, k, x, n, m * n), ("nhAddVectorToMatrixRows", 1, x, x, m, n, bias),
                       ("nhVectorMultiply", x, t, m * n, factor), ("nhVectorSigmoid", t, t, m * n), ("nhVectorEltwiseMultiply", x, t, x, m * n)]
            for _ in range(2):  # ( what the first launch is refused is there for the second, if the pool can give it )
                for name, *args in program[:calls]:
                    s.call(stream, name, *args)
                s.na.check(s.lib.nhStreamSynchronize(stream))
                results.append((x.clone(), t.clone()))
        # sums of k products of values of the size of one and of k^-1/2 in two orders, times what follows, which is no steeper than 1.702 and grows no
        # faster than 1.1 times its argument
        bound = 4 * (k + 40) * 2.0 ** -24 * k ** 0.5
        for i in range(2):
            for x, y in zip(results[i], results[2 + i]):
                assert (x - y).abs().max() <= bound, (i, float((x - y).abs().max()))


def test_scratch_is_no_operand_of_a_waiting_call():
    """An operand that went back to the pool behind the call that reads it is not what that call's launch gets as scratch memory."""
    m, n, k = 8, 64, 8192
    for size in [16 << 10] + [MB * part // 8 for part in (1, 2, 3, 4, 6, 8, 12, 16)]:
        with Pooled(0) as s:
            torch = s.torch
            a, b, bias = s.draw(1, m, k), s.draw(2, n, k) * k ** -0.5, s.draw(3, n)
            own = s.alloc(size)
            operand = a if size >= a.numel() * 4 else bias
            s.call(s.plain, "nhCopyDeviceToDevice", own, operand, operand.numel() * 4)
            s.na.check(s.lib.nhStreamSynchronize(s.plain))
            x = torch.zeros((m, n), device="cuda:0")
            torch.cuda.synchronize()
            s.call(s.stream, "nhMultiplyMatrixByTransposedMatrix", own if operand is a else a, m, k, k, b, n, k, x, n, m * n)
            s.call(s.stream, "nhAddVectorToMatrixRows", 1, x, x, m, n, own if operand is bias else bias)
            s.free(own)
            s.na.check(s.lib.nhStreamSynchronize(s.stream))
            want = a.double() @ b.double().T + bias.double()
            bound = (k + 40) * 2.0 ** -24 * (a.double().abs() @ b.double().abs().T + bias.double().abs())
            assert ((x.double() - want).abs() <= bound).all(), size


def test_an_operand_is_not_released_under_a_waiting_call():
    """... nor is it given back to the device for the launch's sake, at the pool's limit."""
    m, n, k = 8, 64, 8192
    with Pooled(8 * MB) as s:
        torch = s.torch
        a, b, bias = s.draw(1, m, k), s.draw(2, n, k) * k ** -0.5, s.draw(3, n)
        blocks = [s.alloc(1 * MB) for _ in range(8)]
        s.call(s.plain, "nhCopyDeviceToDevice", blocks[0], a, m * k * 4)
        s.na.check(s.lib.nhStreamSynchronize(s.plain))
        x = torch.zeros((m, n), device="cuda:0")
        torch.cuda.synchronize()
        s.call(s.stream, "nhMultiplyMatrixByTransposedMatrix", blocks[0], m, k, k, b, n, k, x, n, m * n)
        s.call(s.stream, "nhAddVectorToMatrixRows", 1, x, x, m, n, bias)
        for p in blocks:
            s.free(p)
        s.na.check(s.lib.nhStreamSynchronize(s.stream))
        want = a.double() @ b.double().T + bias.double()
        bound = (k + 40) * 2.0 ** -24 * (a.double().abs() @ b.double().abs().T + bias.double().abs())
        assert ((x.double() - want).abs() <= bound).all()


# what gives memory back to the device while a product waits that will ask the same pool for scratch: a request at the limit, the release of a
# block that was not from the caches, a clean-up, a stack, the scratch of another stream, a product on another stream
@pytest.mark.parametrize("what", ["request", "direct block", "clean-up", "stack", "stack of blocks", "scratch", "product"])
def test_memory_given_back_while_a_product_waits(what):
    m, n, k = 8, 64, 8192
    with Pooled(8 * MB) as s:
        torch, lib, na = s.torch, s.lib, s.na
        a, b, bias = s.draw(1, m, k), s.draw(2, n, k) * k ** -0.5, s.draw(3, n)
        x, y = torch.zeros((m, n), device="cuda:0"), torch.zeros((m, n), device="cuda:0")
        other = ctypes.c_void_p()
        na.check(lib.nhStreamCreate(ctypes.byref(other)))
        na.check(lib.nhStreamBindPool(other, s.pool))
        try:
            direct, top = ctypes.c_void_p(), []
            if what == "direct block":
                na.check(lib.nhPoolSetReuseMemoryMode(s.pool, 0))
                direct = s.alloc(1 * MB)
                na.check(lib.nhPoolSetReuseMemoryMode(s.pool, 1))
            if what == "stack of blocks":
                na.check(lib.nhPoolSetReuseMemoryMode(s.pool, 0))
            if what in ("stack", "stack of blocks"):
                for size in (100000, 200000):
                    top.append(ctypes.c_void_p())
                    na.check(lib.nhPoolStackAlloc(s.pool, size, ctypes.byref(top[-1])))
            if what == "scratch":
                na.check(lib.nhPoolSetReuseMemoryMode(s.pool, 0))
                s.call(other, "nhMultiplyMatrixByTransposedMatrix", a, m, k, k, b, n, k, y, n, m * n)
                na.check(lib.nhStreamSynchronize(other))
            if what in ("request", "clean-up", "product"):
                for p in [s.alloc(1 * MB) for _ in range(8)]:
                    s.free(p)
            torch.cuda.synchronize()
            s.call(s.stream, "nhMultiplyMatrixByTransposedMatrix", a, m, k, k, b, n, k, x, n, m * n)
            s.call(s.stream, "nhAddVectorToMatrixRows", 1, x, x, m, n, bias)
            if what == "request":
                s.free(s.alloc(3 * MB))
            elif what == "direct block":
                s.free(direct)
            elif what == "clean-up":
                na.check(lib.nhPoolCleanUp(s.pool))
            elif what in ("stack", "stack of blocks"):
                while top:
                    na.check(lib.nhPoolStackFree(s.pool, top.pop()))
                na.check(lib.nhPoolStackAlloc(s.pool, 400000, ctypes.byref(direct)))
                na.check(lib.nhPoolStackFree(s.pool, direct))
                na.check(lib.nhPoolCleanUp(s.pool))
            elif what == "scratch":
                na.check(lib.nhStreamReleaseScratch(other))
            else:
                s.call(other, "nhMultiplyMatrixByTransposedMatrix", a, m, k, k, b, n, k, y, n, m * n)
                na.check(lib.nhStreamSynchronize(other))
            na.check(lib.nhStreamSynchronize(s.stream))
            used, cached = ctypes.c_size_t(), ctypes.c_size_t()
            na.check(lib.nhPoolGetCurrentMemoryUsage(s.pool, ctypes.byref(used)))
            na.check(lib.nhPoolGetMemoryInPools(s.pool, ctypes.byref(cached)))
            assert cached.value <= used.value <= 8 * MB
        finally:
            na.check(lib.nhStreamDestroy(other))
        want = a.double() @ b.double().T
        bound = (k + 40) * 2.0 ** -24 * (a.double().abs() @ b.double().abs().T + bias.double().abs())
        assert ((x.double() - (want + bias.double())).abs() <= bound).all()
        if what in ("scratch", "product"):
            assert ((y.double() - want).abs() <= bound).all()


def test_threads_at_the_limit_of_one_pool():
    """Threads that ask a pool at its limit, each with what the others need in its caches at times, and with calls that wait on streams of
    their own: every request that fits is met."""
    import threading
    m, n, k, threads = 8, 64, 8192, 4
    # one thread's caches come to 3.75 MB at most, so 14 hold what three keep and the largest request of the fourth, and a little scratch; not
    # what all four would keep
    sizes = [MB // 2, MB * 3 // 4, MB, MB * 3 // 2]
    with Pooled(14 * MB) as s:
        torch, lib, na = s.torch, s.lib, s.na
        a, b, bias = s.draw(1, m, k), s.draw(2, n, k) * k ** -0.5, s.draw(3, n)
        results = [torch.zeros((m, n), device="cuda:0") for _ in range(threads)]
        torch.cuda.synchronize()
        errors = []

        def work(i):
            stream = ctypes.c_void_p()
            try:
                na.check(lib.nhStreamCreate(ctypes.byref(stream)))
                na.check(lib.nhStreamBindPool(stream, s.pool))
                na.check(lib.nhStreamDeferSmallOps(stream, 1))
                for r in range(40):
                    s.call(stream, "nhMultiplyMatrixByTransposedMatrix", a, m, k, k, b, n, k, results[i], n, m * n)
                    s.call(stream, "nhAddVectorToMatrixRows", 1, results[i], results[i], m, n, bias)
                    p = s.alloc(sizes[(r + i) % 4])
                    s.call(stream, "nhVectorFill", p, ctypes.c_float(1.0), 1024)
                    s.free(p)
                    if r % 16 == 15:
                        na.check(lib.nhPoolCleanUp(s.pool))
                na.check(lib.nhStreamSynchronize(stream))
            except Exception as e:  # noqa: BLE001
                errors.append(repr(e))
            finally:
                lib.nhStreamDestroy(stream)
                lib.nhPoolCleanUp(s.pool)

        running = [threading.Thread(target=work, args=(i,)) for i in range(threads)]
        for t in running:
            t.start()
        for t in running:
            t.join(60)
        assert not any(t.is_alive() for t in running)
        assert not errors, errors
        want = a.double() @ b.double().T + bias.double()
        bound = (k + 40) * 2.0 ** -24 * (a.double().abs() @ b.double().abs().T + bias.double().abs())
        for x in results:
            assert ((x.double() - want).abs() <= bound).all()


def test_another_thread_frees_what_a_waiting_call_reads():
    """A thread may free the source of a convolution as soon as the call has returned, also while the thread that asked for it is in the call
    behind it."""
    import threading
    import nhtest
    hip = nhtest.Hip()
    d = hip.conv_desc(2, 32, 32, 32, 64, 3, 3, 1, 1, 1, 1)
    with Pooled(0) as s:
        torch, lib, na = s.torch, s.lib, s.na
        x, filt, zero = s.draw(1, 2, 32, 32, 32), s.draw(2, 64, 3, 3, 32) / 17, torch.zeros(1, device="cuda:0")
        want, y = torch.empty(2, 32, 32, 64, device="cuda:0"), torch.empty(2, 32, 32, 64, device="cuda:0")
        s.call(s.plain, "nhBlobConvolution", ctypes.byref(d), x, filt, None, want)
        s.call(s.plain, "nhVectorReLU", want, want, want.numel(), zero)
        na.check(lib.nhStreamSynchronize(s.plain))
        errors = []
        for _ in range(20):
            source, asked = ctypes.c_void_p(), threading.Event()
            na.check(lib.nhRawAlloc(ctypes.byref(source), x.numel() * 4))
            s.call(s.plain, "nhCopyDeviceToDevice", source, x, x.numel() * 4)
            na.check(lib.nhStreamSynchronize(s.plain))

            def free():
                asked.wait()
                if lib.nhRawFree(source) != 0:
                    errors.append(na.last_error())

            thread = threading.Thread(target=free)
            thread.start()
            s.call(s.stream, "nhBlobConvolution", ctypes.byref(d), source, filt, None, y)
            asked.set()
            s.call(s.stream, "nhVectorReLU", y, y, y.numel(), zero)
            na.check(lib.nhStreamSynchronize(s.stream))
            thread.join(60)
            assert not thread.is_alive() and not errors
            # ( sent out with its ReLU or in front of it: the same convolution, the same bits )
            assert torch.equal(y.view(torch.int32), want.view(torch.int32))
