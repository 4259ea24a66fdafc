"""Which kernels the engine's calls launch: a program of its own, so that the profiler it asks stays out of the tests' process.

Standard input: a JSON list of calls, ["nt", batch, m, n, k, pitch of C], ["conv", n, h, w, cin, cout, filter size, padding, stride],
["conv_no_alloc", ...the same], ["conv_backward", ...the same] or ["lstm", steps, batch, width, hidden]. Standard output: a JSON list of lists of the kernels' names."""
import ctypes
import json
import sys

import nhtest


def main():
    from torch.profiler import ProfilerActivity, profile
    hip = nhtest.Hip()
    torch = hip.torch

    def blob(*shape):
        return torch.zeros(shape, device=hip.dev)

    def bound(call):
        kind, *sizes = call
        if kind == "nt":
            batch, m, n, k, pitch = sizes
            a, b, c = blob(batch, m, k), blob(batch, n, k), blob(batch, m, pitch)
            if batch > 1:
                return (a, b, c), lambda: hip.call("nhBatchMultiplyMatrixByTransposedMatrix", batch, hip.p(a), m, k, hip.p(b), n, hip.p(c), c.numel())
            return (a, b, c), lambda: hip.call("nhMultiplyMatrixByTransposedMatrix", hip.p(a), m, k, k, hip.p(b), n, k, hip.p(c), pitch, c.numel())
        if kind == "lstm":
            steps, batch, width, hidden = sizes
            size = ctypes.c_size_t(0)
            hip.na.check(hip.lib.nhLstmWorkspaceSize(hidden, width, steps, batch, ctypes.byref(size)))
            x, y, work = blob(steps, batch, width), blob(steps, batch, hidden), blob(size.value // 4 + 1)
            w_in, w_rec, free = blob(4 * hidden, width), blob(4 * hidden, hidden), blob(4 * hidden)
            return (x, y, work, w_in, w_rec, free), lambda: hip.call(
                "nhLstm", hidden, width, hip.p(w_in), hip.p(free), hip.p(w_rec), hip.p(free), 0, steps, batch, None, None, hip.p(x), None,
                hip.p(y), hip.p(work), size)
        batch, h, w, cin, cout, f, pad, stride = sizes
        d = hip.conv_desc(batch, h, w, cin, cout, f, f, pad, pad, stride, stride)
        x, filt, y = blob(batch, h, w, cin), blob(cout, f, f, cin), blob(batch, d.resultHeight, d.resultWidth, cout)
        if kind in ("conv", "conv_no_alloc"):
            return (x, filt, y), lambda: hip.call("nhBlobConvolution" if kind == "conv" else "nhBlobConvolutionNoAlloc", ctypes.byref(d), hip.p(x), hip.p(filt), None, hip.p(y))
        size = ctypes.c_size_t(0)
        hip.na.check(hip.lib.nhBlobConvolutionBackwardWorkspaceSize(ctypes.byref(d), ctypes.byref(size)))
        work = blob(size.value // 4 + 1)
        return (x, filt, y, work), lambda: hip.call("nhBlobConvolutionBackward", ctypes.byref(d), hip.p(y), hip.p(filt), None, hip.p(x), hip.p(work), size)

    names = []
    for call in json.load(sys.stdin):
        keep, run = bound(call)
        run()  # ( scratch memory is there behind the first call )
        torch.cuda.synchronize()
        with profile(activities=[ProfilerActivity.CUDA]) as trace:
            run()
            torch.cuda.synchronize()
        names.append([e.key for e in trace.key_averages() if "nh::" in e.key])
        del keep
    print(json.dumps(names))


if __name__ == "__main__":
    main()
