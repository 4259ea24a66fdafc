"""The work that a program built on this engine has it do, as cases to time and to compare.

A case is one pass of a network (or of one layer) issued as the engine calls that NeoML's layers make for it, through the
C ABI of libneoml_hip.so, on blobs that stay in device memory. As a network keeps them, the weights, the intermediate blobs, the
workspaces and the calls with their arguments bound exist before the pass. The pass runs on a stream that puts small calls
aside and lets independent LSTMs overlap, which is what the engine adapter asks for its own stream; both are switched off
at its end, which sends out whatever still waits without waiting for the GPU.

    conv      one 3x3 convolution layer with its ReLU: the smallest unit of work
    resnet    image classification, ResNet-18-style: 7x7/2 stem, pad + pooling, four stages of residual blocks, FC, softmax
    mobilenet image classification, MobileNetV2-style: inverted residual blocks, fused as NeoML's graph optimizer leaves them
              or call by call
    encoder   a stack of transformer encoder layers over sequences of vectors
    lines     a text line recogniser: convolutions, two bidirectional LSTM layers, FC, the engine part of CTC decoding
    train     a training step of a residual block: forward, the gradients by input and parameters, the momentum solver
"""
import ctypes
import math

import torch

import neoml_amd

FLOAT = 4  # bytes


def listed():
    return [
        # one layer by itself: 22 us of GPU work, where launching it counts
        {"name": "conv_b32", "kind": "conv", "batch": 32, "height": 32, "width": 32, "cin": 64, "cout": 64},
        # one picture as it arrives: latency, few tiles per layer, the weights are most of the traffic
        {"name": "resnet_b1", "kind": "resnet", "batch": 1, "height": 224, "width": 224},
        # a handful of pictures of a size that is no power of anything
        {"name": "resnet_b9_odd", "kind": "resnet", "batch": 9, "height": 187, "width": 211},
        # throughput: the batch the framework's benchmark uses
        {"name": "resnet_b64", "kind": "resnet", "batch": 64, "height": 224, "width": 224},
        {"name": "mobilenet_b1", "kind": "mobilenet", "batch": 1, "height": 224, "width": 224, "fused": True},
        # the same network where no optimizer has been over the graph, at a middling batch
        {"name": "mobilenet_b24_calls", "kind": "mobilenet", "batch": 24, "height": 160, "width": 192, "fused": False},
        {"name": "mobilenet_b128", "kind": "mobilenet", "batch": 128, "height": 224, "width": 224, "fused": True},
        # one short sentence, its length odd
        {"name": "encoder_b1_s37", "kind": "encoder", "layers": 6, "batch": 1, "seq": 37, "d": 512, "heads": 8},
        {"name": "encoder_b32_s256", "kind": "encoder", "layers": 6, "batch": 32, "seq": 256, "d": 512, "heads": 8},
        # one short line, its width odd
        {"name": "lines_b1_w203", "kind": "lines", "batch": 1, "width": 203},
        {"name": "lines_b64_w512", "kind": "lines", "batch": 64, "width": 512},
        # a training step of a first-stage block of the image network at its benchmark's batch
        {"name": "train_b64", "kind": "train", "batch": 64, "height": 56, "width": 56, "cin": 64, "cout": 64, "stride": 1},
    ]


def _spread(rng, low, high):
    """a whole number, spread over the logarithm of its range"""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    case = _draw(rng)
    while work(case)["flops"] > 3.3e11:  # the largest listed case
        case["batch"] = case["batch"] * 3 // 4
    return case


def _draw(rng):
    kind = rng.choice(["conv", "resnet", "resnet", "mobilenet", "mobilenet", "encoder", "encoder", "lines", "lines", "train", "train"])
    if kind == "conv":
        size = _spread(rng, 7, 112)
        return {"kind": kind, "batch": _spread(rng, 1, 64), "height": size, "width": max(7, size + rng.randint(-3, 3)),
                "cin": 4 * _spread(rng, 8, 64), "cout": 4 * _spread(rng, 8, 64)}
    if kind == "resnet":
        return {"kind": kind, "batch": _spread(rng, 1, 64), "height": rng.randint(96, 224), "width": rng.randint(96, 224)}
    if kind == "mobilenet":
        return {"kind": kind, "batch": _spread(rng, 1, 128), "height": rng.randint(96, 224), "width": rng.randint(96, 224),
                "fused": rng.random() < 0.6}
    if kind == "encoder":
        seq = _spread(rng, 16, 512)
        heads = rng.choice([4, 6, 8])
        return {"kind": kind, "layers": rng.randint(2, 6), "batch": _spread(rng, 1, max(1, 8192 // seq)), "seq": seq, "d": 64 * heads, "heads": heads}
    if kind == "lines":
        return {"kind": kind, "batch": _spread(rng, 1, 64), "width": _spread(rng, 64, 512)}
    # the blocks of the image network's stages: wider where the image is smaller, the first of a stage with stride 2
    stage = rng.randint(0, 3)
    size = max(7, (56 >> stage) + rng.randint(-3, 0))
    stride = rng.choice([1, 1, 2]) if stage < 3 else 1
    cin = 64 << stage
    return {"kind": kind, "batch": _spread(rng, 2, 64), "height": size, "width": max(7, size + rng.randint(-2, 2)), "cin": cin,
            "cout": cin * stride, "stride": stride}


# ---- a network's calls ---------------------------------------------------------------------------------------------


class Calls:
    """Blobs on the GPU and the engine calls over them, arguments bound; shapes are N,H,W,C. Counts the work as it goes: the
    floating point operations of the products and the convolutions, 4 bytes per weight."""

    def __init__(self, seed):
        self.lib = neoml_amd.load()
        self.device = torch.device("cuda:0")
        self.random = torch.Generator(device=self.device)
        self.random.manual_seed(seed)
        self.stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        self.calls = []
        self.keep = []
        self.scalars = {}
        self.work = None

    # blobs
    def empty(self, *shape, dtype=torch.float32):
        t = torch.empty(shape, dtype=dtype, device=self.device)
        self.keep.append(t)
        return t

    def normal(self, std, *shape):
        t = torch.randn(shape, generator=self.random, device=self.device) * std
        self.keep.append(t)
        return t

    def uniform(self, low, high, *shape):
        t = torch.rand(shape, generator=self.random, device=self.device) * (high - low) + low
        self.keep.append(t)
        return t

    def scalar(self, value):
        """one float in device memory, the form in which the engine takes thresholds and factors"""
        if value not in self.scalars:
            self.scalars[value] = torch.full((1,), value, device=self.device)
        return self.scalars[value]

    def call(self, name, *args):
        bound = [self.stream]
        for a in args:
            if isinstance(a, torch.Tensor):
                bound.append(ctypes.c_void_p(a.data_ptr()))
            elif isinstance(a, (ctypes.Structure, ctypes.Array)):
                self.keep.append(a)
                bound.append(ctypes.byref(a) if isinstance(a, ctypes.Structure) else a)
            elif isinstance(a, float):
                bound.append(ctypes.c_float(a))
            else:
                bound.append(a)
        self.calls.append((getattr(self.lib, name), tuple(bound)))

    def size(self, fn, desc):
        n = ctypes.c_size_t(0)
        neoml_amd.check(getattr(self.lib, fn)(ctypes.byref(desc), ctypes.byref(n)))
        return n.value

    # layers
    def conv_desc(self, x, filt, pad, stride, depthwise=False):
        n, h, w, cin = x.shape
        if depthwise:
            d = neoml_amd.ConvDesc(n, h, w, cin, cin, filt.shape[0], filt.shape[1], pad, pad, stride, stride, 1, 1, 0, 0)
            neoml_amd.check(self.lib.nhInitBlobChannelwiseConvolution(ctypes.byref(d)))
        else:
            d = neoml_amd.ConvDesc(n, h, w, cin, filt.shape[0], filt.shape[1], filt.shape[2], pad, pad, stride, stride, 1, 1, 0, 0)
            neoml_amd.check(self.lib.nhInitBlobConvolution(ctypes.byref(d)))
        return d

    def conv(self, x, p, pad, stride):
        d = self.conv_desc(x, p[0], pad, stride)
        y = self.empty(d.batch, d.resultHeight, d.resultWidth, d.filterCount)
        self.call("nhBlobConvolution", d, x, p[0], p[1], y)
        return y

    def conv_act(self, x, p, pad, stride, top):
        """a convolution and its clipped ReLU as one call, the rowwise chain that the graph optimizer makes of them"""
        d = self.conv_desc(x, p[0], pad, stride)
        y = self.empty(d.batch, d.resultHeight, d.resultWidth, d.filterCount)
        if p[0].shape[1] == 1 and pad == 0 and stride == 1:
            self.call("nhPointwiseConvolutionWithActivation", x, x.numel() // x.shape[3], x.shape[3], p[0], p[1], p[0].shape[0], 1, top, y)
        else:
            self.call("nhBlobConvolutionWithActivation", d, x, p[0], p[1], 1, top, y)
        return y

    def depthwise(self, x, p, stride):
        d = self.conv_desc(x, p[0], 1, stride, depthwise=True)
        y = self.empty(d.batch, d.resultHeight, d.resultWidth, d.channels)
        self.call("nhBlobChannelwiseConvolution", d, x, p[0], p[1], y)
        return y

    def block(self, x, expand, channelwise, down, stride, residual):
        """an inverted residual block, fused"""
        n, h, w, cin = x.shape
        e, cout = channelwise[0].shape[2], down[0].shape[0]
        d = neoml_amd.SeparableBlockDesc(n, h, w, cin if expand else 0, e, cout, stride, 1 if residual else 0, 1, 6.0, 1, 6.0)
        y = self.empty(n, (h + stride - 1) // stride, (w + stride - 1) // stride, cout)
        size = self.size("nhMobileNetV2BlockWorkspaceSize" if expand else "nhChannelwiseWith1x1WorkspaceSize", d)
        if self.work is None or self.work.numel() * FLOAT < size:
            self.work = self.empty(size // FLOAT + 1)  # the blocks run one behind the other and share it
        if expand:
            self.call("nhMobileNetV2Block", d, x, expand[0], expand[1], channelwise[0], channelwise[1], down[0], down[1], y, self.work, size)
        else:
            self.call("nhChannelwiseWith1x1", d, x, channelwise[0], channelwise[1], down[0], down[1], y, self.work, size)
        return y

    def relu(self, x, top=0.0):
        self.call("nhVectorReLU", x, x, x.numel(), self.scalar(top))
        return x

    def add(self, a, b, into=None):
        y = self.empty(*a.shape) if into is None else into
        self.call("nhVectorAdd", a, b, y, a.numel())
        return y

    def pad_pool(self, x):
        """a border of zeros, then 3x3/2 max pooling, which has no padding of its own"""
        n, h, w, c = x.shape
        padded = self.empty(n, h + 2, w + 2, c)
        self.call("nhBlobResizeImage", neoml_amd.BlobDesc.of(1, n, 1, h, w, 1, c), x, 1, 1, 1, 1, 0, 0.0,
                  neoml_amd.BlobDesc.of(1, n, 1, h + 2, w + 2, 1, c), padded)
        return self.pool(padded, 3, 3, 2, 2)

    def pool(self, x, fh, fw, sh, sw):
        n, h, w, c = x.shape
        d = neoml_amd.PoolingDesc(n, h, w, c, fh, fw, sh, sw, 0, 0)
        neoml_amd.check(self.lib.nhInitPooling(ctypes.byref(d)))
        y = self.empty(n, d.resultHeight, d.resultWidth, c)
        self.call("nhBlobMaxPooling", d, x, None, y)
        return y

    def global_mean(self, x):
        n, h, w, c = x.shape
        y = self.empty(n, c)
        self.call("nhSumMatrixRows", n, y, x, h * w, c)
        self.call("nhVectorMultiply", y, y, n * c, self.scalar(1.0 / (h * w)))
        return y

    def fc(self, x, p):
        (m, k), n = x.shape, p[0].shape[0]
        y = self.empty(m, n)
        self.call("nhMultiplyMatrixByTransposedMatrix", x, m, k, k, p[0], n, k, y, n, m * n)
        self.call("nhAddVectorToMatrixRows", 1, y, y, m, n, p[1])
        return y

    def softmax(self, x):
        y = self.empty(*x.shape)
        self.call("nhMatrixSoftmaxByRows", x, x.shape[0], x.shape[1], y)
        return y

    def transpose(self, x, b, h, m, w, c):
        """[b,h,m,w,c] -> [b,w,m,h,c]"""
        y = self.empty(b, w, m, h, c)
        self.call("nhTransposeMatrix", b, x, h, m, w, c, y, y.numel())
        return y

    def bmm(self, a, b):
        (batch, m, k), n = a.shape, b.shape[2]
        y = self.empty(batch, m, n)
        self.call("nhBatchMultiplyMatrixByMatrix", batch, a, m, k, b, n, y, y.numel())
        return y

    def scale(self, x, factor):
        self.call("nhVectorMultiply", x, x, x.numel(), self.scalar(factor))
        return x

    def gelu(self, x):
        """x * sigmoid( 1.702 x )"""
        t, n = self.empty(x.numel()), x.numel()
        self.call("nhVectorMultiply", x, t, n, self.scalar(1.702))
        self.call("nhVectorSigmoid", t, t, n)
        self.call("nhVectorEltwiseMultiply", x, t, x, n)
        return x

    def layer_norm(self, x, p):
        """the calls of the object normalization layer"""
        (rows, width), y = x.shape, self.empty(*x.shape)
        mean, dev, square = self.empty(rows), self.empty(rows), self.empty(rows, width)
        self.call("nhSumMatrixColumns", mean, x, rows, width)
        self.call("nhVectorNegMultiply", mean, mean, rows, self.scalar(1.0 / width))
        self.call("nhAddVectorToMatrixColumns", x, square, rows, width, mean)
        self.call("nhVectorEltwiseMultiply", square, square, square, rows * width)
        self.call("nhSumMatrixColumns", dev, square, rows, width)
        self.call("nhVectorMultiply", dev, dev, rows, self.scalar(1.0 / width))
        self.call("nhVectorAddValue", dev, dev, rows, self.scalar(1e-5))
        self.call("nhVectorSqrt", dev, dev, rows)
        self.call("nhVectorInv", dev, dev, rows)
        self.call("nhAddVectorToMatrixColumns", x, y, rows, width, mean)
        self.call("nhMultiplyDiagMatrixByMatrix", dev, rows, y, width, y, rows * width)
        self.call("nhBatchMultiplyMatrixByDiagMatrix", 1, y, rows, width, 0, p[0], 0, y, rows * width)
        self.call("nhAddVectorToMatrixRows", 1, y, y, rows, width, p[1])
        return y

    def lstm(self, x, p, reverse):
        (steps, batch, width), hidden = x.shape, p[2].shape[1]
        size = ctypes.c_size_t(0)
        neoml_amd.check(self.lib.nhLstmWorkspaceSize(hidden, width, steps, batch, ctypes.byref(size)))
        work, y = self.empty(size.value // FLOAT + 1), self.empty(steps, batch, hidden)
        self.call("nhLstm", hidden, width, p[0], p[1], p[2], p[3], 1 if reverse else 0, steps, batch, None, None, x, None, y, work, size.value)
        return y

    def concat(self, a, b):
        """two [rows, width] blobs side by side"""
        rows = a.shape[0]
        y = self.empty(rows, a.shape[1] + b.shape[1])
        descs = (neoml_amd.BlobDesc * 2)(*[neoml_amd.BlobDesc.of(1, rows, 1, 1, 1, 1, t.shape[1]) for t in (a, b)])
        blobs = (ctypes.c_void_p * 2)(a.data_ptr(), b.data_ptr())
        self.call("nhBlobMergeByDim", 6, descs, blobs, 2, neoml_amd.BlobDesc.of(1, rows, 1, 1, 1, 1, y.shape[1]), y)
        return y

    def log(self, x):
        self.call("nhVectorLog", x, x, x.numel())
        return x

    def argmax(self, x):
        rows, width = x.shape
        best, at = self.empty(rows), self.empty(rows, dtype=torch.int32)
        self.call("nhFindMaxValueInRows", x, rows, width, best, at, rows)
        return at

    # training
    def relu_gradient(self, y, grad):
        """the gradient in front of a ReLU, from the ReLU's output"""
        x = self.empty(*grad.shape)
        self.call("nhVectorReLUDiff", y, grad, x, grad.numel(), self.scalar(0.0))
        return x

    def conv_gradients(self, x, p, grad, pad, stride):
        """[by the input, by the filter, by the free term]"""
        d = self.conv_desc(x, p[0], pad, stride)
        by_x, by_f, by_b = self.empty(*x.shape), self.empty(*p[0].shape), self.empty(*p[1].shape)
        size = self.size("nhBlobConvolutionBackwardWorkspaceSize", d)
        self.call("nhBlobConvolutionBackward", d, grad, p[0], None, by_x, self.empty(size // FLOAT + 1), size)
        self.call("nhVectorFill", by_f, 0.0, by_f.numel())
        self.call("nhVectorFill", by_b, 0.0, by_b.numel())
        self.call("nhBlobConvolutionLearnAdd", d, x, grad, by_f)
        self.call("nhSumMatrixRowsAdd", 1, by_b, grad, grad.numel() // grad.shape[3], grad.shape[3])
        return by_x, by_f, by_b

    def momentum_step(self, parameter, grad):
        """the passes of the momentum solver over one parameter blob, with L2 regularisation"""
        history, n = torch.zeros_like(parameter), parameter.numel()
        self.keep.append(history)
        self.call("nhVectorMultiply", history, history, n, self.scalar(0.9))
        self.call("nhVectorMultiplyAndAdd", history, grad, history, n, self.scalar(-1e-6))
        self.call("nhVectorMultiplyAndAdd", history, parameter, history, n, self.scalar(-1e-9))
        self.call("nhVectorAdd", parameter, history, parameter, n)
        return history


# ---- the networks ---------------------------------------------------------------------------------------------------


def _conv_params(c, cout, f, cin):
    return c.normal(math.sqrt(2.0 / (f * f * cin)), cout, f, f, cin), c.normal(0.01, cout)


def _fc_params(c, cout, cin):
    a = math.sqrt(6.0 / (cin + cout))
    return c.uniform(-a, a, cout, cin), c.normal(0.01, cout)


def _conv(c, case):
    x = c.uniform(-1, 1, case["batch"], case["height"], case["width"], case["cin"])
    return {"y": c.relu(c.conv(x, _conv_params(c, case["cout"], 3, case["cin"]), 1, 1))}


def _resnet(c, case):
    y = c.uniform(0, 1, case["batch"], case["height"], case["width"], 3)
    y = c.pad_pool(c.relu(c.conv(y, _conv_params(c, 64, 7, 3), 3, 2)))
    cin = 64
    for stage, cout in enumerate((64, 128, 256, 512)):
        for block in range(2):
            stride = 2 if stage > 0 and block == 0 else 1
            t = c.relu(c.conv(y, _conv_params(c, cout, 3, cin), 1, stride))
            t = c.conv(t, _conv_params(c, cout, 3, cout), 1, 1)
            shortcut = y if cin == cout else c.conv(y, _conv_params(c, cout, 1, cin), 0, stride)
            y = c.relu(c.add(t, shortcut, into=t))
            cin = cout
    logits = c.fc(c.global_mean(y), _fc_params(c, 1000, cin))
    return {"features": y, "logits": logits, "probabilities": c.softmax(logits)}


MOBILENET = ((1, 16, 1, 1), (6, 24, 2, 2), (6, 32, 3, 2), (6, 64, 4, 2), (6, 96, 3, 1), (6, 160, 3, 2), (6, 320, 1, 1))


def _mobilenet(c, case):
    fused = case["fused"]
    y = c.uniform(0, 1, case["batch"], case["height"], case["width"], 3)
    p = _conv_params(c, 32, 3, 3)
    y = c.conv_act(y, p, 1, 2, 6.0) if fused else c.relu(c.conv(y, p, 1, 2), 6.0)
    cin = 32
    for t, cout, count, first_stride in MOBILENET:
        for i in range(count):
            stride, e = first_stride if i == 0 else 1, cin * t
            expand = _conv_params(c, e, 1, cin) if t != 1 else None
            channelwise = c.normal(math.sqrt(2.0 / 9), 3, 3, e), c.normal(0.01, e)
            down = _conv_params(c, cout, 1, e)
            residual = stride == 1 and cin == cout
            if fused:
                y = c.block(y, expand, channelwise, down, stride, residual)
            else:
                z = c.relu(c.conv(y, expand, 0, 1), 6.0) if expand else y
                z = c.conv(c.relu(c.depthwise(z, channelwise, stride), 6.0), down, 0, 1)
                y = c.add(z, y, into=z) if residual else z
            cin = cout
    p = _conv_params(c, 1280, 1, cin)
    y = c.conv_act(y, p, 0, 1, 6.0) if fused else c.relu(c.conv(y, p, 0, 1), 6.0)
    return {"features": y, "logits": c.fc(c.global_mean(y), _fc_params(c, 1000, 1280))}


def _encoder(c, case):
    batch, seq, d, heads = case["batch"], case["seq"], case["d"], case["heads"]
    dk = d // heads
    y = c.normal(1.0, batch * seq, d)
    for _ in range(case["layers"]):
        q, k, v = (c.fc(y, _fc_params(c, d, d)) for _ in range(3))
        q = c.transpose(q, batch, seq, 1, heads, dk).reshape(batch * heads, seq, dk)
        k = c.transpose(k, batch, seq, 1, d, 1).reshape(batch * heads, dk, seq)
        v = c.transpose(v, batch, seq, 1, heads, dk).reshape(batch * heads, seq, dk)
        scores = c.scale(c.bmm(q, k), 1.0 / math.sqrt(dk))
        weights = c.softmax(scores.reshape(batch * heads * seq, seq)).reshape(batch * heads, seq, seq)
        context = c.transpose(c.bmm(weights, v), batch, heads, 1, seq, dk).reshape(batch * seq, d)
        y = c.layer_norm(c.add(y, c.fc(context, _fc_params(c, d, d))), (c.uniform(0.8, 1.2, d), c.normal(0.05, d)))
        z = c.fc(c.gelu(c.fc(y, _fc_params(c, 4 * d, d))), _fc_params(c, d, 4 * d))
        y = c.layer_norm(c.add(y, z), (c.uniform(0.8, 1.2, d), c.normal(0.05, d)))
    return {"encoded": y}


LINES = ((64, (2, 2)), (128, (2, 2)), (256, None), (256, (2, 1)), (256, (2, 1)), (256, (2, 1)))
LINE_HEIGHT, HIDDEN, CLASSES = 32, 256, 101


def _lines(c, case):
    batch = case["batch"]
    y, cin = c.uniform(0, 1, batch, LINE_HEIGHT, case["width"], 1), 1
    for cout, window in LINES:
        y = c.relu(c.conv(y, _conv_params(c, cout, 3, cin), 1, 1))
        if window is not None:
            y = c.pool(y, window[0], window[1], window[0], window[1])
        cin = cout
    steps = y.shape[2]
    seq = c.transpose(y, 1, batch, 1, steps, cin).reshape(steps, batch, cin)
    for _ in range(2):
        a, width = 1.0 / math.sqrt(HIDDEN), seq.shape[2]
        both = []
        for reverse in (False, True):
            p = (c.uniform(-a, a, 4 * HIDDEN, width), c.uniform(-a, a, 4 * HIDDEN), c.uniform(-a, a, 4 * HIDDEN, HIDDEN), c.uniform(-a, a, 4 * HIDDEN))
            both.append(c.lstm(seq, p, reverse).reshape(steps * batch, HIDDEN))
        seq = c.concat(*both).reshape(steps, batch, 2 * HIDDEN)
    logits = c.fc(seq.reshape(steps * batch, 2 * HIDDEN), _fc_params(c, CLASSES, 2 * HIDDEN))
    logits = c.transpose(logits, 1, steps, 1, batch, CLASSES).reshape(batch * steps, CLASSES)
    logs = c.log(c.softmax(logits))
    return {"logs": logs, "labels": c.argmax(logs)}


def _train(c, case):
    batch, h, w, cin, cout, stride = (case[k] for k in ("batch", "height", "width", "cin", "cout", "stride"))
    x = c.uniform(0, 1, batch, h, w, cin)
    p1, p2 = _conv_params(c, cout, 3, cin), _conv_params(c, cout, 3, cout)
    ps = _conv_params(c, cout, 1, cin) if stride != 1 else None
    t = c.relu(c.conv(x, p1, 1, stride))
    y = c.conv(t, p2, 1, 1)
    y = c.relu(c.add(y, c.conv(x, ps, 0, stride) if ps else x, into=y))
    # the gradient that arrives from the layers behind, of the size a mean over the batch gives it
    grad = c.relu_gradient(y, c.normal(1.0 / batch, *y.shape))
    by_t, by_f2, by_b2 = c.conv_gradients(t, p2, grad, 1, 1)
    by_x, by_f1, by_b1 = c.conv_gradients(x, p1, c.relu_gradient(t, by_t), 1, stride)
    gradients = [(p1[0], by_f1), (p1[1], by_b1), (p2[0], by_f2), (p2[1], by_b2)]
    if ps:
        by_s, by_fs, by_bs = c.conv_gradients(x, ps, grad, 0, stride)
        gradients += [(ps[0], by_fs), (ps[1], by_bs)]
    else:
        by_s = grad
    out = {"y": y, "by_x": c.add(by_x, by_s, into=by_x)}
    for i, (parameter, by) in enumerate(gradients):
        out["by_p%d" % i] = by
        out["history%d" % i] = c.momentum_step(parameter, by)
        out["p%d" % i] = parameter
    return out


NETWORKS = {"conv": _conv, "resnet": _resnet, "mobilenet": _mobilenet, "encoder": _encoder, "lines": _lines, "train": _train}


def prepare(case, seed):
    c = Calls(seed)
    outputs = NETWORKS[case["kind"]](c, case)
    return {"calls": c.calls, "outputs": outputs, "keep": c.keep + list(c.scalars.values()), "lib": c.lib, "stream": c.stream}


def run(state):
    lib, stream = state["lib"], state["stream"]
    lib.nhStreamOverlapLstm(stream, 1)
    lib.nhStreamDeferSmallOps(stream, 1)
    for fn, args in state["calls"]:
        rc = fn(*args)
        if rc != 0:
            neoml_amd.check(rc)
    neoml_amd.check(lib.nhStreamDeferSmallOps(stream, 0))
    lib.nhStreamOverlapLstm(stream, 0)
    return state["outputs"]


# ---- what a pass cannot do without -----------------------------------------------------------------------------------


def _image_sizes(h, w):
    """the resolutions behind the stem and the pooling of the residual network, and of its stages"""
    half = lambda v: (v - 1) // 2 + 1  # noqa: E731
    sizes = [(half(h), half(w))]
    for _ in range(4):
        sizes.append((half(sizes[-1][0]), half(sizes[-1][1])))
    return sizes


def work(case):
    """Floating point operations: those of the products and convolutions. Bytes: the input, the weights and the outputs once;
    what passes from layer to layer could stay on the chip."""
    kind, flops, weights, values = case["kind"], 0, 0, 0

    def product(rows, n, k, count=1, own_weights=True):
        nonlocal flops, weights
        flops += 2 * rows * n * k * count
        weights += (n * k + n) * count if own_weights else 0

    b = case["batch"]
    if kind == "conv":
        pixels = b * case["height"] * case["width"]
        product(pixels, case["cout"], 9 * case["cin"])
        values = pixels * (case["cin"] + case["cout"])
    elif kind == "resnet":
        stem, *stages = _image_sizes(case["height"], case["width"])
        product(b * stem[0] * stem[1], 64, 147)
        cin = 64
        for i, ((h, w), cout) in enumerate(zip(stages, (64, 128, 256, 512))):
            product(b * h * w, cout, 9 * cin)
            product(b * h * w, cout, 9 * cout, 3)
            if i > 0:
                product(b * h * w, cout, cin)
            cin = cout
        product(b, 1000, 512)
        values = b * (case["height"] * case["width"] * 3 + h * w * 512 + 2000)
    elif kind == "mobilenet":
        half = lambda v: (v + 1) // 2  # noqa: E731
        h, w, cin = half(case["height"]), half(case["width"]), 32
        product(b * h * w, 32, 27)
        for t, cout, count, first_stride in MOBILENET:
            for i in range(count):
                e = cin * t
                if t != 1:
                    product(b * h * w, e, cin)
                if i == 0 and first_stride == 2:
                    h, w = half(h), half(w)
                product(b * h * w, e, 9)
                product(b * h * w, cout, e)
                cin = cout
        product(b * h * w, 1280, cin)
        product(b, 1000, 1280)
        values = b * (case["height"] * case["width"] * 3 + h * w * 1280 + 1000)
    elif kind == "encoder":
        seq, d, layers = case["seq"], case["d"], case["layers"]
        product(b * seq, d, d, 4 * layers)
        product(b * seq, 4 * d, d, layers)
        product(b * seq, d, 4 * d, layers)
        product(b * seq, seq, d, 2 * layers, own_weights=False)
        values = 2 * b * seq * d
    elif kind == "lines":
        h, w, cin = LINE_HEIGHT, case["width"], 1
        for cout, window in LINES:
            product(b * h * w, cout, 9 * cin)
            if window is not None:
                h, w = h // window[0], w // window[1]
            cin = cout
        for width in (256, 512):
            product(b * w, 4 * HIDDEN, width + HIDDEN, 2)
        product(b * w, CLASSES, 2 * HIDDEN)
        values = b * (LINE_HEIGHT * case["width"] + w * (CLASSES + 1))
    else:
        stride, cin, cout = case["stride"], case["cin"], case["cout"]
        outs = b * ((case["height"] - 1) // stride + 1) * ((case["width"] - 1) // stride + 1)
        product(outs, cout, 9 * cin)
        product(outs, cout, 9 * cout)
        if stride != 1:
            product(outs, cout, cin)
        flops *= 3  # forward, by the input, by the filter
        weights *= 5  # parameters and their history read and written, the gradients written
        values = 2 * b * case["height"] * case["width"] * cin + 2 * outs * cout
    return {"bytes": FLOAT * (weights + values), "flops": flops}


# Largest relative error (2-norm) seen against the same network in 64 bits, over sizes of these ranges, times four: conv
# 3e-7 (8e-7 for the sums in another order), resnet 2.2e-6 (the probabilities of a small batch; logits 3e-7), mobilenet 7e-6 (the
# features in front of the mean, which ReLU6 thins out; logits 1.7e-6), encoder 6e-7,
# lines 6e-8 (of log-probabilities, whose common part is large), train 5e-7 (the gradients by the filters).
RELATIVE = {"conv": 3e-6, "resnet": 9e-6, "mobilenet": 2.5e-5, "encoder": 2.5e-6, "lines": 3e-7, "train": 2e-6}


def tolerance(case):
    if case["kind"] == "lines":
        return {"rel": RELATIVE["lines"], "differ": 0.002}  # labels: the larger of two probabilities that are all but equal
    return {"rel": RELATIVE[case["kind"]]}
