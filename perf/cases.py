"""What a program built on this framework has it do: layers of a network, forward and backward, as the nodes of the host
layer issue them, from a single small product to a whole training step.

Everything runs through the C ABI (deep8_amd.capi) on tensors that the program owns.  A program lays its tensors and its
scratch out once and then issues the same calls every step; `prepare` does the first and lists the calls, `run` issues them.

Kinds of case
  matmul   MatrixMultiply: forward, then both gradients from one call
  dense    a fully connected layer: product + bias + ReLu in one call; ReLu gate + bias gradient; both gradients
  conv     Conv2d + bias + ReLu and its gradients; `first` is a network's first layer (no gradient of the image is wanted),
           `train` 0 is inference (the forward call alone)
  deconv   DeConv2d: forward, then both gradients from one call
  net      one training step of a small convolutional network: two convolutions with max pooling, two fully connected
           layers, L2 loss, backward, an Adam update of every parameter

Gradients are written (the overwrite forms), which is what the executor issues for the first product into a gradient.
Element types are Float32, the framework's default, and Float16; Float64 serves for checking gradients, not for work that
somebody waits for.
"""
import ctypes
import math

import torch

from deep8_amd import capi

TYPES = {"float32": (torch.float32, capi.FLOAT32, 4), "float16": (torch.float16, capi.FLOAT16, 2)}


def listed():
    return [
        # the smallest layers: a product of a few tiles, bound by its launches
        {"name": "matmul_small_f32", "kind": "matmul", "dtype": "float32", "xb": 1, "rows": 64, "inner": 128, "yb": 1, "cols": 256},
        # a batch of matrices against a batch of matrices
        {"name": "matmul_batched_f32", "kind": "matmul", "dtype": "float32", "xb": 32, "rows": 512, "inner": 512, "yb": 32, "cols": 512},
        # the largest product
        {"name": "matmul_square_f16", "kind": "matmul", "dtype": "float16", "xb": 1, "rows": 4096, "inner": 4096, "yb": 1, "cols": 4096},
        # a hidden fully connected layer at an ordinary size
        {"name": "dense_hidden_f16", "kind": "dense", "dtype": "float16", "rows": 1024, "inner": 1024, "cols": 1024},
        # a classifier's last layer: an odd number of outputs
        {"name": "dense_odd_f16", "kind": "dense", "dtype": "float16", "rows": 4096, "inner": 1024, "cols": 1001},
        # a convolution of the first stage of an image network, single precision
        {"name": "conv_3x3_f32", "kind": "conv", "dtype": "float32", "batch": 32, "height": 56, "width": 56, "in": 64, "out": 64,
         "filter": 3, "stride": 1, "dilation": 1, "covered": 1, "first": 0, "train": 1},
        # one of its third stage in half precision: small images, many channels
        {"name": "conv_deep_f16", "kind": "conv", "dtype": "float16", "batch": 32, "height": 14, "width": 14, "in": 256, "out": 256,
         "filter": 3, "stride": 1, "dilation": 1, "covered": 1, "first": 0, "train": 1},
        # its very first layer: a large filter on a three-channel image
        {"name": "conv_stem_f16", "kind": "conv", "dtype": "float16", "batch": 16, "height": 224, "width": 224, "in": 3, "out": 64,
         "filter": 7, "stride": 2, "dilation": 1, "covered": 1, "first": 1, "train": 1},
        # a layer that halves an image of odd size, with channel counts that are no powers of two
        {"name": "conv_odd_f16", "kind": "conv", "dtype": "float16", "batch": 16, "height": 57, "width": 57, "in": 96, "out": 160,
         "filter": 3, "stride": 2, "dilation": 1, "covered": 1, "first": 0, "train": 1},
        # inference on a single image
        {"name": "conv_infer_f32", "kind": "conv", "dtype": "float32", "batch": 1, "height": 28, "width": 28, "in": 128, "out": 128,
         "filter": 3, "stride": 1, "dilation": 1, "covered": 1, "first": 0, "train": 0},
        # a generator's upsampling layer
        {"name": "deconv_f16", "kind": "deconv", "dtype": "float16", "batch": 16, "height": 28, "width": 28, "in": 128, "out": 64,
         "filter": 4, "stride": 2, "covered": 0},
        # training a small network on small grey images
        {"name": "net_f32", "kind": "net", "dtype": "float32", "batch": 64, "height": 28, "width": 28, "in": 1, "c1": 32, "c2": 64,
         "hidden": 256, "classes": 10},
    ]


# ---- more cases of the same ranges ----------------------------------------------------------------------------------
MOST_WORK = {"float32": 2.6e10, "float16": 4.2e11}  # flops of a case: a few hundred microseconds to a few milliseconds
MOST_BYTES = 4e8


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi, grain):
    """a size between lo and hi: mostly multiples of `grain`, some of 8, a few anything"""
    n, r = _log(rng, lo, hi), rng.random()
    g = grain if r < 0.6 else 8 if r < 0.9 else 1
    return max(g if g <= hi else 1, n // g * g, 1)


def _draw_once(rng):
    kind = rng.choices(["matmul", "dense", "conv", "deconv", "net"], [3, 4, 7, 3, 2])[0]
    dtype = "float32" if kind == "net" or rng.random() < 0.5 else "float16"
    if kind == "matmul":
        xb = 1 if rng.random() < 0.4 else _log(rng, 2, 64)
        yb = xb if rng.random() < 0.5 else 1  # a second operand of its own for every matrix, or one that all share
        return {"kind": kind, "dtype": dtype, "xb": xb, "rows": _size(rng, 32, 4096, 64), "inner": _size(rng, 32, 4096, 64), "yb": yb,
                "cols": _size(rng, 32, 4096, 64)}
    if kind == "dense":
        return {"kind": kind, "dtype": dtype, "rows": _size(rng, 16, 8192, 64), "inner": _size(rng, 64, 4096, 64), "cols": _size(rng, 10, 4096, 64)}
    if kind == "conv":
        first = int(rng.random() < 0.2)
        size = _log(rng, 28, 224) if first else _log(rng, 7, 112)
        return {"kind": kind, "dtype": dtype, "batch": _log(rng, 1, 64), "height": size, "width": size if rng.random() < 0.7 else _log(rng, max(7, size // 2), size),
                "in": rng.choice([1, 3]) if first else _size(rng, 16, 512, 64), "out": _size(rng, 16, 512, 64),
                "filter": rng.choice([3, 5, 7]) if first else rng.choice([1, 3, 3, 3, 5]), "stride": rng.choice([1, 1, 2]),
                "dilation": 1 if rng.random() < 0.9 else 2, "covered": int(rng.random() < 0.8), "first": first, "train": int(rng.random() < 0.8)}
    if kind == "deconv":
        size = _log(rng, 4, 56)
        filt, stride = rng.choice([(4, 2), (4, 2), (3, 2), (2, 2), (5, 2), (3, 1)])
        return {"kind": kind, "dtype": dtype, "batch": _log(rng, 1, 64), "height": size, "width": size, "in": _size(rng, 16, 512, 64),
                "out": rng.choice([1, 3]) if rng.random() < 0.15 else _size(rng, 16, 512, 64), "filter": filt, "stride": stride,
                "covered": int(rng.random() < 0.2)}
    return {"kind": kind, "dtype": dtype, "batch": _log(rng, 16, 256), "height": 4 * _log(rng, 5, 16), "width": 4 * _log(rng, 5, 16),
            "in": rng.choice([1, 3]), "c1": 8 * _log(rng, 1, 8), "c2": 8 * _log(rng, 2, 16), "hidden": _size(rng, 64, 512, 64),
            "classes": rng.choice([2, 10, 10, 47, 100])}


def draw(rng):
    while True:
        case = _draw_once(rng)
        if case["kind"] in ("conv", "deconv"):
            reach = (case["filter"] - 1) * case.get("dilation", 1) + 1
            if min(case["height"], case["width"]) < reach:
                continue
        w = work(case)
        if w["flops"] <= MOST_WORK[case["dtype"]] and w["bytes"] <= MOST_BYTES:
            return case


# ---- sizes ----------------------------------------------------------------------------------------------------------
def _conv_size(case):
    n = []
    for size in (case["height"], case["width"]):
        reach = (case["filter"] - 1) * case["dilation"] + 1
        n.append((size - 1) // case["stride"] + 1 if case["covered"] else (size - reach) // case["stride"] + 1)
    return n


def _deconv_size(case):
    add = 1 if case["covered"] else case["filter"]
    return [(size - 1) * case["stride"] + add for size in (case["height"], case["width"])]


def _net_layers(case):
    """rows, inner, cols of the four products of the network's forward pass"""
    B, H, W = case["batch"], case["height"], case["width"]
    return [(B * H * W, 25 * case["in"], case["c1"]), (B * H * W // 4, 25 * case["c1"], case["c2"]),
            (B, H * W // 16 * case["c2"], case["hidden"]), (B, case["hidden"], case["classes"])]


def work(case):
    kind, es = case["kind"], TYPES[case["dtype"]][2]
    if kind == "matmul":
        zb = max(case["xb"], case["yb"])
        nx, ny = case["xb"] * case["rows"] * case["inner"], case["yb"] * case["inner"] * case["cols"]
        nz = zb * case["rows"] * case["cols"]
        return {"bytes": es * (2 * nx + 2 * ny + 2 * nz), "flops": 6.0 * zb * case["rows"] * case["inner"] * case["cols"]}
    if kind == "dense":
        nx, ny, nz = case["rows"] * case["inner"], case["inner"] * case["cols"], case["rows"] * case["cols"]
        return {"bytes": es * (2 * nx + 2 * ny + 2 * nz + 2 * case["cols"]), "flops": 6.0 * case["rows"] * case["inner"] * case["cols"]}
    if kind == "conv":
        OH, OW = _conv_size(case)
        nx, nz = case["batch"] * case["height"] * case["width"] * case["in"], case["batch"] * OH * OW * case["out"]
        nw = case["out"] * case["filter"] ** 2 * case["in"]
        one = 2.0 * case["batch"] * OH * OW * case["filter"] ** 2 * case["in"] * case["out"]
        if not case["train"]:
            return {"bytes": es * (nx + nw + case["out"] + nz), "flops": one}
        if case["first"]:
            return {"bytes": es * (nx + 2 * nw + 2 * nz + 2 * case["out"]), "flops": 2 * one}
        return {"bytes": es * (2 * nx + 2 * nw + 2 * nz + 2 * case["out"]), "flops": 3 * one}
    if kind == "deconv":
        OH, OW = _deconv_size(case)
        nx, nz = case["batch"] * case["height"] * case["width"] * case["in"], case["batch"] * OH * OW * case["out"]
        nw = case["out"] * case["filter"] ** 2 * case["in"]
        return {"bytes": es * (2 * nx + 2 * nw + 2 * nz),
                "flops": 6.0 * case["batch"] * case["height"] * case["width"] * case["in"] * case["filter"] ** 2 * case["out"]}
    layers = _net_layers(case)
    flops = sum(6.0 * m * k * n for m, k, n in layers) - 2.0 * layers[0][0] * layers[0][1] * layers[0][2]
    nx = case["batch"] * case["height"] * case["width"] * case["in"]
    params = sum(k * n + n for _, k, n in layers)
    # the image and the targets; the activations that the backward pass needs again are written and read once each; a
    # parameter and its two moments are read and written, its gradient is written
    acts = sum(m * n for m, _, n in layers)
    return {"bytes": es * (nx + layers[3][0] * layers[3][2] + 2 * acts + 7 * params), "flops": flops}


# Relative errors (2-norm) against the same calls in 64-bit arithmetic: Float32 layers 0.9e-7 to 5.3e-7, and 1.2e-6 for the
# longest chain of additions (a reduction of 4096 that is not cut); Float16 layers 2.1e-4 to 3.1e-4, which is the rounding of
# the result, whatever the sizes.  Four times the largest is stated.  In the network a sum that rounds differently can also
# move a maximum to its neighbour or open a gate: one such element among the tens of thousands of a layer is what the wider
# bound admits.
TOLERANCE = {"float32": 5e-6, "float16": 1.2e-3, "net": 2e-3}


def tolerance(case):
    return {"rel": TOLERANCE["net" if case["kind"] == "net" else case["dtype"]]}


# ---- tensors and calls ----------------------------------------------------------------------------------------------
class _Program:
    """tensors of one program and the calls it issues every step"""

    def __init__(self, dtype, seed):
        self.lib = capi.init()
        self.torch_type, self.dt, _ = TYPES[dtype]
        self.rng = torch.Generator(device="cuda").manual_seed(seed)
        self.calls, self.out, self.keep = [], {}, []
        self.scratch_need, self.scratch_users = 16, []
        self.steps = ctypes.c_long(0)

    def normal(self, *shape, scale=1.0):
        return (torch.randn(shape, generator=self.rng, device="cuda") * scale).to(self.torch_type)

    def activations(self, *shape):
        """what the layer before leaves: half of it cut to zero by its ReLu"""
        return torch.relu(torch.randn(shape, generator=self.rng, device="cuda")).to(self.torch_type)

    def empty(self, *shape):
        return torch.empty(shape, dtype=self.torch_type, device="cuda")

    def zeros(self, *shape):
        return torch.zeros(shape, dtype=self.torch_type, device="cuda")

    def call(self, name, *args):
        """the next call of a step: tensors as arguments stand for their addresses, the element type and the (default)
        stream are added"""
        self.keep.append(args)
        self.calls.append((getattr(self.lib, name), [a.data_ptr() if isinstance(a, torch.Tensor) else a for a in (self.dt,) + args + (None,)]))

    def call_with_scratch(self, need, name, *args):
        """... of an entry point whose last arguments are a scratch block and its size; the calls of a step run one after
        the other and share one block"""
        self.scratch_need = max(self.scratch_need, need)
        self.scratch_users.append(len(self.calls))
        self.call(name, *args, None, need)

    def finish(self):
        self.scratch = torch.empty(self.scratch_need, dtype=torch.uint8, device="cuda")
        for i in self.scratch_users:
            self.calls[i][1][-3] = self.scratch.data_ptr()
        self.calls = [(fn, tuple(args)) for fn, args in self.calls]
        return self


def _dims(*shape):
    """Deep8's enlarged form [batch, d0 .. d3], dimensions right-aligned"""
    return (ctypes.c_int * 5)(*((shape[0],) + (1,) * (5 - len(shape)) + tuple(shape[1:])))


def _column_sum(p, grad, src, rows, cols):
    """grad[cols] = column sums of src[rows][cols]: the gradient of a bias"""
    gd, zd = _dims(1, 1, cols), _dims(1, rows, cols)
    p.call_with_scratch(p.lib.d8_add_grad_scratch_bytes(p.dt, gd, zd), "d8_add_grad_overwrite", grad, gd, src, zd)


def _relu_gate(p, z, dz, dpre, dbias, rows, cols):
    p.call_with_scratch(p.lib.d8_bias_relu_grad_scratch_bytes(p.dt, rows, cols), "d8_bias_relu_grad", z, dz, dpre, dbias, rows, cols, 0)


def _dense_forward(p, x, w, b, relu, z, rows, inner, cols):
    need = p.lib.d8_matmul_scratch_bytes(p.dt, 0, 1, rows, inner, 1, inner, cols)
    p.call_with_scratch(need, "d8_matmul_bias_relu", x, 1, rows, inner, w, 1, inner, cols, b, relu, z)


def _dense_gradients(p, x, gx, w, gw, dz, rows, inner, cols):
    need = p.lib.d8_matmul_scratch_bytes(p.dt, 3, 1, rows, inner, 1, inner, cols)
    p.call_with_scratch(need, "d8_matmul_grad_xy", x, gx, 1, rows, inner, w, gw, 1, inner, cols, dz, 3)


def _conv_forward(p, x, w, b, z, image, filt, geo):
    need = p.lib.d8_conv2d_scratch_bytes(p.dt, 0, *image, *filt, *geo)
    p.call_with_scratch(need, "d8_conv2d_bias_relu", x, *image, w, *filt, b, 1, z, *geo)


def _conv_gradients(p, x, gx, w, gw, dz, image, filt, geo):
    if gx is None:
        need = p.lib.d8_conv2d_scratch_bytes(p.dt, 2, *image, *filt, *geo)
        p.call_with_scratch(need, "d8_conv2d_grad_y_overwrite", x, *image, gw, *filt, dz, *geo)
    else:
        need = p.lib.d8_conv2d_scratch_bytes(p.dt, 3, *image, *filt, *geo)
        p.call_with_scratch(need, "d8_conv2d_grad_xy", x, gx, *image, w, gw, *filt, dz, *geo, 3)


def _prepare_matmul(p, case):
    xb, yb, rows, inner, cols = case["xb"], case["yb"], case["rows"], case["inner"], case["cols"]
    zb = max(xb, yb)
    x, y = p.normal(xb, rows, inner), p.normal(yb, inner, cols, scale=inner ** -0.5)
    dz = p.normal(zb, rows, cols)
    z, gx, gy = p.empty(zb, rows, cols), p.empty(xb, rows, inner), p.empty(yb, inner, cols)
    shape = (xb, rows, inner), (yb, inner, cols)
    p.call_with_scratch(p.lib.d8_matmul_scratch_bytes(p.dt, 0, *shape[0], *shape[1]), "d8_matmul", x, *shape[0], y, *shape[1], z)
    p.call_with_scratch(p.lib.d8_matmul_scratch_bytes(p.dt, 3, *shape[0], *shape[1]), "d8_matmul_grad_xy", x, gx, *shape[0], y, gy,
                        *shape[1], dz, 3)
    p.out = {"z": z, "gx": gx, "gy": gy}


def _prepare_dense(p, case):
    rows, inner, cols = case["rows"], case["inner"], case["cols"]
    x, w, b = p.activations(rows, inner), p.normal(inner, cols, scale=(2.0 / inner) ** 0.5), p.normal(cols, scale=0.1)
    dz = p.normal(rows, cols)
    z, dpre, gb, gx, gw = p.empty(rows, cols), p.empty(rows, cols), p.empty(cols), p.empty(rows, inner), p.empty(inner, cols)
    _dense_forward(p, x, w, b, 1, z, rows, inner, cols)
    _relu_gate(p, z, dz, dpre, gb, rows, cols)
    _dense_gradients(p, x, gx, w, gw, dpre, rows, inner, cols)
    p.out = {"z": z, "gb": gb, "gx": gx, "gw": gw}


def _prepare_conv(p, case):
    image = case["batch"], case["height"], case["width"], case["in"]
    filt = case["out"], case["filter"], case["filter"]
    geo = case["covered"], case["stride"], case["stride"], case["dilation"], case["dilation"]
    OH, OW = _conv_size(case)
    fan = filt[1] * filt[2] * image[3]
    x = p.normal(*image) if case["first"] else p.activations(*image)
    w, b = p.normal(*filt, image[3], scale=(2.0 / fan) ** 0.5), p.normal(filt[0], scale=0.1)
    z = p.empty(image[0], OH, OW, filt[0])
    _conv_forward(p, x, w, b, z, image, filt, geo)
    p.out = {"z": z}
    if case["train"]:
        dz, dpre, gb = p.normal(*z.shape), p.empty(*z.shape), p.empty(filt[0])
        gx, gw = None if case["first"] else p.empty(*image), p.empty(*w.shape)
        _relu_gate(p, z, dz, dpre, gb, image[0] * OH * OW, filt[0])
        _conv_gradients(p, x, gx, w, gw, dpre, image, filt, geo)
        p.out.update(gb=gb, gw=gw, **({} if gx is None else {"gx": gx}))


def _prepare_deconv(p, case):
    image = case["batch"], case["height"], case["width"], case["in"]
    filt = case["out"], case["filter"], case["filter"]
    geo = case["covered"], case["stride"], case["stride"]
    OH, OW = _deconv_size(case)
    x = p.activations(*image)
    w = p.normal(*filt, image[3], scale=(2.0 * case["stride"] ** 2 / (filt[1] * filt[2] * image[3])) ** 0.5)
    dz, z = p.normal(image[0], OH, OW, filt[0]), p.empty(image[0], OH, OW, filt[0])
    gx, gw = p.empty(*image), p.empty(*w.shape)
    p.call_with_scratch(p.lib.d8_deconv2d_scratch_bytes(p.dt, 0, *image, *filt, *geo), "d8_deconv2d", x, *image, w, *filt, z, *geo)
    p.call_with_scratch(p.lib.d8_deconv2d_scratch_bytes(p.dt, 3, *image, *filt, *geo), "d8_deconv2d_grad_xy", x, gx, *image, w, gw, *filt,
                        dz, *geo, 3)
    p.out = {"z": z, "gx": gx, "gw": gw}


def _prepare_net(p, case):
    B, H, W, C = case["batch"], case["height"], case["width"], case["in"]
    c1, c2, hidden, classes = case["c1"], case["c2"], case["hidden"], case["classes"]
    H2, W2, H4, W4 = H // 2, W // 2, H // 4, W // 4
    flat, geo, pool = H4 * W4 * c2, (1, 1, 1, 1, 1), (2, 2, 0, 2, 2)
    x, target = p.normal(B, H, W, C), p.normal(B, classes)
    shapes = [(c1, 5, 5, C), (c2, 5, 5, c1), (flat, hidden), (hidden, classes)]
    fans = [25 * C, 25 * c1, flat, hidden]
    w = [p.normal(*s, scale=(2.0 / f) ** 0.5) for s, f in zip(shapes, fans)]
    b = [p.zeros(n) for n in (c1, c2, hidden, classes)]
    gw, gb = [p.empty(*t.shape) for t in w], [p.empty(*t.shape) for t in b]
    a1, p1, a2, p2 = p.empty(B, H, W, c1), p.empty(B, H2, W2, c1), p.empty(B, H2, W2, c2), p.empty(B, H4, W4, c2)
    h, y, e = p.empty(B, hidden), p.empty(B, classes), p.empty(B, classes)
    norm, loss, dloss = p.empty(B), p.empty(1), torch.ones(1, dtype=p.torch_type, device="cuda")
    # forward
    _conv_forward(p, x, w[0], b[0], a1, (B, H, W, C), (c1, 5, 5), geo)
    p.call("d8_maxpool2d", a1, p1, B, H, W, c1, *pool)
    _conv_forward(p, p1, w[1], b[1], a2, (B, H2, W2, c1), (c2, 5, 5), geo)
    p.call("d8_maxpool2d", a2, p2, B, H2, W2, c2, *pool)
    _dense_forward(p, p2, w[2], b[2], 1, h, B, flat, hidden)
    _dense_forward(p, h, w[3], b[3], 0, y, B, hidden, classes)
    rows, ed, one = _dims(B, 1), _dims(B, classes), _dims(1, 1)
    p.call("d8_minus", y, ed, target, ed, e, ed)
    p.call_with_scratch(p.lib.d8_add_grad_scratch_bytes(p.dt, rows, ed), "d8_l2norm", e, norm, B, classes)
    p.call_with_scratch(p.lib.d8_add_grad_scratch_bytes(p.dt, one, rows), "d8_reduce_mean", norm, rows, loss, one)
    # backward: the loss
    dnorm, dy = p.empty(B), p.empty(B, classes)
    p.call("d8_fill", dnorm, B, 0.0)
    p.call("d8_reduce_mean_grad", dnorm, rows, dloss, one)
    p.call("d8_fill", dy, B * classes, 0.0)
    p.call("d8_l2norm_grad", e, dy, norm, dnorm, B, classes)
    # the fully connected layers
    dh, dhp, dp2 = p.empty(B, hidden), p.empty(B, hidden), p.empty(B, H4, W4, c2)
    _column_sum(p, gb[3], dy, B, classes)
    _dense_gradients(p, h, dh, w[3], gw[3], dy, B, hidden, classes)
    _relu_gate(p, h, dh, dhp, gb[2], B, hidden)
    _dense_gradients(p, p2, dp2, w[2], gw[2], dhp, B, flat, hidden)
    # the convolutions
    da2, da2p, dp1 = p.empty(*a2.shape), p.empty(*a2.shape), p.empty(*p1.shape)
    p.call("d8_maxpool2d_grad_overwrite", a2, da2, dp2, B, H2, W2, c2, *pool)
    _relu_gate(p, a2, da2, da2p, gb[1], B * H2 * W2, c2)
    _conv_gradients(p, p1, dp1, w[1], gw[1], da2p, (B, H2, W2, c1), (c2, 5, 5), geo)
    da1, da1p = p.empty(*a1.shape), p.empty(*a1.shape)
    p.call("d8_maxpool2d_grad_overwrite", a1, da1, dp1, B, H, W, c1, *pool)
    _relu_gate(p, a1, da1, da1p, gb[0], B * H * W, c1)
    _conv_gradients(p, x, None, w[0], gw[0], da1p, (B, H, W, C), (c1, 5, 5), geo)
    # the update
    for value, grad in zip(w + b, gw + gb):
        m, v = p.zeros(*value.shape), p.zeros(*value.shape)
        p.call("d8_adam_update", value, grad, m, v, 0.9, 0.999, 1e-7, 1e-4, 0.0, p.steps, value.numel())
    p.out = {"loss": loss, "y": y, "gw": gw, "gb": gb, "w": w, "b": b}


def prepare(case, seed):
    p = _Program(case["dtype"], seed)
    {"matmul": _prepare_matmul, "dense": _prepare_dense, "conv": _prepare_conv, "deconv": _prepare_deconv, "net": _prepare_net}[case["kind"]](p, case)
    return p.finish()


def run(state):
    state.steps.value += 1
    for fn, args in state.calls:
        rc = fn(*args)
        if rc:
            capi.check(rc)
    return state.out
