"""Performance cases of the library: the calls its users make, each as one repeatable pass through the public entry points.

Every case is a training step (or, for `infer`, an inference pass) of something the repository is used for: matrix
products, a dense layer, a convolution layer, a residual block, and the networks of the benchmark configurations. All
tensors are fp32, NCHW, in device memory, as the C ABI takes them; torch supplies memory and the random inputs only.

`listed()` gives the cases, `draw()` another of the same ranges, `prepare()` what a program holds before the call,
`run()` one pass, `work()` the bytes and operations it cannot do without, `tolerance()` how far another correct fp32
implementation may be off.
"""
import math

import torch

from crusaderbackend_amd import capi
from crusaderbackend_amd.vgg16_step import Vgg16Step

# (input channels, image, output channels, stride, layers): the 3x3 convolutions of ResNet-56 on CIFAR images
RESNET56 = ((16, 32, 16, 1, 19), (32, 16, 32, 1, 17), (64, 8, 64, 1, 18), (16, 32, 32, 2, 1), (32, 16, 64, 2, 1))
# (image, first input width): the three stages of DenseNet-BC-100, k = 12: 16 x (1x1 IC->48, 3x3 48->12) each
DENSENET = ((32, 24), (16, 108), (8, 150))
# VGG-16 (CIFAR variant): (input channels, image, output channels); None is a 2x2 max pooling
VGG16 = ((3, 32, 64), (64, 32, 64), None, (64, 16, 128), (128, 16, 128), None, (128, 8, 256), (256, 8, 256), (256, 8, 256), None,
         (256, 4, 512), (512, 4, 512), (512, 4, 512), None, (512, 2, 512), (512, 2, 512), (512, 2, 512), None)


def listed():
    return [
        # the classifier at the end of the CIFAR networks: three launches of a few microseconds, all latency
        {"name": "dense_512x10_b128", "kind": "dense", "batch": 128, "IN": 512, "OUT": 10},
        # wide fully connected layer at a training batch: forward, data gradient and weight gradient (NT, NN, TN products)
        {"name": "dense_4096_b256", "kind": "dense", "batch": 256, "IN": 4096, "OUT": 4096},
        # plain products: the small square one, the large one, and one no tile size divides and no 16-byte load fits
        {"name": "gemm_nn_1024", "kind": "gemm", "form": "nn", "M": 1024, "N": 1024, "K": 1024},
        {"name": "gemm_nn_4096", "kind": "gemm", "form": "nn", "M": 4096, "N": 4096, "K": 4096},
        {"name": "gemm_tn_ragged", "kind": "gemm", "form": "tn", "M": 1003, "N": 1505, "K": 777},
        # the benchmark's headline step: every 3x3 convolution of ResNet-56, both directions, weight gradients summed once
        {"name": "resnet56_conv_step_b128", "kind": "resnet", "batch": 128},
        # whole training step of VGG-16: convolutions, ReLU, pooling, dense head, loss and momentum update
        {"name": "vgg16_train_step_b128", "kind": "vgg", "batch": 128},
        # classifying one image: dataset bytes -> normalised input -> VGG-16 forward -> probabilities
        {"name": "vgg16_infer_b1", "kind": "infer", "batch": 1},
        # DenseNet-BC-100 convolutions as the reference's operands issue them: three calls per layer
        {"name": "densenet_conv_step_b64", "kind": "densenet", "batch": 64},
        # residual blocks on ImageNet-sized feature maps (two 3x3 convolutions, two normalisations, identity shortcut),
        # forward and backward: the widest image and a deep, narrow one
        {"name": "block_64_56_b32", "kind": "block", "batch": 32, "C": 64, "H": 56},
        {"name": "block_256_14_b32", "kind": "block", "batch": 32, "C": 256, "H": 14},
        # a convolution layer off every grid: odd channels, non-square odd image, 5x5 filter, stride 2
        {"name": "conv_5x5s2_ragged", "kind": "conv", "batch": 24, "IC": 30, "H": 61, "W": 47, "OC": 75, "F": 5, "s": 2, "p": 2},
    ]


def draw(rng):
    def log(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    kind = rng.choice(("dense", "dense", "gemm", "gemm", "gemm", "conv", "conv", "conv", "block", "block", "resnet", "vgg", "infer",
                       "densenet"))
    if kind == "dense":
        # half of the widths are multiples of 64, as layers usually are; the others are whatever comes
        r = 64 if rng.random() < 0.5 else 1
        return {"kind": kind, "batch": log(16, 512), "IN": max(64, log(64, 4096) // r * r), "OUT": max(10, log(10, 4096) // r * r)}
    if kind == "gemm":
        r = 64 if rng.random() < 0.5 else 1
        return {"kind": kind, "form": rng.choice(("nn", "nt", "tn")), "M": max(64, log(64, 4096) // r * r),
                "N": max(64, log(64, 4096) // r * r), "K": max(64, log(64, 4096) // r * r)}
    if kind == "conv":
        F = rng.choice((1, 3, 3, 3, 5))
        s = rng.choice((1, 1, 2))
        H = log(7, 64)
        c = {"kind": kind, "batch": log(4, 64), "IC": log(8, 256), "H": H, "W": max(7, H + rng.randint(-5, 5)), "OC": log(8, 256),
             "F": F, "s": s, "p": F // 2}
        while c["batch"] > 1 and 2.0 * c["batch"] * c["OC"] * (c["H"] // s) * (c["W"] // s) * c["IC"] * F * F > 8e9:
            c["batch"] = c["batch"] // 2
        return c
    if kind == "block":
        H = rng.choice((56, 48, 40, 28, 24, 20, 14, 12, 7, rng.randint(7, 56)))
        C = max(16, min(512, int(3600 / H) // 16 * 16))
        return {"kind": kind, "batch": log(4, 32), "C": rng.choice((C, C // 2 if C >= 32 else C)), "H": H}
    if kind == "infer":
        return {"kind": kind, "batch": log(1, 64)}
    return {"kind": kind, "batch": log(8, 64 if kind == "densenet" else 128)}


# ---- inputs ----------------------------------------------------------------------------------------------------------
class Source:
    """Random tensors on the GPU from one seed: activations and gradients N(0,1), filters He-normal, products U[-1,1]."""

    def __init__(self, seed):
        self.dev = torch.device("cuda:0")
        self.gen = torch.Generator(device=self.dev).manual_seed(seed)

    def normal(self, *shape, std=1.0):
        t = torch.randn(*shape, generator=self.gen, device=self.dev)
        return t if std == 1.0 else t.mul_(std)

    def uniform(self, *shape):
        return torch.rand(*shape, generator=self.gen, device=self.dev).mul_(2).sub_(1)

    def empty(self, *shape):
        return torch.empty(*shape, dtype=torch.float32, device=self.dev)

    def zeros(self, *shape):
        return torch.zeros(*shape, dtype=torch.float32, device=self.dev)

    def scratch(self, nbytes):
        return self.empty(nbytes // 4) if nbytes else None


def _gemm_shapes(c):
    M, N, K = c["M"], c["N"], c["K"]
    return {"nn": ((M, K), (K, N)), "nt": ((M, K), (N, K)), "tn": ((K, M), (K, N))}[c["form"]]


def _resnet_layers(batch):
    return [(capi.ConvGeom.make(batch, IC, H, H, OC, 3, 3, s, s, 1, 1), n) for IC, H, OC, s, n in RESNET56]


def _densenet_layers(batch):
    """Per stage: (1x1 geometries, the 3x3 geometry they share)."""
    return [([capi.ConvGeom.make(batch, base + 12 * i, H, H, 48, 1, 1) for i in range(16)], capi.ConvGeom.make(batch, 48, H, H, 12, 3, 3, 1, 1, 1, 1))
            for H, base in DENSENET]


def _geom(c):
    return capi.ConvGeom.make(c["batch"], c["IC"], c["H"], c["W"], c["OC"], c["F"], c["F"], c["s"], c["s"], c["p"], c["p"])


def prepare(case, seed):
    return {"dense": _prepare_dense, "gemm": _prepare_gemm, "conv": _prepare_conv, "block": _prepare_block, "resnet": _prepare_resnet,
            "densenet": _prepare_densenet, "vgg": _prepare_vgg, "infer": _prepare_infer}[case["kind"]](case, Source(seed), seed)


def run(state):
    return state["pass"](state)


# ---- matrix products -------------------------------------------------------------------------------------------------
def _prepare_gemm(c, src, seed):
    a, b = _gemm_shapes(c)
    return {"pass": _run_gemm, "case": c, "A": src.uniform(*a), "B": src.uniform(*b), "C": src.empty(c["M"], c["N"])}


def _run_gemm(s):
    c = s["case"]
    getattr(capi, "sgemm_" + c["form"])(s["A"], s["B"], s["C"], c["M"], c["N"], c["K"])
    return s["C"]


# ---- dense layer: forward, data gradient, weight and bias gradient ------------------------------------------------------
def _prepare_dense(c, src, seed):
    n, i, o = c["batch"], c["IN"], c["OUT"]
    return {"pass": _run_dense, "case": c, "X": src.normal(n, i), "W": src.normal(o, i, std=math.sqrt(2.0 / i)), "b": src.normal(o, std=math.sqrt(2.0 / i)),
            "dY": src.normal(n, o), "Y": src.empty(n, o), "dX": src.empty(n, i), "dW": src.zeros(o, i), "dB": src.zeros(o)}


def _run_dense(s):
    n, i, o = s["case"]["batch"], s["case"]["IN"], s["case"]["OUT"]
    capi.linear_fwd(s["X"], s["W"], s["b"], s["Y"], n, i, o)
    capi.linear_dgrad(s["dY"], s["W"], s["dX"], n, i, o)
    capi.linear_wgrad(s["dY"], s["X"], s["dW"], s["dB"], n, i, o)
    return s["Y"], s["dX"], s["dW"], s["dB"]


# ---- one convolution layer: forward with bias, then both gradients in one call -----------------------------------------
def _prepare_conv(c, src, seed):
    g = _geom(c)
    fan = g.IC * g.FH * g.FW
    return {"pass": _run_conv, "g": g, "X": src.normal(g.N, g.IC, g.IH, g.IW), "W": src.normal(g.OC, g.IC, g.FH, g.FW, std=math.sqrt(2.0 / fan)),
            "b": src.normal(g.OC), "dY": src.normal(g.N, g.OC, g.OH, g.OW), "Y": src.empty(g.N, g.OC, g.OH, g.OW), "dX": src.empty(g.N, g.IC, g.IH, g.IW),
            "dW": src.zeros(g.OC, g.IC, g.FH, g.FW), "ws": src.scratch(capi.conv_wgrad_workspace_bytes(g))}


def _run_conv(s):
    capi.conv_fwd(s["W"], s["X"], s["Y"], s["b"], s["g"])
    capi.conv_bwd(s["W"], s["dY"], s["X"], s["dX"], s["dW"], s["g"], workspace=s["ws"])
    return s["Y"], s["dX"], s["dW"]


# ---- residual block: conv, norm + ReLU, conv, norm + shortcut + ReLU, and back ------------------------------------------
# Forward of one micro-batch, then backward of the one before it, whose activations are in hand: the usual order when
# gradients are accumulated over several. (It also keeps a rounding difference at a ReLU's zero out of the gradients, where
# one flipped mask is a difference as large as a value.)
def _prepare_block(c, src, seed):
    n, C, H = c["batch"], c["C"], c["H"]
    g = capi.ConvGeom.make(n, C, H, H, C, 3, 3, 1, 1, 1, 1)
    F = C * H * H
    s = {"pass": _run_block, "g": g, "F": F, "ws": src.scratch(capi.conv_wgrad_workspace_bytes(g))}
    for k in ("X", "savedX", "savedZ1", "savedZ2", "dOut"):
        s[k] = src.normal(n, C, H, H)
    for k in ("savedA1", "savedOut"):
        s[k] = src.normal(n, C, H, H).clamp_(min=0)
    for k in ("Z1", "A1", "Z2", "Out", "dZ2", "dShort", "dA1", "dZ1", "dX"):
        s[k] = src.empty(n, C, H, H)
    for k in ("1", "2"):
        s["W" + k], s["dW" + k] = src.normal(C, C, 3, 3, std=math.sqrt(2.0 / (C * 9))), src.zeros(C, C, 3, 3)
        s["gamma" + k], s["beta" + k] = src.normal(F, std=0.1).add_(1), src.normal(F, std=0.1)
        for v in ("mean", "var", "dGamma", "dBeta"):
            s[v + k] = src.empty(F)
    return s


def _run_block(s):
    g, F, N = s["g"], s["F"], s["g"].N
    capi.conv_fwd(s["W1"], s["X"], s["Z1"], None, g)
    capi.batchnorm_relu_fwd(s["Z1"], s["beta1"], s["gamma1"], s["mean1"], s["var1"], s["A1"], N, F)
    capi.conv_fwd(s["W2"], s["A1"], s["Z2"], None, g)
    capi.batchnorm_relu_fwd(s["Z2"], s["beta2"], s["gamma2"], s["mean2"], s["var2"], s["Out"], N, F, addend=s["X"])
    capi.batchnorm_relu_bwd(s["dOut"], s["savedOut"], s["gamma2"], s["savedZ2"], s["dZ2"], N, F, dGamma=s["dGamma2"], dBeta=s["dBeta2"],
                            dYmasked=s["dShort"])
    capi.conv_bwd(s["W2"], s["dZ2"], s["savedA1"], s["dA1"], s["dW2"], g, workspace=s["ws"])
    capi.batchnorm_relu_bwd(s["dA1"], s["savedA1"], s["gamma1"], s["savedZ1"], s["dZ1"], N, F, dGamma=s["dGamma1"], dBeta=s["dBeta1"])
    capi.conv_bwd(s["W1"], s["dZ1"], s["savedX"], s["dX"], s["dW1"], g, workspace=s["ws"])
    capi.tensor_add_inplace(s["dX"], s["dShort"], s["dX"].numel())
    return [s[k] for k in ("Z1", "Z2", "Out", "dX", "dW1", "dW2", "dGamma1", "dBeta1", "dGamma2", "dBeta2")]


# ---- ResNet-56: one forward and one backward call per layer, all weight gradients completed by one launch ----------------
def _prepare_resnet(c, src, seed):
    groups, sums = [], []
    for g, n in _resnet_layers(c["batch"]):
        d = {"g": g, "n": n, "X": src.normal(n, g.N, g.IC, g.IH, g.IW), "W": src.normal(n, g.OC, g.IC, 3, 3, std=math.sqrt(2.0 / (g.IC * 9))),
             "dY": src.normal(n, g.N, g.OC, g.OH, g.OW), "Y": src.empty(n, g.N, g.OC, g.OH, g.OW), "dX": src.empty(n, g.N, g.IC, g.IH, g.IW),
             "dW": src.zeros(n, g.OC, g.IC, 3, 3)}
        slices, nbytes = capi.conv_bwd_slices(g), capi.conv_wgrad_workspace_bytes(g)
        d["ws"] = [src.scratch(nbytes) for _ in range(n)]
        d["sliced"] = slices > 0
        # what a program keeps per layer: the tensors of that layer
        d["layers"] = [tuple(d[k][i] for k in ("W", "X", "Y", "dY", "dX", "dW")) + (d["ws"][i],) for i in range(n)]
        if slices:
            sums += [(d["ws"][i], d["dW"][i], slices) for i in range(n)]
        groups.append(d)
    return {"pass": _run_resnet, "groups": groups, "table": capi.slice_sum_table(sums) if sums else None}


def _run_resnet(s):
    for d in s["groups"]:
        for W, X, Y, dY, dX, dW, ws in d["layers"]:
            capi.conv_fwd(W, X, Y, None, d["g"])
    for d in reversed(s["groups"]):
        for W, X, Y, dY, dX, dW, ws in d["layers"]:
            if d["sliced"]:
                capi.conv_bwd_sliced(W, dY, X, dX, d["g"], ws)
            else:
                capi.conv_bwd(W, dY, X, dX, dW, d["g"], workspace=ws)
    if s["table"] is not None:
        capi.sum_slices_multi(s["table"])
    return [[d[k] for k in ("Y", "dX", "dW")] for d in s["groups"]]


# ---- DenseNet-BC-100: forward, data gradient and weight gradient as three calls per layer --------------------------------
def _prepare_densenet(c, src, seed):
    stages = []
    for ones, g3 in _densenet_layers(c["batch"]):
        n, H = g3.N, g3.IH
        x_sizes, w_sizes = [n * g.IC * H * H for g in ones], [48 * g.IC for g in ones]
        X1, dX1, W1, dW1 = src.normal(sum(x_sizes)), src.empty(sum(x_sizes)), src.normal(sum(w_sizes)), src.zeros(sum(w_sizes))
        st = {"Y1": src.empty(16, n, 48, H, H), "dY1": src.normal(16, n, 48, H, H), "dX1": dX1, "dW1": dW1,
              "X3": src.normal(16, n, 48, H, H), "W3": src.normal(16, 12, 48, 3, 3, std=math.sqrt(2.0 / 432)), "Y3": src.empty(16, n, 12, H, H),
              "dY3": src.normal(16, n, 12, H, H), "dX3": src.empty(16, n, 48, H, H), "dW3": src.zeros(16, 12, 48, 3, 3), "layers": []}
        ws3 = src.scratch(capi.conv_wgrad_workspace_bytes(g3))
        parts = [t.split(sizes) for t, sizes in ((X1, x_sizes), (dX1, x_sizes), (W1, w_sizes), (dW1, w_sizes))]
        for i, g in enumerate(ones):
            x, dx, w, dw = (p[i] for p in parts)
            w.mul_(math.sqrt(2.0 / g.IC))
            st["layers"].append((g, w, x, st["Y1"][i], st["dY1"][i], dx, dw, src.scratch(capi.conv_wgrad_workspace_bytes(g))))
            st["layers"].append((g3, st["W3"][i], st["X3"][i], st["Y3"][i], st["dY3"][i], st["dX3"][i], st["dW3"][i], ws3))
        stages.append(st)
    return {"pass": _run_densenet, "stages": stages}


def _run_densenet(s):
    for st in s["stages"]:
        for g, W, X, Y, dY, dX, dW, ws in st["layers"]:
            capi.conv_fwd(W, X, Y, None, g)
    for st in reversed(s["stages"]):
        for g, W, X, Y, dY, dX, dW, ws in reversed(st["layers"]):
            capi.conv_dgrad(W, dY, dX, g)
            capi.conv_wgrad(dY, X, dW, g, workspace=ws)
    return [[st[k] for k in ("Y1", "dX1", "dW1", "Y3", "dX3", "dW3")] for st in s["stages"]]


# ---- VGG-16: whole training step, and classification from dataset bytes ---------------------------------------------------
def _prepare_vgg(c, src, seed):
    return {"pass": _run_vgg, "net": Vgg16Step(torch, capi, src.dev, batch=c["batch"], seed=seed)}


def _run_vgg(s):
    net = s["net"]
    net.step()
    # the update clears the gradients and leaves them in the weights and their momentum
    return [net.probs, net.loss, net.dx] + [[st[k] for k in ("W", "b", "mW", "mB")] for st in net.layers()]


def _prepare_infer(c, src, seed):
    n = c["batch"]
    layers = []
    for l in VGG16:
        if l is None:
            shape = layers[-1][-1].shape
            layers.append(("pool", shape, src.empty(*shape), src.empty(shape[0], shape[1], shape[2] // 2, shape[3] // 2)))
        else:
            IC, H, OC = l
            layers.append(("conv", capi.ConvGeom.make(n, IC, H, H, OC, 3, 3, 1, 1, 1, 1), src.normal(OC, IC, 3, 3, std=math.sqrt(2.0 / (IC * 9))),
                           src.normal(OC, std=0.1), src.empty(n, OC, H, H)))
    dense = [(512, o, flags, src.normal(o, 512, std=math.sqrt(2.0 / 512)), src.normal(o, std=0.05), src.empty(n, o)) for o, flags in ((512, capi.CRB_FLAG_RELU), (10, 0))]
    return {"pass": _run_infer, "n": n, "bytes": torch.randint(0, 256, (n, 3, 32, 32), generator=src.gen, dtype=torch.uint8, device=src.dev),
            "x": src.empty(n, 3, 32, 32), "layers": layers, "dense": dense, "probs": src.empty(n, 10)}


def _run_infer(s):
    n, cur = s["n"], s["x"]
    capi.images_from_bytes(s["bytes"], cur, n, 3, 32, 32, capi.NORM_DISTRIBUTION, 0.0, 1.0)
    for l in s["layers"]:
        if l[0] == "conv":
            _, g, W, b, out = l
            capi.conv_fwd(W, cur, out, b, g, capi.CRB_FLAG_RELU)
        else:
            _, shape, record, out = l
            capi.maxpool_fwd(cur, out, record, shape[0] * shape[1], shape[2], shape[3], 2, 2, 2, 2)
        cur = out
    for IN, OUT, flags, W, b, out in s["dense"]:
        capi.linear_fwd(cur, W, b, out, n, IN, OUT, flags)
        cur = out
    capi.softmax(cur, s["probs"], n, 10)
    return cur, s["probs"]


# ---- what a pass cannot do without ------------------------------------------------------------------------------------
def _conv_work(g, passes=3, batch_tensors=4, weights=2):
    """Operands of a layer's passes, each once (X, dY in; Y, dX out; W in, dW out), and their multiply-adds."""
    x, y, w = g.N * g.IC * g.IH * g.IW, g.N * g.OC * g.OH * g.OW, g.OC * g.IC * g.FH * g.FW
    return 4.0 * ((x + y) * batch_tensors / 2 + w * weights), 2.0 * passes * y * g.IC * g.FH * g.FW


def _vgg_work(batch, train):
    b, f = 0.0, 0.0
    for l in VGG16:
        if l is not None:
            g = capi.ConvGeom.make(batch, l[0], l[1], l[1], l[2], 3, 3, 1, 1, 1, 1)
            # a training step reads W and its momentum and writes both (the gradient in between stays inside the step)
            lb, lf = _conv_work(g, 3 if train else 1, 4 if train else 2, 4 if train else 1)
            b, f = b + lb, f + lf
    for o in (512, 10):
        b, f = b + 4.0 * ((4 if train else 1) * 512 * o + (4 if train else 2) * batch * (512 + o) / 2), f + 2.0 * (3 if train else 1) * batch * 512 * o
    return b, f


def work(case):
    c, kind = case, case["kind"]
    if kind == "gemm":
        M, N, K = c["M"], c["N"], c["K"]
        b, f = 4.0 * (M * K + K * N + M * N), 2.0 * M * N * K
    elif kind == "dense":
        n, i, o = c["batch"], c["IN"], c["OUT"]
        # X, W, b, dY and the old dW, dB in; Y, dX, dW, dB out
        b, f = 4.0 * (2 * n * (i + o) + 3 * i * o + 3 * o), 6.0 * n * i * o
    elif kind == "conv":
        b, f = _conv_work(_geom(c), weights=3)
    elif kind == "block":
        n, C, H = c["batch"], c["C"], c["H"]
        cf = _conv_work(capi.ConvGeom.make(n, C, H, H, C, 3, 3, 1, 1, 1, 1))[1]
        # X, the saved activations and dOut in; Z1, A1, Z2, Out and dX out
        b, f = 4.0 * n * C * H * H * 12 + 2 * 4.0 * 3 * C * C * 9, 2 * cf
    elif kind == "resnet":
        b = f = 0.0
        for g, n in _resnet_layers(c["batch"]):
            lb, lf = _conv_work(g, weights=3)
            b, f = b + n * lb, f + n * lf
    elif kind == "densenet":
        b = f = 0.0
        for ones, g3 in _densenet_layers(c["batch"]):
            for g in ones + [g3] * 16:
                lb, lf = _conv_work(g, weights=3)
                b, f = b + lb, f + lf
    else:
        b, f = _vgg_work(c["batch"], kind == "vgg")
    return {"bytes": b, "flops": f}


def tolerance(case):
    """How far another correct fp32 implementation may be off: about four times the distance of these results from float64.

    One contraction of length K was seen 1.2e-8 ... 1.8e-8 * sqrt(K) away in the 2-norm (2e-7 at K = 512, 1.15e-6 at 4096), and
    not under 1e-7. The chains: 1.1e-6 for the logits of VGG-16, 9e-7 for the forward half of a block. In the VGG training step
    a rounding difference also flips a few ReLU masks and pooling choices among tens of millions; every flip is a whole value
    in the gradients behind it (3.5e-3 in the 2-norm, 0.18 of the rms in the largest element)."""
    c, kind = case, case["kind"]
    if kind == "vgg":
        return {"rel": 1.4e-2, "max": 0.75}
    if kind in ("infer", "block"):
        return {"rel": 5e-6}
    K = {"gemm": lambda: c["K"], "dense": lambda: max(c["IN"], c["OUT"], c["batch"]), "conv": lambda: max(c["IC"], c["OC"]) * c["F"] ** 2,
         "resnet": lambda: 576, "densenet": lambda: 432}[kind]()
    return {"rel": max(1e-6, 7e-8 * math.sqrt(K))}
