"""The work a user of this framework has it do, as cases that can be timed and compared.

A case is one call pattern through the public entry points of `matconvnet_amd.vlapi`, the MATLAB-style functions and
the network drivers, on device tensors (a MATLAB array H x W x C x N is a contiguous tensor of shape (N, C, W, H)):

  conv      vl_nnconv: the output, the derivatives, or a layer's forward and backward pass one after the other
  bnorm     vl_nnbnorm, batch moments
  pool      vl_nnpool
  unit      a ResNet bottleneck unit, forward and backward, in the schedule that bench.py times
  train     a training step of ResNet-50: forward, loss derivative, backward, solver
  evaluate  a forward pass of ResNet-50 with the stored moments

`listed()` holds the cases, `draw()` gives more of the same ranges.
"""
import ctypes
import math

import torch

from matconvnet_amd import vlapi

# --------------------------------------------------------------------------------------------------- the cases


def listed():
    return [
        # the single small layer: 5x5x3x32 on a batch of 100 32x32 images; a matter of launches and host work
        _conv("conv first layer", H=32, W=32, C=3, N=100, FH=5, FW=5, K=32, pad=2, bias=True, what="both"),
        # a wide 3x3 layer at a training batch, its derivatives: the largest single layer
        _conv("conv wide 3x3", H=56, W=56, C=256, N=64, FH=3, FW=3, K=256, pad=1, what="backward"),
        # a grouped 5x5 layer on odd planes, as two-column networks have them
        _conv("conv grouped odd", H=27, W=27, C=96, N=128, FH=5, FW=5, K=256, pad=2, groups=2, bias=True, what="both"),
        # a fully connected layer behind 6x6 maps: one output pixel, the bank is what is read
        _conv("conv fully connected", H=6, W=6, C=256, N=128, FH=6, FW=6, K=4096, bias=True, what="both"),
        # a residual network's 3x3 layer in double precision
        _conv("conv double", H=56, W=56, C=64, N=32, FH=3, FW=3, K=64, pad=1, what="backward", double=True),
        # batch normalisation of the widest tensor of a residual unit
        dict(name="bnorm backward", family="bnorm", H=56, W=56, C=256, N=32, what="backward"),
        # the pooling layer behind a residual network's first convolution
        _pool("maxpool backward", H=112, W=112, C=64, N=32, pool=3, stride=2, pad=1, method="max", what="backward"),
        # overlapping max pooling of odd planes, both directions
        _pool("maxpool odd planes", H=55, W=55, C=96, N=128, pool=3, stride=2, pad=0, method="max", what="both"),
        # the bottleneck unit of the headline benchmark
        dict(name="unit", family="unit", H=56, W=56, C=256, M=64, Cout=256, N=32, stride=1, adapter=False),
        # the whole network: a training step, one image to classify, a batch to classify
        dict(name="train", family="train", S=224, N=32, classes=1000),
        dict(name="evaluate one image", family="evaluate", S=224, N=1, classes=1000),
        dict(name="evaluate batch", family="evaluate", S=224, N=32, classes=1000),
    ]


def _conv(name, H, W, C, N, FH, FW, K, what, stride=1, pad=0, groups=1, bias=False, double=False):
    c = dict(family="conv", H=H, W=W, C=C, N=N, FH=FH, FW=FW, K=K, stride=stride, pad=pad, groups=groups, bias=bias,
             what=what, double=double)
    return dict(c, name=name) if name else c


def _pool(name, H, W, C, N, pool, stride, pad, method, what, double=False):
    c = dict(family="pool", H=H, W=W, C=C, N=N, pool=pool, stride=stride, pad=pad, method=method, what=what, double=double)
    return dict(c, name=name) if name else c


def _log_int(rng, low, high):
    """A whole number, spread evenly over its logarithm."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))



def draw(rng):
    family = rng.choice(["conv", "conv", "conv", "bnorm", "pool", "unit", "train", "evaluate", "evaluate"])
    while True:
        if family == "conv":
            kind = rng.choice(["square", "square", "pointwise", "first", "connected"])
            double = rng.random() < 0.15
            groups = 1
            if kind == "connected":
                H = rng.randint(1, 7)
                size, stride, pad = H, 1, 0
                C, K = _log_int(rng, 64, 2048), _log_int(rng, 10, 4096)
            elif kind == "first":
                H = _log_int(rng, 24, 224)
                size, C, K = rng.choice([3, 5, 7]), rng.choice([1, 3]), rng.choice([16, 20, 32, 48, 64, 96])
                stride, pad = rng.choice([1, 1, 2]), size // 2
            else:
                H = _log_int(rng, 7, 112)
                size = 1 if kind == "pointwise" else rng.choice([3, 3, 3, 5])
                groups = 2 if size > 1 and rng.random() < 0.25 else 1
                C, K = groups * _log_int(rng, 16, 512 // groups), groups * _log_int(rng, 16, 512 // groups)
                if rng.random() < 0.6:  # (most layers have round numbers of channels)
                    C, K = (max(16 * groups, v // 32 * 32) for v in (C, K))
                stride, pad = (2 if rng.random() < 0.2 else 1), size // 2
            W = H if kind == "connected" or rng.random() < 0.7 else max(size, H - rng.randint(1, max(1, H // 4)))
            case = _conv(None, H=H, W=W, C=C, N=_log_int(rng, 1, 128), FH=size, FW=size, K=K, stride=stride, pad=pad, groups=groups,
                         bias=rng.random() < 0.5, what=rng.choice(["forward", "backward", "both"]), double=double)
            w = work(case)
            if w["flops"] <= (3e10 if double else 4e11) and w["flops"] >= 2e8 and w["bytes"] <= 1.5e9:
                return case
        elif family == "bnorm":
            case = dict(family="bnorm", H=_log_int(rng, 1, 112), W=0, C=_log_int(rng, 16, 2048), N=_log_int(rng, 1, 256),
                        what=rng.choice(["forward", "backward", "both"]))
            case["W"] = case["H"]
            if 1 << 15 <= case["H"] * case["W"] * case["C"] * case["N"] <= 1 << 26 and case["H"] * case["W"] * case["N"] >= 16:
                return case
        elif family == "pool":
            H = _log_int(rng, 7, 224)
            pool, stride, pad = rng.choice([(3, 2, 0), (3, 2, 1), (2, 2, 0), (3, 1, 1), (0, 1, 0)])
            case = _pool(None, H=H, W=H if rng.random() < 0.7 else max(7, H - rng.randint(1, max(1, H // 4))), C=_log_int(rng, 3, 512),
                         N=_log_int(rng, 1, 256), pool=pool, stride=stride, pad=pad, method=rng.choice(["max", "max", "avg"]),
                         what=rng.choice(["forward", "backward", "both"]), double=rng.random() < 0.15)
            if pool == 0:  # one window over the whole plane, as before a classifier
                H = rng.randint(5, 9)
                case.update(H=H, W=H, pool=H, method="avg")
            if 1 << 16 <= case["H"] * case["W"] * case["C"] * case["N"] <= 3 << 24:
                return case
        elif family == "unit":
            M = rng.choice([32, 64, 64, 128, 256, 512])
            H = max(7, min(64, int(round(3584 / M * rng.uniform(0.7, 1.3)))))
            adapter = rng.random() < 0.3
            case = dict(family="unit", H=H, W=H if rng.random() < 0.8 else max(7, H - rng.randint(1, 5)), C=4 * M, M=M, Cout=4 * M,
                        N=_log_int(rng, 1, 64), stride=1, adapter=adapter)
            if adapter:
                case.update(C=2 * M, stride=2)
            if work(case)["flops"] <= 1.7e11:
                return case
        else:
            train = family == "train"
            case = dict(family=family, S=32 * rng.randint(4 if train else 2, 8), N=_log_int(rng, 8 if train else 1, 64),
                        classes=rng.choice([10, 100, 365, 1000]))
            if case["S"] ** 2 * case["N"] <= 224 ** 2 * 32:
                return case


# ------------------------------------------------------------------------- what a program has in hand, and one pass


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, *shape, dtype=torch.float32):
    return torch.randn(*shape, device="cuda", dtype=dtype, generator=g)


def _out(size, window, stride, pad):
    return (size + 2 * pad - window) // stride + 1


class _DeviceArray:
    """A driver's own buffer, for torch to look at; keeps the driver alive as long as it is looked at."""

    def __init__(self, owner, pointer, count):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=(count,), typestr="<f4", data=(pointer, False), version=2, strides=None)


class _Handle:
    """A network driver, released with the state and the views that hold it."""

    def __init__(self, driver, address):
        self.driver, self.address = driver, address

    def where(self, name):
        n = ctypes.c_size_t(0)
        p = self.address(self.driver.h, name.encode(), ctypes.byref(n))
        if not p:
            raise KeyError(name)
        return p, n.value

    def _tensor(self, pointer, count):
        t = torch.as_tensor(_DeviceArray(self, pointer, count), device="cuda")
        t.owner = self  # (the memory is the driver's: it must outlive every view that is handed out)
        return t

    def view(self, name):
        return self._tensor(*self.where(name))

    def span(self, first, last):
        """The arena from one named buffer to another (all parameters lie in one arena, their derivatives in a second)."""
        (a, _), (b, n) = self.where(first), self.where(last)
        return self._tensor(a, (b - a) // 4 + n)

    def __del__(self):
        torch.cuda.synchronize()
        self.driver.close()


def prepare(case, seed):
    g = _generator(seed)
    family = case["family"]
    if family == "conv":
        dtype = torch.float64 if case["double"] else torch.float32
        fan_in = case["FH"] * case["FW"] * (case["C"] // case["groups"])
        s = dict(case=case)
        s["x"] = _normal(g, case["N"], case["C"], case["W"], case["H"], dtype=dtype)
        s["f"] = _normal(g, case["K"], case["C"] // case["groups"], case["FW"], case["FH"], dtype=dtype) * math.sqrt(2.0 / fan_in)
        s["b"] = 0.1 * _normal(g, case["K"], 1, dtype=dtype) if case["bias"] else torch.empty(0, device="cuda", dtype=dtype)
        Ho, Wo = _out(case["H"], case["FH"], case["stride"], case["pad"]), _out(case["W"], case["FW"], case["stride"], case["pad"])
        s["dy"] = _normal(g, case["N"], case["K"], Wo, Ho, dtype=dtype)
        return s
    if family == "bnorm":
        C = case["C"]
        mean, std = _normal(g, 1, C, 1, 1), 0.5 + 1.5 * torch.rand(1, C, 1, 1, device="cuda", generator=g)
        x = _normal(g, case["N"], C, case["W"], case["H"]) * std + mean
        return dict(case=case, x=x, g=0.5 + torch.rand(C, device="cuda", generator=g), b=0.1 * _normal(g, C), dy=_normal(g, *x.shape))
    if family == "pool":
        dtype = torch.float64 if case["double"] else torch.float32
        # what a pooling layer meets: the output of a ReLU, with its runs of equal values, or (average) plain values
        x = _normal(g, case["N"], case["C"], case["W"], case["H"], dtype=dtype)
        if case["method"] == "max":
            x = torch.clamp_min(x, 0)
        Ho, Wo = (_out(case[d], case["pool"], case["stride"], case["pad"]) for d in "HW")
        return dict(case=case, x=x, dy=_normal(g, case["N"], case["C"], Wo, Ho, dtype=dtype))
    if family == "unit":
        u = vlapi.Bottleneck(H=case["H"], W=case["W"], Cc=case["C"], M=case["M"], N=case["N"], fused=True, Cout=case["Cout"],
                             stride=case["stride"], adapter=case["adapter"], packed=True, deferred=True, epilogue_sums=True,
                             mask_bits=True)
        h = _Handle(u, u.L.vlh_bottleneck_buffer)
        fill_filters(h, g, "", case["C"], case["M"], case["adapter"])
        for layer in ("1", "2", "3") + (("s",) if case["adapter"] else ()):
            v = h.view("g" + layer)
            v.copy_(0.5 + torch.rand(v.numel(), device="cuda", generator=g))
            v = h.view("b" + layer)
            v.copy_(0.1 * _normal(g, v.numel()))
        for name in ("x", "dzdy"):
            v = h.view(name)
            v.copy_(_normal(g, v.numel()))
        h.view("x").clamp_min_(0)  # (a unit's input is the previous unit's ReLU)
        # An element whose last ReLU has its argument within rounding of zero passes all of its derivative or none of it, and
        # over an identity shortcut that element of dzdx is the derivative itself: two correct implementations differ by its
        # whole size there.  (Behind an adapter it is one term of a product.)
        names = ["y"] + (["dzdx"] if case["adapter"] else []) + [d + l for l in ("1", "2", "3") + (("s",) if case["adapter"] else ()) for d in ("df", "dg", "db", "m")]
        return dict(case=case, handle=h, outputs={n: h.view(n) for n in names})
    # the network (the options are those bench.py reports)
    net = vlapi.ResNet50(N=case["N"], image_size=case["S"], classes=case["classes"], channel_sums=True, overlap=True)
    h = _Handle(net, net.L.vlh_resnet50_buffer)
    _he(h, g, "stem.f", 7 * 7 * 3)
    layers, C = ["stem."], 64
    for i, (section, first) in enumerate([(s, l == 0) for s, n in enumerate((3, 4, 6, 3)) for l in range(n)]):
        fill_filters(h, g, "unit%d." % i, C, 64 << section, first)
        layers += ["unit%d.%s" % (i, l) for l in ("1", "2", "3") + (("s",) if first else ())]
        C = 256 << section
    _he(h, g, "fc.f", C)
    for layer in layers:
        head, tail = layer.split(".")
        v = h.view("%s.g%s" % (head, tail))
        v.copy_(0.8 + 0.4 * torch.rand(v.numel(), device="cuda", generator=g))
        v = h.view("%s.b%s" % (head, tail))
        v.copy_(0.1 * _normal(g, v.numel()))
    h.view("fc.b").zero_()
    h.view("input").copy_(_normal(g, h.view("input").numel()))
    h.view("labels").copy_(torch.randint(1, case["classes"] + 1, (case["N"],), device="cuda", generator=g).float())
    net.pack()
    if family == "evaluate":
        # stored moments: those of another batch of this network
        net.forward()
        for layer in layers:
            head, tail = layer.split(".")
            h.view("running.%s.m%s" % (head, tail)).copy_(h.view("%s.m%s" % (head, tail)))
        net.set_test_mode(True)
        h.view("input").copy_(_normal(g, h.view("input").numel()))
        outputs = dict(prediction=h.view("prediction"), features=h.view("avg"), maps=h.view("unit15.y"))
    else:
        # The updated network.  Through fifty layers of ReLUs a rounding changes the derivatives by 1 to 2 %, single elements
        # by all of their size, whatever the implementation, and the next step's prediction with them: the derivatives are
        # seen in the parameters they change (by about 1 % over two steps), the forward pass in the moments.
        outputs = dict(parameters=h.span("stem.f", "fc.b"), stored_moments=h.span("running.stem.m", "running.unit15.m3"))
    return dict(case=case, handle=h, outputs=outputs)


def _he(h, g, name, fan_in):
    v = h.view(name)
    v.copy_(_normal(g, v.numel()) * math.sqrt(2.0 / fan_in))


def fill_filters(h, g, prefix, C, M, adapter):
    _he(h, g, prefix + "f1", C)
    _he(h, g, prefix + "f2", 9 * M)
    _he(h, g, prefix + "f3", M)
    if adapter:
        _he(h, g, prefix + "fs", C)


def run(s):
    case = s["case"]
    family = case["family"]
    if family == "conv":
        options = ("stride", case["stride"], "pad", case["pad"])
        y = vlapi.vl_nnconv(s["x"], s["f"], s["b"], *options) if case["what"] != "backward" else None
        d = vlapi.vl_nnconv(s["x"], s["f"], s["b"], s["dy"], *options) if case["what"] != "forward" else (None, None, None)
        if not case["bias"]:
            d = (d[0], d[1], None)
        return dict(y=y, dzdx=d[0], dzdf=d[1], dzdb=d[2])
    if family == "bnorm":
        y = m = None
        d = (None, None, None, None)
        if case["what"] != "backward":
            y, m = vlapi.vl_nnbnorm(s["x"], s["g"], s["b"], "epsilon", 1e-4, nout=2)
        if case["what"] != "forward":
            d = vlapi.vl_nnbnorm(s["x"], s["g"], s["b"], s["dy"], "epsilon", 1e-4, nout=4)
        return dict(y=y, moments=m, dzdx=d[0], dzdg=d[1], dzdb=d[2], backward_moments=d[3])
    if family == "pool":
        options = ("stride", case["stride"], "pad", case["pad"], "method", case["method"])
        y = vlapi.vl_nnpool(s["x"], case["pool"], *options) if case["what"] != "backward" else None
        d = vlapi.vl_nnpool(s["x"], case["pool"], s["dy"], *options) if case["what"] != "forward" else None
        return dict(y=y, dzdx=d)
    if family == "unit":
        s["handle"].driver.run(1)
        return s["outputs"]
    net = s["handle"].driver
    net.forward()
    if family == "train":
        net.loss_derivative()
        net.backward()
        net.sgd_step(1e-3)
    return s["outputs"]


# ------------------------------------------------------------------------------------- what a pass cannot do without


def _both(case):
    return (case["what"] != "backward"), (case["what"] != "forward")


def _unit_work(H, W, C, M, Cout, N, stride, adapter):
    """Products per direction of a unit, and the tensors a forward and a backward pass read and write."""
    Ho, Wo = (H - 1) // stride + 1, (W - 1) // stride + 1
    flops = 2.0 * N * (H * W * C * M + Ho * Wo * (9 * M * M + M * Cout + (C * Cout if adapter else 0)))
    filters = C * M + 9 * M * M + M * Cout + (C * Cout if adapter else 0)
    inside = N * (H * W * M + Ho * Wo * M)  # what the two inner layers hand on
    ends = N * (H * W * C + Ho * Wo * Cout)
    return flops, filters, inside, ends


def work(case):
    family = case["family"]
    if family == "conv":
        size = 8 if case["double"] else 4
        Ho, Wo = _out(case["H"], case["FH"], case["stride"], case["pad"]), _out(case["W"], case["FW"], case["stride"], case["pad"])
        x, y = case["H"] * case["W"] * case["C"] * case["N"], Ho * Wo * case["K"] * case["N"]
        f = case["FH"] * case["FW"] * (case["C"] // case["groups"]) * case["K"]
        product = 2.0 * Ho * Wo * case["N"] * f
        forward, backward = _both(case)
        return dict(bytes=size * (forward * (x + f + y) + backward * (x + f + y + x + f)), flops=product * (forward + 2 * backward))
    if family == "bnorm":
        e = case["H"] * case["W"] * case["C"] * case["N"]
        forward, backward = _both(case)
        return dict(bytes=4.0 * e * (2 * forward + 3 * backward), flops=float(e * (5 * forward + 9 * backward)))
    if family == "pool":
        size = 8 if case["double"] else 4
        Ho, Wo = (_out(case[d], case["pool"], case["stride"], case["pad"]) for d in "HW")
        planes = case["C"] * case["N"]
        x, y = case["H"] * case["W"] * planes, Ho * Wo * planes
        forward, backward = _both(case)
        reads_x = case["method"] == "max"
        return dict(bytes=float(size * (forward * (x + y) + backward * (x * (1 + reads_x) + y))),
                    flops=float(y * case["pool"] ** 2 * (forward + backward)))
    if family == "unit":
        flops, filters, inside, ends = _unit_work(*(case[k] for k in ("H", "W", "C", "M", "Cout", "N", "stride", "adapter")))
        # forward: the input, the output, the two inner tensors written once; backward: the two ends' derivatives, the
        # input, and the inner tensors read again
        return dict(bytes=4.0 * (2.5 * ends + 2 * inside + 3 * filters), flops=3 * flops)
    # the network
    S, N = case["S"], case["N"]
    flops, filters = 2.0 * N * (S // 2) ** 2 * 147 * 64, 147 * 64
    tensors = 3.0 * N * S * S
    H, C = S // 4, 64
    for section, length in enumerate((3, 4, 6, 3)):
        for l in range(length):
            M, stride = 64 << section, 2 if l == 0 and section else 1
            a, b, inside, ends = _unit_work(H, H, C, M, 4 * M, N, stride, l == 0)
            flops, filters, tensors = flops + a, filters + b, tensors + inside + ends / 2
            H, C = (H - 1) // stride + 1, 4 * M
    flops, filters = flops + 2.0 * N * C * case["classes"], filters + C * case["classes"]
    if family == "train":
        # values, derivatives and momentum read and written by the solver; activations written forward, read backward
        return dict(bytes=4.0 * (7 * filters + 2 * tensors), flops=3 * flops)
    return dict(bytes=4.0 * (filters + 3 * N * S * S + N * case["classes"]), flops=flops)


def tolerance(case):
    """Four times what was seen of the path against itself in 64 bits (conv, bnorm) or with the convolutions' sums in other
    orders (unit, train, evaluate: the general kernels in place of the fast ones); pooling selects and adds in a fixed order."""
    return {
        "conv": {"rel": 1e-14, "max": 1e-13} if case.get("double") else {"rel": 1e-5, "max": 6e-5},  # 2.1e-6, 1.2e-5 (its longest sums)
        "bnorm": {"rel": 3e-7, "max": 1e-6},  # 5.7e-8, 2.0e-7
        "pool": "exact",
        "unit": {"rel": 2.6e-3, "max": 7e-2},  # 6.5e-4, 1.7e-2
        "train": {"rel": 2.4e-3, "max": 1e-1},  # 5.9e-4, 2.2e-2 (two steps)
        "evaluate": {"rel": 3e-4, "max": 2e-3},  # 5.6e-5, 4.1e-4 (the last maps)
    }[case["family"]]
