"""Timed cases: the work a user of tmq_amd has it do, through its public entry points.

Five kinds of work, each over the range of sizes it is used at:

  linear      one compact (2-bit) tmq_amd.Linear: a decoder step (one row, a few rows), a prefill (thousands of rows),
              odd row counts and ragged reduction lengths, fp16 rows and the default fp32 rows
  conv        one compact convolution layer: dense, depthwise or transposed; fp32 NCHW tensors as a plain PyTorch model
              passes them, or fp16 channels_last as a fused network hands them on
  resnet      a whole ResNet-18 forward through optimize_for_inference: one image (latency) up to a batch of 64
  qat         quantization-aware training: a full step of a small MLP (launches count), and the weight passes of a step
              over a model's list of layers (soft weights + loss, gradients, clamp), up to tens of millions of weights
  checkpoint  saving a trained model (range-coded or bit-stuffed), loading it into another one, expanding back to fp32

listed() names twelve of them, draw() gives further ones from the same ranges.
"""
import math

import torch
from torch import nn

import tmq_amd
from tmq_amd import ops

DEVICE = "cuda"


def listed():
    return [
        # a decoder step of one sequence: one fp16 row against a 4096 x 4096 layer, latency only
        {"name": "linear_row", "kind": "linear", "M": 1, "K": 4096, "N": 4096, "dtype": "f16", "out": "f32", "bias": False},
        # a few fp32 rows (what a plain PyTorch model passes) through a layer of odd sizes
        {"name": "linear_fp32_rows", "kind": "linear", "M": 5, "K": 1000, "N": 3000, "dtype": "f32", "out": "f32", "bias": True},
        # an fp32 batch of ragged size through a ragged layer
        {"name": "linear_fp32_batch", "kind": "linear", "M": 333, "K": 2000, "N": 1000, "dtype": "f32", "out": "f32", "bias": True},
        # a prefill: matrix-product bound
        {"name": "linear_prefill", "kind": "linear", "M": 4096, "K": 4096, "N": 4096, "dtype": "f16", "out": "f32", "bias": False},
        # a convolution layer in the user's own fp32 NCHW model
        {"name": "conv_fp32", "kind": "conv", "form": "dense", "B": 32, "C": 128, "N": 128, "H": 28, "W": 28, "k": 3, "s": 1,
         "dtype": "f32", "out": "f32", "bias": True},
        # a depthwise layer and an upsampling layer between fp16 channels_last neighbours
        {"name": "conv_depthwise", "kind": "conv", "form": "depthwise", "B": 64, "C": 128, "N": 128, "H": 56, "W": 56, "k": 3,
         "s": 1, "dtype": "f16", "out": "f16", "bias": True},
        {"name": "conv_transposed", "kind": "conv", "form": "transposed", "B": 32, "C": 128, "N": 64, "H": 56, "W": 56, "k": 4,
         "s": 2, "dtype": "f16", "out": "f16", "bias": True},
        # one image, and a full batch, through a whole network
        {"name": "resnet18_image", "kind": "resnet", "B": 1, "size": 224, "dtype": "f32"},
        {"name": "resnet18_batch", "kind": "resnet", "B": 64, "size": 224, "dtype": "f16"},
        # a training step of the README's MLP; the weight passes of a ResNet-18's step (21 layers, 11.2 M weights)
        {"name": "qat_mlp", "kind": "mlp", "batch": 64, "features": 256, "hidden": 128, "classes": 10},
        {"name": "qat_layers", "kind": "qat", "layers": 21, "smallest": 9408, "largest": 2359296},
        # save, load and expand a trained model of 2.3 M weights in range-coded form
        {"name": "checkpoint", "kind": "checkpoint", "layers": 4, "smallest": 52224, "largest": 1048576, "strong": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi, multiple):
    """A size spread over the logarithm of lo .. hi: a multiple of `multiple` half of the time, any number otherwise."""
    n = _log(rng, lo, hi)
    return max(lo, min(hi, (n + multiple // 2) // multiple * multiple if rng.random() < 0.5 else n))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "conv", "conv", "conv", "resnet", "mlp", "qat", "checkpoint"])
    if kind == "linear":
        K, N = _size(rng, 64, 16384, 256), _size(rng, 64, 16384, 64)
        top = max(1, min(4096, int(4096 ** 3 / (K * N))))
        M = rng.randint(1, 16) if rng.random() < 0.4 else _log(rng, 1, top)
        return {"kind": kind, "M": min(M, top), "K": K, "N": N, "dtype": rng.choice(["f16", "f32"]),
                "out": rng.choice(["f16", "f32"]), "bias": rng.random() < 0.5}
    if kind == "conv":
        form = rng.choice(["dense", "dense", "depthwise", "transposed"])
        dtype = rng.choice(["f16", "f32"])
        k, s = (rng.choice([2, 3, 4]), 2) if form == "transposed" else (rng.choice([1, 3, 3, 5]), rng.choice([1, 1, 2]))
        C = 3 if form == "dense" and rng.random() < 0.15 else _size(rng, 16, 512, 32)
        N = C if form == "depthwise" else _size(rng, 16, 512, 32)
        H, W = _size(rng, 7, 112, 7), _size(rng, 7, 112, 4)
        mac, out = k * k * (C * N if form != "depthwise" else C), H * W * (C + (4 if form == "transposed" else 1) * N)
        top = max(1, min(64, int(7e9 / (mac * H * W)), int(5e7 / out)))
        return {"kind": kind, "form": form, "B": _log(rng, 1, top), "C": C, "N": N, "H": H, "W": W, "k": k, "s": s,
                "dtype": dtype, "out": "f16" if dtype == "f16" else "f32", "bias": rng.random() < 0.5}
    if kind == "resnet":
        size = 32 * rng.randint(3, 8)
        return {"kind": kind, "B": _log(rng, 1, max(1, 64 * 224 * 224 // (size * size))) if size > 224 else _log(rng, 1, 64),
                "size": size, "dtype": rng.choice(["f16", "f32"])}
    if kind == "mlp":
        return {"kind": kind, "batch": _log(rng, 16, 512), "features": _size(rng, 64, 2048, 64),
                "hidden": _size(rng, 64, 2048, 64), "classes": rng.randint(2, 200)}
    small = _log(rng, 100, 60000)
    if kind == "qat":
        return {"kind": kind, "layers": rng.randint(1, 21), "smallest": small, "largest": _log(rng, small, 1 << 21)}
    return {"kind": kind, "layers": rng.randint(1, 4), "smallest": small, "largest": _log(rng, small, 1 << 20),
            "strong": rng.random() < 0.7}


# ---- inputs --------------------------------------------------------------------------------------------------------
_DTYPE = {"f16": torch.float16, "f32": torch.float32}


def _ternary(shape, gen):
    """Trained weights: half of them zero, the rest +-1."""
    u = torch.rand(shape, generator=gen, device=DEVICE)
    return (u < 0.25).float() - (u > 0.75).float()


def _spread(count, lo, hi):
    """`count` sizes from lo to hi, evenly over their logarithm."""
    return [int(round(lo * (hi / lo) ** (i / max(1, count - 1)))) for i in range(count)]


class _Block(nn.Module):
    def __init__(self, cin, cout, stride):
        super().__init__()
        self.conv1, self.bn1 = nn.Conv2d(cin, cout, 3, stride, 1, bias=False), nn.BatchNorm2d(cout)
        self.conv2, self.bn2 = nn.Conv2d(cout, cout, 3, 1, 1, bias=False), nn.BatchNorm2d(cout)
        self.downsample = None
        if stride != 1 or cin != cout:
            self.downsample = nn.Sequential(nn.Conv2d(cin, cout, 1, stride, 0, bias=False), nn.BatchNorm2d(cout))

    def forward(self, x):
        idt = x if self.downsample is None else self.downsample(x)
        out = torch.relu(self.bn1(self.conv1(x)))
        return torch.relu(self.bn2(self.conv2(out)) + idt)


class _ResNet18(nn.Module):
    def __init__(self, classes=102):
        super().__init__()
        self.conv1, self.bn1 = nn.Conv2d(3, 64, 7, 2, 3, bias=False), nn.BatchNorm2d(64)
        self.maxpool = nn.MaxPool2d(3, 2, 1)
        stages, cin = [], 64
        for i, c in enumerate((64, 128, 256, 512)):
            stages.append(nn.Sequential(_Block(cin, c, 1 if i == 0 else 2), _Block(c, c, 1)))
            cin = c
        self.layer1, self.layer2, self.layer3, self.layer4 = stages
        self.avgpool = nn.AdaptiveAvgPool2d(1)
        self.fc = nn.Linear(512, classes)

    def forward(self, x):
        x = self.maxpool(torch.relu(self.bn1(self.conv1(x))))
        x = self.layer4(self.layer3(self.layer2(self.layer1(x))))
        return self.fc(torch.flatten(self.avgpool(x), 1))


class _Mlp(nn.Module):
    def __init__(self, features, hidden, classes):
        super().__init__()
        # (no biases: a BatchNorm behind the layer takes them out again)
        self.fc1, self.bn1 = nn.Linear(features, hidden, bias=False), nn.BatchNorm1d(hidden)
        self.fc2, self.bn2 = nn.Linear(hidden, classes, bias=False), nn.BatchNorm1d(classes)

    def forward(self, x):
        return self.bn2(self.fc2(torch.relu(self.bn1(self.fc1(x)))))


def _train(model, gen, layers=(nn.Linear, nn.Conv2d, nn.ConvTranspose2d)):
    """Give the `layers` of `model` trained ternary weights and its norms the statistics that go with them."""
    with torch.no_grad():
        for m in model.modules():
            if isinstance(m, layers):
                m.weight.data = _ternary(m.weight.shape, gen)
                if m.bias is not None:
                    m.bias.data.normal_(generator=gen)
            elif isinstance(m, nn.BatchNorm2d):
                # statistics of a trained network: they divide by the spread the layer's sums have
                m.running_mean.normal_(0, 1, generator=gen)
                m.running_var.uniform_(0.8, 1.25, generator=gen)
                m.weight.uniform_(0.75, 1.25, generator=gen)
                m.bias.normal_(0, 0.1, generator=gen)
        convs = [m for m in model.modules() if isinstance(m, layers) and m.weight.dim() == 4]
        norms = [m for m in model.modules() if isinstance(m, nn.BatchNorm2d)]
        for conv, bn in zip(convs, norms):
            bn.running_var.mul_(0.5 * conv.weight[0].numel())
    return model


def _compact(model, gen):
    """Swap the layers of `model` for quantized ones, give them trained ternary weights and pack them."""
    ctrl = tmq_amd.QuantizationControl(post_scale=False)
    tmq_amd.quantize_model(model, ctrl)
    model.to(DEVICE).eval()
    _train(model, gen, tmq_amd.TMQLayer)
    tmq_amd.compressed_state_dict(model)
    return model


class _Layers(nn.Module):
    """Linear and 3 x 3 convolution layers in turn, `sizes` weights each (rounded to whole filters)."""

    def __init__(self, sizes):
        super().__init__()
        made = []
        for i, n in enumerate(sizes):
            if i % 2 == 0:
                a = max(1, int(round(n ** 0.5)))
                made.append(nn.Linear(a, max(1, n // a), bias=False))
            else:
                a = max(1, int(round((n / 9) ** 0.5)))
                made.append(nn.Conv2d(a, max(1, n // (9 * a)), 3, bias=False))
        self.layers = nn.ModuleList(made)


def _conv_layer(case):
    C, N, k, s = case["C"], case["N"], case["k"], case["s"]
    if case["form"] == "transposed":
        return nn.ConvTranspose2d(C, N, k, s, (k - s) // 2, bias=case["bias"])
    return nn.Conv2d(C, N, k, s, k // 2, groups=C if case["form"] == "depthwise" else 1, bias=case["bias"])


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    kind, st = case["kind"], {"case": case}
    if kind == "linear":
        model = _compact(nn.Sequential(nn.Linear(case["K"], case["N"], bias=case["bias"])), gen)
        st["layer"] = model[0]
        st["x"] = torch.randn(case["M"], case["K"], generator=gen, device=DEVICE).to(_DTYPE[case["dtype"]])
    elif kind == "conv":
        st["layer"] = _compact(nn.Sequential(_conv_layer(case)), gen)[0]
        x = torch.randn(case["B"], case["C"], case["H"], case["W"], generator=gen, device=DEVICE)
        st["x"] = x if case["dtype"] == "f32" else x.to(dtype=torch.float16, memory_format=torch.channels_last)
    elif kind == "resnet":
        st["session"] = tmq_amd.optimize_for_inference(_compact(_ResNet18(), gen))
        st["x"] = torch.randn(case["B"], 3, case["size"], case["size"], generator=gen, device=DEVICE).to(_DTYPE[case["dtype"]])
    elif kind == "mlp":
        ctrl = tmq_amd.QuantizationControl(epoch_knots=tmq_amd.QuantizationScheduleBuilder.default_schedule(150),
                                           qpenalty_range=(5e-4, 5e-4))
        model = _Mlp(case["features"], case["hidden"], case["classes"])
        tmq_amd.quantize_model(model, ctrl)
        model.to(DEVICE).train()
        for m in model.modules():
            if isinstance(m, tmq_amd.TMQLayer):
                m.weight.data = 2 * torch.rand(m.weight.shape, generator=gen, device=DEVICE) - 1
        for epoch in range(60):
            ctrl.step(epoch)
        st.update(model=model, ctrl=ctrl, opt=torch.optim.SGD(model.parameters(), lr=1e-4))
        st["x"] = torch.randn(case["batch"], case["features"], generator=gen, device=DEVICE)
        st["labels"] = torch.randint(0, case["classes"], (case["batch"],), generator=gen, device=DEVICE)
    elif kind == "qat":
        sizes = _spread(case["layers"], case["smallest"], case["largest"])
        st["weights"] = [(2.04 * torch.rand(n, generator=gen, device=DEVICE) - 1.02) for n in sizes]
        st["grads"] = [1e-2 * torch.randn(n, generator=gen, device=DEVICE) for n in sizes]
        st["upstream"] = torch.ones(1, device=DEVICE)
        st["clamped"] = [w.clone() for w in st["weights"]]        # what an optimizer step would leave to clamp
        st["table"] = ops.SegmentTable(st["clamped"])
    else:
        sizes = _spread(case["layers"], case["smallest"], case["largest"])
        model, other = _Layers(sizes), _Layers(sizes)
        for m in (model, other):
            tmq_amd.quantize_model(m, tmq_amd.QuantizationControl())
            m.to(DEVICE).eval()
        for layer in model.layers:
            layer.weight.data = _ternary(layer.weight.shape, gen)
        st.update(model=model, other=other)
    return st


# ---- one pass ------------------------------------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("linear", "conv"):
        if case["out"] == "f32":                 # the default
            return state["layer"](state["x"])
        before = tmq_amd.set_compact_output_dtype(torch.float16)
        y = state["layer"](state["x"])
        tmq_amd.set_compact_output_dtype(before)
        return y
    if kind == "resnet":
        return state["session"](state["x"])
    if kind == "mlp":
        model, ctrl, opt = state["model"], state["ctrl"], state["opt"]
        opt.zero_grad()
        out = model(state["x"])
        loss = nn.functional.cross_entropy(out, state["labels"]) + ctrl.quantization_loss()
        loss.backward()
        opt.step()
        ctrl.clamp()
        return [loss.detach(), out.detach()] + [p.grad for p in model.parameters() if p.grad is not None] + \
            [model.fc1.weight.detach(), model.fc2.weight.detach()]
    if kind == "qat":
        ys, loss = ops.softstep_fwd_all(state["weights"], 3.0004, True, 5.0, 5e-4)
        dws = ops.softstep_bwd_all(state["weights"], state["grads"], state["upstream"], 3.0004, 5.0, 5e-4)
        ops.clamp_multi_(state["table"], -1.0, 1.0)
        return list(ys) + [loss] + list(dws) + state["clamped"]
    model, other = state["model"], state["other"]
    saved = tmq_amd.compressed_state_dict(model, strong=case["strong"])
    tmq_amd.load_compressed_state_dict(other, saved)
    tmq_amd.expand_compact_layers(model)
    # a stream's length depends on the weights: hand it back in a buffer of the size every stream of the layer fits
    streams = [saved["layers.%d.weight" % i].reshape(-1) for i in range(len(model.layers))]
    if case["strong"]:
        streams = [nn.functional.pad(s, (0, layer.weight.numel() // 4 + 64 - s.numel())) for s, layer in zip(streams, model.layers)]
    return streams + \
        [layer.weight.data for layer in other.layers] + [layer.weight.data for layer in model.layers]


# ---- the same in 64 bits, plain torch ------------------------------------------------------------------------------
def _conv64(x, layer):
    """A convolution layer of torch.nn on a float64 tensor, as columns and one matrix product."""
    w, k, s, p = layer.weight.double(), layer.kernel_size, layer.stride, layer.padding
    B, C, H, W = x.shape
    if isinstance(layer, nn.ConvTranspose2d):
        size = [(n - 1) * s[i] - 2 * p[i] + k[i] for i, n in enumerate((H, W))]
        cols = (w.reshape(C, -1).t() @ x.permute(1, 0, 2, 3).reshape(C, -1)).view(-1, B, H * W).permute(1, 0, 2)
        y = nn.functional.fold(cols, size, k, stride=s, padding=p)
    else:
        size = [(n + 2 * p[i] - k[i]) // s[i] + 1 for i, n in enumerate((H, W))]
        cols = nn.functional.unfold(x, k, padding=p, stride=s)
        if layer.groups != 1:
            y = (cols.view(B, C, k[0] * k[1], -1) * w.view(1, C, -1, 1)).sum(2)
        else:
            y = (w.reshape(len(w), -1) @ cols.permute(1, 0, 2).reshape(cols.shape[1], -1)).view(len(w), B, -1).permute(1, 0, 2)
        y = y.reshape(B, -1, *size)
    return y if layer.bias is None else y + layer.bias.double().view(1, -1, 1, 1)


def _norm64(x, bn):
    v = [t.double().view(1, -1, 1, 1) for t in (bn.running_mean, bn.running_var, bn.weight, bn.bias)]
    return (x - v[0]) / (v[1] + bn.eps).sqrt() * v[2] + v[3]


def _resnet64(net, x):
    x = nn.functional.max_pool2d(torch.relu(_norm64(_conv64(x, net.conv1), net.bn1)), 3, 2, 1)
    for stage in (net.layer1, net.layer2, net.layer3, net.layer4):
        for block in stage:
            idt = x if block.downsample is None else _norm64(_conv64(x, block.downsample[0]), block.downsample[1])
            y = torch.relu(_norm64(_conv64(x, block.conv1), block.bn1))
            x = torch.relu(_norm64(_conv64(y, block.conv2), block.bn2) + idt)
    return x.mean((2, 3)) @ net.fc.weight.double().t() + net.fc.bias.double()


def _staircase64(w, d, order):
    """The soft staircase of steepness d (order 0), its slope (1) and the slope's derivative (2)."""
    half = min(3.0, d / 2)
    c = 2 * half * (half * half + 27) / (27 + 9 * half * half)
    x = (d * (w - w.floor()) - d / 2).clamp(-3, 3)
    b = x * x + 3
    if order == 0:
        return x * (x * x + 27) / (9 * b) / c + 0.5 + w.floor()
    return d * (b - 12) ** 2 / (9 * b * b) / c if order == 1 else d * d * 16 * x * (b - 12) / (3 * b ** 3) / c


class _Soft64(torch.autograd.Function):
    """The staircase with the slope the training rule gives it, order 0, or the penalty on it, order 1."""

    @staticmethod
    def forward(ctx, w, d, order, strength):
        ctx.save_for_backward(w)
        ctx.args = d, order, strength
        return strength * _staircase64(w, d, order)

    @staticmethod
    def backward(ctx, g):
        d, order, strength = ctx.args
        return g * strength * _staircase64(ctx.saved_tensors[0], d, order + 1), None, None, None


@torch.enable_grad()
def exact(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    kind = case["kind"]
    if kind == "linear":
        layer = _train(nn.Sequential(nn.Linear(case["K"], case["N"], bias=case["bias"])).to(DEVICE), gen)[0]
        x = torch.randn(case["M"], case["K"], generator=gen, device=DEVICE).to(_DTYPE[case["dtype"]])
        y = x.double() @ layer.weight.detach().double().t()
        return y if layer.bias is None else y + layer.bias.detach().double()
    if kind == "conv":
        layer = _train(nn.Sequential(_conv_layer(case)).to(DEVICE), gen)[0].requires_grad_(False)
        x = torch.randn(case["B"], case["C"], case["H"], case["W"], generator=gen, device=DEVICE)
        return _conv64(x.to(_DTYPE[case["dtype"]]).double(), layer)
    if kind == "resnet":
        net = _train(_ResNet18().to(DEVICE).eval(), gen).requires_grad_(False)
        x = torch.randn(case["B"], 3, case["size"], case["size"], generator=gen, device=DEVICE).to(_DTYPE[case["dtype"]])
        return _resnet64(net, x.double())
    if kind == "mlp":
        net = _Mlp(case["features"], case["hidden"], case["classes"]).to(DEVICE).double().train()
        for m in (net.fc1, net.fc2):
            m.weight.data = (2 * torch.rand(m.weight.shape, generator=gen, device=DEVICE) - 1).double()
        x = torch.randn(case["batch"], case["features"], generator=gen, device=DEVICE).double()
        labels = torch.randint(0, case["classes"], (case["batch"],), generator=gen, device=DEVICE)
        schedule = tmq_amd.QuantizationControl(epoch_knots=tmq_amd.QuantizationScheduleBuilder.default_schedule(150),
                                               qpenalty_range=(5e-4, 5e-4))
        for epoch in range(60):
            schedule.step(epoch)
        w1, w2 = (_Soft64.apply(m.weight, schedule.digamma, 0, 1.0) for m in (net.fc1, net.fc2))
        out = net.bn2(torch.relu(net.bn1(x @ w1.t())) @ w2.t())
        loss = nn.functional.cross_entropy(out, labels)
        for m in (net.fc1, net.fc2):
            loss = loss + _Soft64.apply(m.weight, schedule.qpenalty_sharpness, 1, schedule.qpenalty).mean()
        loss.backward()
        grads = [p.grad for p in net.parameters()]
        return [loss.detach(), out.detach()] + grads + [(m.weight.detach() - 1e-4 * m.weight.grad).clamp(-1, 1) for m in (net.fc1, net.fc2)]
    if kind == "qat":
        sizes = _spread(case["layers"], case["smallest"], case["largest"])
        ws = [(2.04 * torch.rand(n, generator=gen, device=DEVICE) - 1.02).double() for n in sizes]
        gs = [(1e-2 * torch.randn(n, generator=gen, device=DEVICE)).double() for n in sizes]
        loss = sum(5e-4 * _staircase64(w, 5.0, 1).mean() for w in ws)
        return [_staircase64(w, 3.0004, 0) for w in ws] + [loss] + \
            [g * _staircase64(w, 3.0004, 1) + 5e-4 / w.numel() * _staircase64(w, 5.0, 2) for w, g in zip(ws, gs)] + \
            [w.clamp(-1, 1) for w in ws]
    return None                                    # bytes, words and whole numbers


# ---- what a pass cannot do without ---------------------------------------------------------------------------------
def _conv_out(case):
    H, W, k, s = case["H"], case["W"], case["k"], case["s"]
    if case["form"] == "transposed":
        p = (k - s) // 2
        return (H - 1) * s - 2 * p + k, (W - 1) * s - 2 * p + k
    return (H + 2 * (k // 2) - k) // s + 1, (W + 2 * (k // 2) - k) // s + 1


def work(case):
    kind = case["kind"]
    width = {"f16": 2, "f32": 4}
    if kind == "linear":
        M, K, N = case["M"], case["K"], case["N"]
        return {"bytes": M * K * width[case["dtype"]] + K * N / 4 + M * N * width[case["out"]], "flops": 2 * M * K * N}
    if kind == "conv":
        B, C, N, H, W, k = (case[v] for v in ("B", "C", "N", "H", "W", "k"))
        ho, wo = _conv_out(case)
        per = 1 if case["form"] == "depthwise" else C
        where = H * W if case["form"] == "transposed" else ho * wo
        return {"bytes": B * C * H * W * width[case["dtype"]] + per * N * k * k / 4 + B * N * ho * wo * width[case["out"]],
                "flops": 2 * B * N * per * k * k * where}
    if kind == "resnet":
        B, area = case["B"], case["size"] ** 2
        return {"bytes": B * 3 * area * width[case["dtype"]] + 11.22e6 / 4 + B * 102 * 4, "flops": 3.627e9 * B * area / 224 ** 2}
    if kind == "mlp":
        n = case["hidden"] * (case["features"] + case["classes"])
        # soft weights 8, gradients 12, update 12 and clamp 8 bytes a weight; three products
        return {"bytes": 40 * n + 4 * case["batch"] * (case["features"] + case["classes"]), "flops": 6 * n * case["batch"]}
    n = sum(_spread(case["layers"], case["smallest"], case["largest"]))
    if kind == "qat":
        # forward reads w and writes y, backward reads w and g and writes dw, the clamp reads and writes w
        return {"bytes": 28 * n, "flops": 60 * n}
    # fp32 in, the stored form out and in, compact words in the other model, fp32 back
    return {"bytes": 4 * n + 2 * (0.19 if case["strong"] else 0.25) * n + 0.25 * n + 4 * n, "flops": 2 * n}


def tolerance(case):
    """Four times what the path differs by from a 64-bit computation of the same case (mlp: from itself with the rows in
    another order, sums in another order)."""
    kind = case["kind"]
    if kind == "checkpoint":
        return "exact"
    if kind == "qat":
        return {"rel": 1e-6}                   # element-wise outputs are the same bits; the loss is a sum
    if kind == "mlp":
        return {"rel": 2e-6}                   # 2e-7 .. 4e-7
    if kind == "resnet":
        return {"rel": 1.2e-3}                 # 3.0e-4: fp16 between the layers
    if kind == "conv" or case["out"] == "f16":
        return {"rel": 9e-4}                   # 2.1e-4: an fp32 input goes in as one fp16 term, fp16 results are rounded
    return {"rel": 5e-6}                       # 1.2e-6: fp32 sums
