"""The work a user of this package has it do, as cases that can be timed: single SC operations, layer training
steps, inference and training steps of the two networks of the training script.

A case is a dict of plain values.  ``kind`` says which public entry point runs:

* ``op``     one call of ``sc_extension_cuda`` (forward counts, int32), as external callers of the module make it
* ``func``   ``utils_functional.conv2d_generic`` forward and backward on unquantised float data (the benchmark's step)
* ``layer``  ``utils_class.Conv2d_Add_Partial`` forward and backward, as a layer inside a training loop
* ``infer``  a network in eval mode: module by module (``fused`` 0), or the 4-layer CNN's ``forward_fused`` replayed
             from its HIP graph (``fused`` 1)
* ``train``  ``network.train_step`` of a network (fused blocks, Adam), eager or as a recorded step (``graph`` 1)

Sizes are those of ``geo_amd.workloads``, of the networks of ``geo_amd.network`` with the training script's defaults,
and odd ones between them.
"""
import math

import torch

from geo_amd import _native, network, utils_class, utils_functional

# image side, channels in and out, kernel, padding, layers of that shape: the convolutions of the two networks
_NETS = {
    "cnn4": [(32, 3, 32, 5, 2, 1), (16, 32, 32, 5, 2, 1), (8, 32, 64, 5, 2, 1), (4, 64, 10, 4, 0, 1)],
    "vgg16": [(32, 3, 64, 3, 1, 1), (32, 64, 64, 3, 1, 1), (16, 64, 128, 3, 1, 1), (16, 128, 128, 3, 1, 1),
              (8, 128, 256, 3, 1, 1), (8, 256, 256, 3, 1, 2), (4, 256, 512, 3, 1, 1), (4, 512, 512, 3, 1, 2),
              (2, 512, 512, 3, 1, 3), (1, 512, 10, 1, 0, 1)],
}


def _conv(kind, name, n, c_in, w, h, c_out, k_w, k_h, pad, L, mode="1d_bin", z_unit=32, weights="init", load=2):
    return dict(name=name, kind=kind, n=n, c_in=c_in, w=w, h=h, c_out=c_out, k_w=k_w, k_h=k_h, pad=pad, L=L, mode=mode,
                z_unit=z_unit, weights=weights, load=load)


def _net(kind, name, net, n, err, gain=1.0, fused=0, graph=0):
    return dict(name=name, kind=kind, net=net, n=n, err=err, gain=gain, fused=fused, graph=graph)


def listed():
    return [
        # one image through the 4-layer CNN: launches and host time only
        _net("infer", "cnn4_infer_1", "cnn4", 1, 7, gain=2.0),
        # a small serving batch from the recorded inference graph
        _net("infer", "cnn4_serve_16", "cnn4", 16, 7, gain=2.0, fused=1),
        # the validation pass of the training script at its default batch
        _net("infer", "cnn4_infer_256", "cnn4", 256, 7, gain=2.0),
        # the training script's default step, eager, as training starts
        _net("train", "cnn4_train_256", "cnn4", 256, 7),
        # the same at the benchmark's stream length, recorded and replayed
        _net("train", "cnn4_train_graph_256", "cnn4", 256, 6, graph=1),
        # the training script's larger network (--size 1), under way: with the initial weights of its 512-channel
        # layers nearly every stream is empty
        _net("infer", "vgg16_infer_50", "vgg16", 50, 7, gain=3.0),
        _net("train", "vgg16_train_128", "vgg16", 128, 7, gain=3.0),
        # the smallest convolution of the reference's CPU-runnable range as one module call
        _conv("op", "op_first_layer_32", 32, 3, 32, 32, 32, 3, 3, 1, 64, weights="uniform", load=8),
        # the headline layer step of the benchmark: unquantised floats, uniform weights
        _conv("func", "step_128ch_256", 256, 128, 16, 16, 128, 3, 3, 1, 128, weights="uniform", load=8),
        # the 56 x 56 layer at the longest stream, as a layer of a network
        _conv("layer", "layer_56px_128", 128, 64, 56, 56, 64, 3, 3, 1, 256),
        # the 4096 x 4096 linear layer in OR groups of 16, written as a convolution
        _conv("layer", "linear_4096_1024", 1024, 16, 1, 256, 4096, 1, 256, 0, 128),
        # ragged everything: odd batch, channels and image, block-wise accumulation with a ragged last block
        _conv("layer", "layer_ragged_yz_77", 77, 45, 27, 19, 83, 3, 3, 1, 128, mode="yz_bin", z_unit=32),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _gain(rng, net):
    return round(rng.uniform(1, 3) if net == "cnn4" else rng.uniform(3, 5), 2)


def draw(rng):
    kind = rng.choice(["infer", "infer", "train", "op", "func", "layer", "layer", "layer"])
    if kind == "infer":
        net = rng.choice(["cnn4", "cnn4", "vgg16"])
        return _drop(_net(kind, "", net, _log(rng, 1, 256 if net == "cnn4" else 100), rng.choice([6, 7, 7] if net == "cnn4" else [7, 8]),
                          gain=_gain(rng, net), fused=rng.choice([0, 1]) if net == "cnn4" else 0))
    if kind == "train":
        net = rng.choice(["cnn4", "cnn4", "vgg16"])
        return _drop(_net(kind, "", net, _log(rng, 16, 300 if net == "cnn4" else 120), rng.choice([6, 7, 7] if net == "cnn4" else [7, 8]),
                          gain=_gain(rng, net), graph=rng.choice([0, 1]) if net == "cnn4" else 0))
    L = rng.choice([32, 64, 128, 128, 256])
    mode = "1d_bin"
    if rng.random() < 0.2:  # a linear layer: OR groups of 16 inputs, one image row
        c_in, w, h, k_w, pad = 16, 1, _log(rng, 16, 256), 1, 0
        k_h, c_out, n = h, _log(rng, 64, 4096), _log(rng, 8, 1024)
    else:
        k_w = k_h = rng.choice([1, 3, 3, 3, 5])
        pad = k_w // 2
        c_in, c_out = _log(rng, 3, 512), _log(rng, 8, 512)
        w, h = _log(rng, 4, 64), _log(rng, 4, 64)
        n = _log(rng, 1, 256)
        mode = rng.choice(["1d_bin", "1d_bin", "1d_bin", "yz_bin", "z_bin"])
    if kind == "op" and mode == "1d_bin" and rng.random() < 0.15:
        mode = "acc"  # the accurate-random generator
    weights = rng.choice(["init", "init", "uniform"])
    if c_in * k_w > 400:  # uniform weights over more members: every gradient under the smallest float
        weights = "init"
    c = _conv(kind, "", n, c_in, w, h, c_out, k_w, k_h, pad, L, mode, rng.choice([4, 8, 32]), weights,
              rng.choice([2, 2, 8]))
    # no dearer than a sixth of the largest listed one by its products (small OR groups cost more per product)
    while c["n"] > 1 and _macs(c) * L > 6e11:
        c["n"] = (c["n"] + 1) // 2
    while c["c_out"] > 8 and _macs(c) * L > 6e11:
        c["c_out"] = (c["c_out"] + 1) // 2
    return _drop(c)


def _drop(case):
    case.pop("name")
    return case


def _out_shape(c):
    return c["n"], c["c_out"], c["w"] + 2 * c["pad"] - c["k_w"] + 1, c["h"] + 2 * c["pad"] - c["k_h"] + 1


def _macs(c):
    n, c_out, wo, ho = _out_shape(c)
    return n * c_out * wo * ho * c["c_in"] * c["k_w"] * c["k_h"]


def _q7(t):
    return (t * 128).round().clamp(-127, 127) / 128


def prepare(case, seed):
    torch.manual_seed(seed)  # module initialisation, dropout masks
    g = torch.Generator(device="cuda").manual_seed(seed)
    dev = torch.device("cuda", torch.cuda.current_device())
    if case["kind"] in ("infer", "train"):
        cls = network.CONV_tiny_add_partial if case["net"] == "cnn4" else network.VGG16_add_partial
        net = cls().to(dev)
        net.err = [case["err"]] * len(net.err)
        for m in net.modules():  # training widens the initial weights
            if isinstance(m, utils_class.Conv2d_Add_Partial):
                m.weight_org.mul_(case["gain"]).clamp_(-1, 0.999)
                m.weight.data.copy_(m.weight_org)
        # 8-bit images, as ToTensor gives them
        x = torch.randint(256, (case["n"], 3, 32, 32), generator=g, device=dev).float() / 255
        if case["kind"] == "infer":
            for m in net.modules():  # running statistics as a few hundred training steps leave them: not 0 and 1
                if isinstance(m, (torch.nn.BatchNorm1d, torch.nn.BatchNorm2d)):
                    m.running_mean.uniform_(-0.1, 0.1, generator=g)
                    m.running_var.uniform_(0.02, 0.1, generator=g)
            net.eval()
            return dict(kind="infer", net=net, x=x, fused=case["fused"])
        net.train()
        net.fused_blocks = True
        target = torch.randint(10, (case["n"],), generator=g, device=dev)
        masters = network.make_param_copies(net)
        criterion = torch.nn.CrossEntropyLoss()
        opt = torch.optim.Adam(masters, lr=2e-3, weight_decay=0, capturable=bool(case["graph"]))
        st = dict(kind="train", net=net, x=x, target=target, masters=masters, criterion=criterion, opt=opt, graph=None)
        if case["graph"]:
            st["graph"] = network.GraphedTrainStep(net, criterion, opt, masters, x, target)
        return st
    n, c_in = case["n"], case["c_in"]
    x = torch.rand((n, c_in, case["w"], case["h"]), generator=g, device=dev)
    w_shape = (case["c_out"], c_in, case["k_w"], case["k_h"])
    w = torch.rand(w_shape, generator=g, device=dev) * 2 - 1
    if case["weights"] == "init":  # torch's convolution default: U(-1, 1) / sqrt(fan_in)
        w = w / math.sqrt(c_in * case["k_w"] * case["k_h"])
    if case["kind"] != "func":
        # between layers activations are Hardtanh(0, 1) outputs: a part of them zero, the rest below 1
        x = (x * 1.6 - 0.6).clamp_(0, 1)
    if case["kind"] == "op":
        return dict(kind="op", case=dict(case), x=_q7(x), w=_q7(w) if case["weights"] == "init" else w)
    up = torch.randn(_out_shape(case), generator=g, device=dev) * 1e-2
    st = dict(kind=case["kind"], case=dict(case), x=x, up=up)
    if case["kind"] == "layer":
        layer = utils_class.Conv2d_Add_Partial(c_in, case["c_out"], kernel_size=(case["k_w"], case["k_h"]),
                                               padding=case["pad"], bias=False).to(dev)
        layer.weight_org.copy_(w)
        layer.weight.data.copy_(w)
        st["layer"] = layer
    else:
        st["w"] = w
    return st


def run(state):
    kind = state["kind"]
    if kind == "infer":
        with torch.no_grad():
            if state["fused"]:
                return state["net"].forward_fused(state["x"], graph=True)
            return state["net"](state["x"].detach())
    if kind == "train":
        if state["graph"] is not None:
            loss = state["graph"](state["x"], state["target"])
        else:
            loss = network.train_step(state["net"], state["x"].detach(), state["target"], state["criterion"],
                                      state["opt"], state["masters"])
        return [loss] + [p.data for p in state["net"].parameters()]
    c = state["case"]
    pad = (c["pad"], c["pad"])
    if kind == "op":
        ext = _native.module("sc_extension_cuda")
        if c["mode"] == "acc":
            return ext.conv2d_add_partial_acc_acc(state["x"], state["w"], c["L"], pad, (1, 1), False, 2)
        if c["mode"] == "yz_bin":
            return ext.conv2d_add_yz_variable_acc(state["x"], state["w"], c["L"], pad, (1, 1), 7, c["load"], 2, 2, False,
                                                  c["z_unit"])
        return ext.conv2d_add_partial_variable_acc(state["x"], state["w"], c["L"], pad, (1, 1), 7, c["load"], 2, False,
                                                   0 if c["mode"] == "z_bin" else 2)
    x = state["x"].detach().requires_grad_(True)
    if kind == "layer":
        layer = state["layer"]
        layer.weight.grad = None
        y = layer(x, err=c["L"].bit_length() - 1, forward=c["mode"], z_unit=c["z_unit"], load_unit=c["load"])
        y.backward(state["up"])
        return dict(y=y.detach(), grad_x=x.grad, grad_w=layer.weight.grad)
    w = state["w"].detach().requires_grad_(True)
    y = utils_functional.conv2d_generic(x, w, pad, (1, 1), bit_length=c["L"], forward=c["mode"], generator="lfsr",
                                        z_unit=c["z_unit"], load_unit=c["load"], load_wait_w=2, load_wait_a=2)
    y.backward(state["up"])
    return dict(y=y.detach(), grad_x=x.grad, grad_w=w.grad)


def work(case):
    """``flops``: of the forward one AND and one OR per 32 stream bits and product (a weight has one non-zero rail);
    of the backward 12 per product (recomputation and two gradients on two rails)."""
    train = case["kind"] not in ("op", "infer")
    if case["kind"] in ("infer", "train"):
        macs = weights = 0
        for side, c_in, c_out, k, pad, times in _NETS[case["net"]]:
            out = side + 2 * pad - k + 1
            macs += times * case["n"] * c_out * out * out * c_in * k * k
            weights += times * c_out * c_in * k * k
        L = 2 ** case["err"]
        # images and logits or loss once; each parameter read once, and in training the master copy, two moments,
        # weight_org and the parameter written once as well
        moved = 4 * (case["n"] * (3 * 32 * 32 + 10) + weights * (7 if train else 1))
    else:
        macs, L = _macs(case), case["L"]
        n, c_out, wo, ho = _out_shape(case)
        x, y, w = n * case["c_in"] * case["w"] * case["h"], n * c_out * wo * ho, macs // (n * wo * ho)
        moved = 4 * ((x + w + y) + ((x + w + y) if train else 0))
    return {"bytes": float(moved), "flops": 2.0 * macs * L / 32 + (12.0 * macs if train else 0.0)}


def tolerance(case):
    if case["kind"] == "op":
        return "exact"
    if case["kind"] == "infer":
        # integer counts and one rounding each: the logits of another correct implementation are the same
        return {"rel": 1e-6}
    if case["kind"] == "train":
        # the first Adam step divides a gradient by its own size: where a gradient is all rounding error the weight
        # moves the other way by up to two steps of 2e-3 (weights of rms 0.02); gradients perturbed by 4e-7 moved all
        # weights of a tensor together by 8e-6 at most
        return {"rel": 1e-4, "max": 0.25}
    # z of up to 50 in exp(-z) at fp32: a relative error of 3e-6 against float64 for saturated groups, 5e-7 else
    return {"rel": 1.2e-5, "max": 1.3e-4}


def exact(case, seed):
    """Gradients of a layer in float64 from their closed form: per add group G (a kernel column, a channel, or a block
    of channels and a kernel column) and rail, z = sum over G of x w, value 1 - exp(-z).  The values ``y`` are counts
    over a power of two; the networks' results go through 8-bit roundings: neither has a 64-bit value of its own."""
    if case["kind"] not in ("func", "layer"):
        return None
    st = prepare(case, seed)
    if case["kind"] == "layer":
        x, w = _q7(st["x"]).double(), _q7(st["layer"].weight_org).double()
    else:
        x, w = st["x"].double(), st["w"].double()
    n, c_out, wo, ho = _out_shape(case)
    k_w, k_h, pad = case["k_w"], case["k_h"], case["pad"]
    grad_x, grad_w = torch.empty_like(x), [torch.zeros_like(w), torch.zeros_like(w)]
    rails = (w.clamp(0, 100), (-w).clamp(0, 100))
    if case["mode"] == "z_bin":
        groups = [(slice(c, c + 1), range(k_h)) for c in range(case["c_in"])]
    else:
        step = case["z_unit"] if case["mode"] == "yz_bin" else case["c_in"]
        groups = [(slice(c, min(c + step, case["c_in"])), [v]) for c in range(0, case["c_in"], step) for v in range(k_h)]
    items = max(1, 2 ** 27 // (wo * ho * max(c_out, case["c_in"] * k_w)))
    for n0 in range(0, n, items):
        xp = torch.nn.functional.pad(x[n0:n0 + items], (pad, pad, pad, pad))
        g = st["up"][n0:n0 + items].double().permute(1, 0, 2, 3).reshape(c_out, -1)
        gxp = torch.zeros_like(xp)
        for c, columns in groups:
            taps = [(u, v) for u in range(k_w) for v in columns]
            # (tap, channel, item, a, b) of the group, as rows of one matrix
            col = torch.stack([xp[:, c, u:u + wo, v:v + ho].transpose(0, 1) for u, v in taps])
            shape, col = col.shape, col.reshape(-1, g.shape[1])
            dcol = torch.zeros_like(col)
            for rail, sign, into in ((rails[0], 1, grad_w[0]), (rails[1], -1, grad_w[1])):
                wm = torch.cat([rail[:, c, u, v] for u, v in taps], 1)
                e = g * torch.exp(-(wm @ col)) * sign
                dcol += wm.t() @ e
                dw = (e @ col.t()).reshape(c_out, len(taps), -1)
                for t, (u, v) in enumerate(taps):
                    into[:, c, u, v] += dw[:, t]
            for t, (u, v) in enumerate(taps):
                gxp[:, c, u:u + wo, v:v + ho] += dcol.reshape(shape)[t].transpose(0, 1)
        grad_x[n0:n0 + items] = gxp[:, :, pad:pad + case["w"], pad:pad + case["h"]]
    grad_w = grad_w[0] * (w >= 0) - grad_w[1] * (w <= 0)
    return dict(y=None, grad_x=grad_x, grad_w=grad_w)
