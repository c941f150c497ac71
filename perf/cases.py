"""Performance cases of the fused spiking-network inference path.

What a program built on this package runs, through its public entry points:
``catfuse_amd.optimize`` on a SpikingJelly-style model or layer, then either
eager calls of the fused model or a replay captured with
``catfuse_amd.capture``, and the functional LIF tails in
``catfuse_amd.kernels``.  Single layers and blocks are called eagerly (what a
program does that fuses part of its model), the classifier layer and whole
networks as captured replays (how a serving loop runs them).

A case is a dict: ``kind`` names the path, the rest its sizes.

conv         Conv2d -> BatchNorm2d -> LIF on spikes [T, B, cin, h, w]
stage        two SEW basic blocks (the first strided, with a downsample)
linear       Linear -> LIF on spikes [T, B, cin], captured
tblock       a Spikformer block (attention, then MLP) on tokens [T, B, N, dim]
sps          the Spikformer patch splitter on images, four pooled stages
sew          SEW-ResNet18 on images, captured; returns logits
vgg          spiking VGG-11-BN on 32 x 32 images, captured; returns logits
spikformer   a Spikformer on images, captured; returns logits
tail         an element-wise LIF tail on fp32 tensors

Weights are kaiming-normal and the BatchNorm statistics those of the
repository's benchmark.  Random weights at the usual threshold of 1 leave deep
layers silent, which trained networks are not, so networks run at the lower
thresholds of the benchmark's live setting (firing rates of 0.2-0.5).
"""
from __future__ import annotations

import math

import torch
import torch.nn as nn
import torch.nn.functional as F

import catfuse_amd
from catfuse_amd import kernels, snn
from catfuse_amd.sparseflow.lif_seq_kernel import lif_sequential

EPS = 1e-5
TAU = 2.0


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # The smallest fused call: one 64-channel layer on CIFAR-size maps,
        # where the launch and the host path count.
        dict(name="conv_c0", kind="conv", cin=64, cout=64, k=3, stride=1, h=32, w=32, T=4, B=8,
             rate=0.15, v_th=0.5),
        # Ragged everything: channels off every tile, a strided conv of a
        # non-square map, a step count off the time block.
        dict(name="conv_ragged", kind="conv", cin=90, cout=170, k=3, stride=2, h=45, w=61, T=6,
             B=5, rate=0.3, v_th=0.5),
        # The middle layer of a ResNet at a serving batch.
        dict(name="conv_c1", kind="conv", cin=256, cout=256, k=3, stride=1, h=14, w=14, T=4, B=32,
             rate=0.2, v_th=0.5),
        # A whole residual stage: strided conv + downsample, three 3x3 convs,
        # two residual adds.
        dict(name="stage2", kind="stage", cin=64, cout=128, h=56, w=56, T=4, B=32, rate=0.3,
             v_th=0.3),
        # Throughput of the headline network at its benchmark batch.
        dict(name="sew_b32", kind="sew", size=224, T=4, B=32, v_th=0.1),
        # The same network on one image: latency.
        dict(name="sew_b1", kind="sew", size=224, T=4, B=1, v_th=0.1),
        # A CIFAR network at its benchmark batch: small maps, AvgPool -> LIF,
        # wide Linear -> LIF layers.
        dict(name="vgg_b64", kind="vgg", T=4, B=64, v_th=0.1),
        # The convolutional front of a spiking transformer: large maps, few
        # channels, max pools.
        dict(name="sps_b8", kind="sps", size=224, dim=384, T=4, B=8, v_th=0.3),
        # One transformer block at the benchmark's width, tokens and batch.
        dict(name="tblock_b32", kind="tblock", dim=384, heads=12, N=196, T=4, B=32, rate=0.3,
             v_th=0.3),
        # A whole spiking transformer on one image: latency.
        dict(name="spikformer_b1", kind="spikformer", size=224, dim=384, heads=12, depth=8, T=4,
             B=1, v_th=0.3),
        # VGG's widest classifier layer.
        dict(name="linear_b64", kind="linear", cin=4096, cout=4096, T=4, B=64, rate=0.25,
             v_th=0.3),
        # An unfused residual add into a neuron, at the first stage's size.
        dict(name="add_lif", kind="tail", op="add", T=4, B=32, C=64, h=56, w=56),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed kinds; sizes over the ranges the listed
    ones stand for (batch 1 to the benchmark's, maps of 7 to 64 pixels,
    channels of 16 to 512, 1 to 8 steps)."""
    kind = rng.choice(["conv", "conv", "conv", "stage", "linear", "tblock", "sps", "sew", "sew",
                       "vgg", "spikformer", "tail"])
    v_th = rng.choice([0.1, 0.2, 0.3])
    T = rng.choice([1, 2, 4, 4, 4, 4, 5, 6, 8])
    rate = round(rng.uniform(0.02, 0.5), 3)
    if kind == "conv":
        c = dict(kind=kind, cin=_log(rng, 16, 512), cout=_log(rng, 16, 512),
                 k=rng.choice([3, 3, 3, 1]), stride=rng.choice([1, 1, 1, 2]), h=_log(rng, 7, 64),
                 w=_log(rng, 7, 64), T=T, B=_log(rng, 1, 32), rate=rate, v_th=0.5)
        if rng.random() < 0.4:       # whole channel groups, as networks mostly have
            c["cin"], c["cout"] = (max(32, 32 * round(c[n] / 32)) for n in ("cin", "cout"))
        while c["B"] > 1 and work(c)["flops"] > 8e10:
            c["B"] = (c["B"] + 1) // 2
        return c
    if kind == "stage":
        cin = rng.choice([32, 64, 64, 128, 256])
        size = rng.randint(max(7, 1792 // cin), 4096 // cin)
        return dict(kind=kind, cin=cin, cout=2 * cin, h=size, w=size, T=rng.choice([2, 4, 4, 6]),
                    B=_log(rng, 1, 32), rate=rate, v_th=v_th)
    if kind == "linear":
        return dict(kind=kind, cin=_log(rng, 64, 4096), cout=_log(rng, 64, 4096), T=T,
                    B=_log(rng, 1, 256), rate=rate, v_th=0.3)
    if kind == "tblock":
        heads = rng.randint(4, 16)
        return dict(kind=kind, dim=32 * heads, heads=heads, N=rng.choice([49, 64, 100, 144, 196]),
                    T=rng.choice([2, 4, 4, 4]), B=_log(rng, 1, 32), rate=rate, v_th=0.3)
    if kind == "sps":
        return dict(kind=kind, size=16 * rng.randint(6, 14), dim=32 * rng.choice([8, 12, 12, 16]),
                    T=rng.choice([2, 4, 4, 6]), B=_log(rng, 1, 16), v_th=v_th)
    if kind == "sew":
        return dict(kind=kind, size=rng.choice([96, 128, 160, 192, 200, 224, 224]),
                    T=rng.choice([2, 4, 4, 6]), B=_log(rng, 1, 24), v_th=v_th)
    if kind == "vgg":
        return dict(kind=kind, T=rng.choice([2, 4, 4, 8]), B=_log(rng, 1, 128), v_th=0.1)
    if kind == "spikformer":
        heads = rng.choice([8, 12])
        return dict(kind=kind, size=rng.choice([128, 160, 192, 224]), dim=32 * heads, heads=heads,
                    depth=rng.randint(2, 8), T=4, B=_log(rng, 1, 4), v_th=0.3)
    return dict(kind="tail", op=rng.choice(["lif", "bn", "add", "avgpool"]), T=T,
                B=_log(rng, 1, 32), C=_log(rng, 16, 256), h=2 * _log(rng, 4, 28),
                w=2 * _log(rng, 4, 28))


# ---------------------------------------------------------------------------
# parameters: (name, shape) in a fixed order, values from the seed
# ---------------------------------------------------------------------------

def _bn(name, c):
    return [(f"{name}.weight", (c,), "gamma"), (f"{name}.bias", (c,), "normal"),
            (f"{name}.running_mean", (c,), "normal"), (f"{name}.running_var", (c,), "var")]


def _conv(name, cin, cout, k):
    return [(f"{name}.weight", (cout, cin, k, k), "kaiming")]


def _lin(name, cin, cout):
    return [(f"{name}.weight", (cout, cin), "kaiming"), (f"{name}.bias", (cout,), "zero")]


def _lbn(name, cin, cout):
    return _lin(name, cin, cout) + _bn(name + "_bn", cout)


def _basic_block(p, cin, cout, stride):
    s = _conv(p + "conv1", cin, cout, 3) + _bn(p + "bn1", cout)
    s += _conv(p + "conv2", cout, cout, 3) + _bn(p + "bn2", cout)
    if stride != 1 or cin != cout:
        s += _conv(p + "downsample.0", cin, cout, 1) + _bn(p + "downsample.1", cout)
    return s


def _token_block(p, dim):
    s = []
    for n in "qkv":
        s += _lbn(f"{p}attn.{n}", dim, dim)
    return s + _lbn(f"{p}attn.proj", dim, dim) + _lbn(f"{p}mlp.fc1", dim, 4 * dim) + \
        _lbn(f"{p}mlp.fc2", 4 * dim, dim)


def _splitter(p, dim):
    s, cin = [], 3
    for i, c in enumerate((dim // 8, dim // 4, dim // 2, dim)):
        s += _conv(f"{p}conv{i}", cin, c, 3) + _bn(f"{p}bn{i}", c)
        cin = c
    return s + _conv(p + "rpe_conv", dim, dim, 3) + _bn(p + "rpe_bn", dim)


VGG = (64, "M", 128, "M", 256, 256, "M", 512, 512, "M", 512, 512, "M")


def _vgg_layers():
    """(conv index, bn index, cin, cout, pooled) of the feature layers."""
    out, i, cin = [], 0, 3
    for j, c in enumerate(VGG):
        if c == "M":
            continue
        pooled = VGG[j + 1] == "M"
        out.append((i, i + 1, cin, c, pooled))
        i, cin = i + (4 if pooled else 3), c
    return out


def _shapes(case):
    kind = case["kind"]
    if kind == "conv":
        return _conv("0", case["cin"], case["cout"], case["k"]) + _bn("1", case["cout"])
    if kind == "stage":
        return _basic_block("0.", case["cin"], case["cout"], 2) + \
            _basic_block("1.", case["cout"], case["cout"], 1)
    if kind == "linear":
        return _lin("0", case["cin"], case["cout"])
    if kind == "tblock":
        return _token_block("0.", case["dim"])
    if kind == "sps":
        return _splitter("0.", case["dim"])
    if kind == "sew":
        s, cin = _conv("conv1", 3, 64, 7) + _bn("bn1", 64), 64
        for n, c in enumerate((64, 128, 256, 512), 1):
            s += _basic_block(f"layer{n}.0.", cin, c, 1 if n == 1 else 2)
            s += _basic_block(f"layer{n}.1.", c, c, 1)
            cin = c
        return s + _lin("fc", 512, 1000)
    if kind == "vgg":
        s = []
        for ci, bi, cin, c, _ in _vgg_layers():
            s += _conv(f"features.{ci}", cin, c, 3) + _bn(f"features.{bi}", c)
        return s + _lin("classifier.0", 512, 4096) + _lin("classifier.2", 4096, 4096) + \
            _lin("classifier.4", 4096, 10)
    s = _splitter("patch_embed.", case["dim"])
    for i in range(case["depth"]):
        s += _token_block(f"blocks.{i}.", case["dim"])
    return s + _lin("head", case["dim"], 1000)


def _parameters(case, seed):
    g = torch.Generator(device="cuda").manual_seed(2 * seed + 1)
    p = {}
    for name, shape, how in _shapes(case):
        if how == "kaiming":
            fan_out = shape[0] * math.prod(shape[2:])
            t = torch.randn(shape, generator=g, device="cuda") * math.sqrt(2.0 / fan_out)
        elif how == "zero":
            t = torch.zeros(shape, device="cuda")
        elif how == "normal":
            t = torch.randn(shape, generator=g, device="cuda") * 0.1
        else:
            t = torch.rand(shape, generator=g, device="cuda")
            t = t * 0.4 + 0.8 if how == "gamma" else t + 0.5
        p[name] = t
    return p


def _input(case, seed):
    g = torch.Generator(device="cuda").manual_seed(2 * seed)
    T, B, kind = case["T"], case["B"], case["kind"]
    if kind in ("sew", "vgg", "spikformer", "sps"):
        n = case.get("size", 32)
        img = torch.randn((B, 3, n, n), generator=g, device="cuda")
        return img.unsqueeze(0).expand(T, B, 3, n, n)     # the same frame at every step
    shape = {"conv": lambda: (T, B, case["cin"], case["h"], case["w"]),
             "stage": lambda: (T, B, case["cin"], case["h"], case["w"]),
             "linear": lambda: (T, B, case["cin"]),
             "tblock": lambda: (T, B, case["N"], case["dim"])}[kind]()
    x = (torch.rand(shape, generator=g, device="cuda") < case["rate"]).float()
    if kind in ("stage", "tblock"):      # a residual stream: sums of spikes
        x += (torch.rand(shape, generator=g, device="cuda") < case["rate"]).float()
    return x


def _tail_inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(2 * seed)
    shape = (case["T"], case["B"], case["C"], case["h"], case["w"])
    z = torch.randn(shape, generator=g, device="cuda")
    v = torch.rand(shape[1:3] + ((case["h"] // 2, case["w"] // 2) if case["op"] == "avgpool"
                                 else shape[3:]), generator=g, device="cuda") * 0.9
    s = {"z": z, "v": v}
    if case["op"] == "add":
        s["z2"] = (torch.rand(shape, generator=g, device="cuda") < 0.3).float()
    if case["op"] == "bn":
        s["scale"] = torch.rand(case["C"], generator=g, device="cuda") * 0.4 + 0.8
        s["shift"] = torch.randn(case["C"], generator=g, device="cuda") * 0.1
    return s


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------

def _model(case):
    kind = case["kind"]
    lif = dict(tau=TAU, v_threshold=case["v_th"], v_reset=0.0, step_mode="m")
    if kind == "conv":
        m = nn.Sequential(
            snn.Conv2d(case["cin"], case["cout"], case["k"], case["stride"], case["k"] // 2,
                       bias=False), snn.BatchNorm2d(case["cout"]), snn.LIFNode(**lif))
    elif kind == "stage":
        cin, c = case["cin"], case["cout"]
        down = nn.Sequential(snn.Conv2d(cin, c, 1, 2, bias=False), snn.BatchNorm2d(c))
        m = nn.Sequential(snn.BasicBlock(cin, c, 2, down, **lif), snn.BasicBlock(c, c, **lif))
    elif kind == "linear":
        m = nn.Sequential(snn.Linear(case["cin"], case["cout"]), snn.LIFNode(**lif))
    elif kind == "tblock":
        m = nn.Sequential(snn.SpikformerBlock(case["dim"], case["heads"], 4.0, case["v_th"],
                                              0.125))
    elif kind == "sps":
        m = nn.Sequential(snn.SpikformerSPS(3, case["dim"], case["v_th"], (0, 1, 2, 3)))
    elif kind == "sew":
        m = snn.sew_resnet18(num_classes=1000, cnf="ADD", **lif)
    elif kind == "vgg":
        m = snn.spiking_vgg11_bn(num_classes=10, **lif)
    else:
        m = snn.Spikformer(img_size=case["size"], embed_dim=case["dim"],
                           num_heads=case["heads"], depth=case["depth"], T=case["T"],
                           v_threshold=case["v_th"], scale=0.125)
    snn.functional.set_step_mode(m, "m")
    return m.eval()


def prepare(case, seed):
    """The fused model (or its captured replay) and its input; for a tail the
    pre-activations and the carried potential."""
    if case["kind"] == "tail":
        return dict(_tail_inputs(case, seed), case=case)
    with torch.device("cuda"), torch.no_grad():     # modules made on the GPU
        m = _model(case)
    p = _parameters(case, seed)
    missing, unexpected = m.load_state_dict(p, strict=False)
    if unexpected or any("num_batches_tracked" not in n for n in missing):
        raise RuntimeError(f"parameters do not fit the model: {missing} {unexpected}")
    fused, _ = catfuse_amd.optimize(m, device="cuda:0", T=case["T"])
    fused.eval()
    x = _input(case, seed)
    if case["kind"] in ("sew", "vgg", "spikformer", "linear"):
        return {"case": case, "x": x, "call": catfuse_amd.capture(fused, x)}
    return {"case": case, "x": x, "model": fused}


def _tail(op, s):
    if op == "lif":
        return lif_sequential(s["z"], s["v"], tau=TAU)
    if op == "bn":
        return kernels.bn_lif(s["z"], s["scale"], s["shift"], s["v"], tau=TAU)
    if op == "add":
        return kernels.add_lif(s["z"], s["z2"], s["v"], tau=TAU)
    return kernels.avgpool_lif(s["z"], s["v"], tau=TAU)


def run(state):
    """One forward from the initial state: a captured network's logits (or
    spikes), an eager layer's spikes as an fp32 tensor, with the final
    potential where the layer is a single neuron."""
    case = state["case"]
    if case["kind"] == "tail":
        return _tail(case["op"], state)
    if "call" in state:
        return state["call"](state["x"])
    with torch.no_grad():
        snn.functional.reset_net(state["model"])
        # a plain fp32 tensor: what the next operation outside the fused model
        # reads (the fused output fills its fp32 form on first use)
        y = state["model"](state["x"]).detach()
        if case["kind"] == "conv":
            return y, state["model"][0].state.tensor.detach()
        return y


# ---------------------------------------------------------------------------
# work and tolerance
# ---------------------------------------------------------------------------

def _out(n, k, stride):
    return (n + 2 * (k // 2) - k) // stride + 1


def _splitter_flops(case):
    fl, n, cin = 0, case["size"], 3
    for i, c in enumerate((case["dim"] // 8, case["dim"] // 4, case["dim"] // 2, case["dim"])):
        fl += (1 if i == 0 else case["T"]) * 18 * cin * c * n * n     # the image once
        n, cin = (n + 1) // 2, c
    return case["B"] * (fl + case["T"] * 18 * cin * cin * n * n), n


def _block_flops(rows, N, dim):
    return 2 * rows * dim * 12 * dim + 4 * rows * 32 * dim


def work(case):
    """Bytes: inputs, weights (fp32) and outputs once; the final potentials
    of the single-neuron cases.  FLOPs: two per multiply-add, the conv of a
    repeated image once."""
    T, B, kind = case["T"], case["B"], case["kind"]
    if kind == "tail":
        n = B * case["C"] * case["h"] * case["w"]
        if case["op"] == "avgpool":
            return {"bytes": 4 * T * n + T * n + 2 * n, "flops": 0}
        return {"bytes": (8 + 4 * (case["op"] == "add")) * T * n + 8 * n, "flops": 0}
    params = 4 * sum(math.prod(s) for _, s, _ in _shapes(case))
    if kind == "conv":
        ho, wo = (_out(case[n], case["k"], case["stride"]) for n in "hw")
        out, k = B * case["cout"] * ho * wo, case["k"]
        return {"bytes": params + 4 * (T * B * case["cin"] * case["h"] * case["w"] + T * out + out),
                "flops": 2 * T * out * case["cin"] * k * k}
    if kind == "stage":
        ho, wo, ci, c = _out(case["h"], 3, 2), _out(case["w"], 3, 2), case["cin"], case["cout"]
        px = T * B * ho * wo
        return {"bytes": params + 4 * (T * B * ci * case["h"] * case["w"] + px * c),
                "flops": 2 * px * c * (10 * ci + 27 * c)}
    if kind == "linear":
        return {"bytes": params + 4 * T * B * (case["cin"] + case["cout"]),
                "flops": 2 * T * B * case["cin"] * case["cout"]}
    if kind == "tblock":
        rows = T * B * case["N"]
        return {"bytes": params + 8 * rows * case["dim"],
                "flops": _block_flops(rows, case["N"], case["dim"])}
    if kind == "sps":
        fl, n = _splitter_flops(case)
        return {"bytes": params + 12 * B * case["size"] ** 2 + 4 * T * B * n * n * case["dim"],
                "flops": fl}
    if kind == "spikformer":
        fl, n = _splitter_flops(case)
        fl += case["depth"] * _block_flops(T * B * n * n, n * n, case["dim"])
        return {"bytes": params + 12 * B * case["size"] ** 2 + 4000 * T * B, "flops": fl}
    if kind == "vgg":
        fl, n = 0, 32
        for _, _, cin, c, pooled in _vgg_layers():
            fl += (1 if cin == 3 else T) * 18 * cin * c * n * n
            n = n // 2 if pooled else n
        fl += 2 * T * (512 * 4096 + 4096 * 4096 + 40960)
        return {"bytes": params + 12 * B * 1024 + 40 * T * B, "flops": B * fl}
    n = _out(case["size"], 7, 2)
    fl, n, cin = 2 * 147 * 64 * n * n, (n + 1) // 2, 64
    for i, c in enumerate((64, 128, 256, 512)):
        n = n if i == 0 else (n + 1) // 2
        fl += 2 * T * n * n * c * (9 * cin + 27 * c + (cin if i else 0))
        cin = c
    fl += 2 * T * 512000
    return {"bytes": params + 12 * B * case["size"] ** 2 + 4000 * T * B, "flops": B * fl}


def tolerance(case):
    """fp32 tails round each step alike on every path.  Behind a conv or
    linear, spikes are thresholds of sums held to about 22 bits: a sum in
    another order moves a potential by 1e-7 to 1e-6, so of a million neurons
    a few may fire one step apart (a relative error of the spikes near 1e-3
    in one layer; 0.01 and 0.02 were seen against 64 bits after a stage's
    four layers and the splitter's five), and in a network such spikes travel
    on.  Spikes are 0 or 1, so one that moved is off by its whole value."""
    if case["kind"] == "tail":
        return {"rel": 1e-5, "max": 1e-3}
    if case["kind"] in ("sew", "vgg", "spikformer"):
        return {"rel": 2e-2, "max": 0.2}
    return {"rel": 2e-2 if case["kind"] in ("stage", "sps") else 4e-3, "max": 0.99}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

def _lif64(z, v_th, v=None):
    v = torch.zeros_like(z[0]) if v is None else v.clone()
    out = torch.empty_like(z)
    for t in range(z.shape[0]):
        v = v + (z[t] - v) / TAU
        s = (v >= v_th).double()
        out[t], v = s, (1.0 - s) * v
    return out, v


def _conv64(x, w, stride=1):
    """Zero-padded convolution of [T, B, C, H, W] as one product a step."""
    w = w.double()
    k = w.shape[-1]
    ho, wo = _out(x.shape[-2], k, stride), _out(x.shape[-1], k, stride)
    out = torch.empty((*x.shape[:2], w.shape[0], ho, wo), dtype=torch.float64, device=x.device)
    for t in range(x.shape[0]):
        for b in range(0, x.shape[1], 8):
            u = F.unfold(x[t, b:b + 8].double(), k, padding=k // 2, stride=stride)
            out[t, b:b + 8] = torch.matmul(w.reshape(w.shape[0], -1), u).unflatten(-1, (ho, wo))
    return out


def _bn64(z, p, name, dim=2):
    shape = [1] * z.dim()
    shape[dim] = -1
    g, b, m, v = (p[f"{name}.{n}"].double().reshape(shape)
                  for n in ("weight", "bias", "running_mean", "running_var"))
    return (z - m) / torch.sqrt(v + EPS) * g + b


def _layer64(x, p, conv, bn, v_th, stride=1):
    return _lif64(_bn64(_conv64(x, p[conv + ".weight"], stride), p, bn), v_th)[0]


def _basic_block64(x, p, pre, v_th, stride):
    y = _layer64(x, p, pre + "conv1", pre + "bn1", v_th, stride)
    y = _layer64(y, p, pre + "conv2", pre + "bn2", v_th)
    if pre + "downsample.0.weight" in p:
        x = _layer64(x, p, pre + "downsample.0", pre + "downsample.1", v_th, stride)
    return x + y


def _maxpool64(x):
    return F.max_pool2d(x.flatten(0, 1), 3, 2, 1).unflatten(0, x.shape[:2])


def _splitter64(x, p, pre, v_th):
    T = x.shape[0]
    z = _bn64(_conv64(x[:1], p[pre + "conv0.weight"]), p, pre + "bn0")
    y = _maxpool64(_lif64(z.expand(T, *z.shape[1:]), v_th)[0])
    for i in (1, 2, 3):
        y = _maxpool64(_layer64(y, p, f"{pre}conv{i}", f"{pre}bn{i}", v_th))
    y = _layer64(y, p, pre + "rpe_conv", pre + "rpe_bn", v_th) + y
    return y.flatten(-2).transpose(-1, -2).contiguous()


def _linear64(x, p, name):
    return torch.matmul(x, p[name + ".weight"].double().t().contiguous()) + \
        p[name + ".bias"].double()


def _token_block64(x, p, pre, heads, v_th):
    def lbl(x, name):
        return _lif64(_bn64(_linear64(x, p, name), p, name + "_bn", 3), v_th)[0]

    q, k, v = (lbl(x, f"{pre}attn.{n}").unflatten(-1, (heads, -1)).transpose(2, 3).contiguous()
               for n in "qkv")
    a = torch.matmul(q, torch.matmul(k.transpose(-1, -2).contiguous(), v)) * 0.125
    a = _lif64(a.transpose(2, 3).flatten(-2), v_th)[0]
    x = x + lbl(a, pre + "attn.proj")
    return x + lbl(lbl(x, pre + "mlp.fc1"), pre + "mlp.fc2")


def _tail64(case, seed):
    s = {k: v.double() for k, v in _tail_inputs(case, seed).items()}
    z = s["z"]
    if case["op"] == "bn":
        z = z * s["scale"].view(-1, 1, 1) + s["shift"].view(-1, 1, 1)
    elif case["op"] == "add":
        z = z + s["z2"]
    elif case["op"] == "avgpool":
        z = F.avg_pool2d(z.flatten(0, 1), 2).unflatten(0, z.shape[:2])
    return _lif64(z, 1.0, s["v"])


def exact(case, seed):
    """What run() returns, from plain torch in 64 bits.  None for whole
    networks: a spike that rounding moves in an early layer changes the
    layers behind it, so two correct evaluations end in different logits."""
    kind = case["kind"]
    if kind in ("sew", "vgg", "spikformer"):
        return None
    if kind == "tail":
        return _tail64(case, seed)
    p, x, v_th = _parameters(case, seed), _input(case, seed), case["v_th"]
    if kind == "sps":
        return _splitter64(x, p, "0.", v_th)
    x = x.double()
    if kind == "conv":
        return _lif64(_bn64(_conv64(x, p["0.weight"], case["stride"]), p, "1"), v_th)
    if kind == "stage":
        return _basic_block64(_basic_block64(x, p, "0.", v_th, 2), p, "1.", v_th, 1)
    if kind == "linear":
        return _lif64(_linear64(x, p, "0"), v_th)[0]
    return _token_block64(x, p, "0.", case["heads"], v_th)
