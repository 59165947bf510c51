"""The work a user of this package has it do, as measurable cases.

Every case goes through the public classes: the autograd functions of the operator (max/average separation, attention
compression), the block that separates a whole pyramid (`AlternateCorrBlockSepflow.separate`), its windowed lookup
and the lookup in the separated volumes (`CorrBlock1D`), each in the direction(s) it is used in.  Sizes are those of
feature maps (1/8 of the image).  Image 2 is image 1 displaced, plus noise, as two frames of a video are: the maxima of
the correlation then lie where a matching network finds them.
"""
import math

import torch

from separableflowthesis_amd import (AlternateCorrBlockSepflow, ComputeMaxArgmaxAvgFunction, ComputeMaxAvgFunction,
                                     ComputeSelfCompressionFunction, CorrBlock1D)

RADIUS = 4


def listed():
    return [
        # a thumbnail pair: the smallest call, nearly all launch and hand-over
        dict(name="maxavg_24x32", kind="maxavg", B=1, H=24, W=32, C=256),
        # inference on a small crop (384x512 image)
        dict(name="maxavg_48x64", kind="maxavg", B=1, H=48, W=64, C=256),
        # training step of the max/average operator alone, small batch
        dict(name="maxavg_train_48x64_b4", kind="maxavg_train", B=4, H=48, W=64, C=256),
        # training step of both operators on 440x1024 images: the benchmark's headline workload
        dict(name="op_train_55x128_b2", kind="op_train", B=2, H=55, W=128, C=256, K=4),
        # inference of both operators on a full-HD image: the largest volume
        dict(name="op_136x240", kind="op", B=1, H=136, W=240, C=256, K=4),
        # odd sizes, a feature count that is no multiple of the tiles, two attention channels
        dict(name="op_train_47x61_c100", kind="op_train", B=2, H=47, W=61, C=100, K=2),
        # inference of the block on a 440x1024 pair: four levels, attention included
        dict(name="separate_55x128", kind="separate", B=1, H=55, W=128, C=256, K=4),
        # the same on wide driving scenes (375x1242, padded to 376x1248): ragged at every level
        dict(name="separate_47x156", kind="separate", B=1, H=47, W=156, C=256, K=2),
        # training step of the block, 440x1024
        dict(name="separate_train_55x128_b2", kind="separate_train", B=2, H=55, W=128, C=256, K=4),
        # training step of the block on 320x448 crops with the batch that is trained with
        dict(name="separate_train_40x56_b12", kind="separate_train", B=12, H=40, W=56, C=256, K=4),
        # what one flow iteration reads at inference: window lookup and lookup in both separated volumes
        dict(name="lookup_55x128", kind="lookup", B=1, H=55, W=128, C=256),
        # the same with its backward pass, as one flow iteration of a training step
        dict(name="lookup_train_55x128_b2", kind="lookup_train", B=2, H=55, W=128, C=256),
    ]


def draw(rng):
    """Sizes spread over their logarithm between thumbnails and 1/8 of a full-HD image; odd ones as likely as even ones."""
    def between(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["maxavg", "maxavg_train", "op", "op_train", "separate", "separate_train", "lookup", "lookup_train"])
    case = dict(kind=kind, B=between(1, 12), H=between(16, 136), W=between(24, 240),
                C=256 if rng.random() < 0.7 else between(32, 256))
    if kind in ("op", "op_train", "separate", "separate_train"):
        case["K"] = rng.choice([1, 2, 3, 4, 4])
    # no dearer than the largest listed case of its kind allows (a training step: the larger of the two listed ones)
    limit = 2.5e11 if kind.endswith("train") else 1.0e12
    if kind.startswith("lookup"):
        while case["B"] * case["H"] * case["W"] > 30000:
            case["B" if case["B"] > 1 else "H"] = max(1, int(case["B" if case["B"] > 1 else "H"] * 0.7))
    while work(case)["flops"] > limit:
        if case["B"] > 1:
            case["B"] = max(1, case["B"] // 2)
        else:
            case["H"], case["W"] = max(16, int(case["H"] * 0.8)), max(24, int(case["W"] * 0.8))
    return case


def _features(case, g):
    """Two (B,C,H,W) feature maps of unit variance, the second the first displaced by a few pixels plus noise."""
    B, H, W, C = case["B"], case["H"], case["W"], case["C"]
    fmap1 = torch.randn(B, C, H, W, generator=g, device="cuda")
    fmap2 = 0.8 * torch.roll(fmap1, shifts=(2, -5), dims=(2, 3)) + 0.6 * torch.randn(B, C, H, W, generator=g, device="cuda")
    return fmap1, fmap2


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    kind, B, H, W, C = case["kind"], case["B"], case["H"], case["W"], case["C"]
    K = case.get("K", 0)
    train = kind.endswith("train")
    fmap1, fmap2 = _features(case, g)
    s = {"kind": kind}
    if kind.startswith(("maxavg", "op")):
        # the operator's own layout, image 1 scaled as its caller scales it
        s["f1"] = (fmap1.permute(0, 2, 3, 1).contiguous() / math.sqrt(C)).requires_grad_(train)
        s["f2"] = fmap2.permute(0, 2, 3, 1).contiguous().requires_grad_(train)
        s["grads"] = [_randn(g, B, H, W, 2, H), _randn(g, B, H, W, 2, W)] if train else []
        if K:
            s["a_u"] = _randn(g, B, H, W, K, W).softmax(-1).requires_grad_(train)
            s["a_v"] = _randn(g, B, H, W, K, H).softmax(-1).requires_grad_(train)
            s["grads"] += [_randn(g, B, H, W, K, H), _randn(g, B, H, W, K, W)] if train else []
    elif kind.startswith("separate"):
        s["fmap1"], s["fmap2"] = fmap1.requires_grad_(train), fmap2.requires_grad_(train)
        s["attention"] = []
        for _ in range(2):
            conv = torch.nn.Conv3d(2, K, 3, padding=1).cuda().requires_grad_(train)
            with torch.no_grad():
                for p in conv.parameters():
                    p.copy_((torch.rand(p.shape, generator=g, device="cuda") * 2 - 1) / math.sqrt(54))
            s["attention"].append(conv)
        if train:
            s["grads"] = [_randn(g, B, (2 + K) * 4, W, H, W), _randn(g, B, (2 + K) * 4, H, H, W)]
    else:
        # a smooth flow of some pixels on top of the pixel grid, and the aggregated volumes (one channel)
        flow = torch.nn.functional.interpolate(4 * _randn(g, B, 2, max(2, H // 8), max(2, W // 8)), (H, W), mode="bilinear",
                                               align_corners=True)
        y, x = torch.meshgrid(torch.arange(H, device="cuda"), torch.arange(W, device="cuda"), indexing="ij")
        s["coords"] = torch.stack((x, y)).float()[None] + flow
        s["fmap1"], s["fmap2"] = fmap1.requires_grad_(train), fmap2.requires_grad_(train)
        s["corr1"] = _randn(g, B, 1, W, H, W).requires_grad_(train)
        s["corr2"] = _randn(g, B, 1, H, H, W).requires_grad_(train)
        if train:
            s["grads"] = [_randn(g, B, 4 * (2 * RADIUS + 1) ** 2, H, W)]
            s["grads"] += [_randn(g, B, 4 * (2 * RADIUS + 1), H, W) for _ in range(2)]
        else:
            # a block outlives a pair's flow iterations: its features are laid out once
            s["block"] = AlternateCorrBlockSepflow(fmap1, fmap2, None, radius=RADIUS)
            s["block1d"] = CorrBlock1D(s["corr1"], s["corr2"], radius=RADIUS)
            with torch.no_grad():
                s["block"](s["coords"])
    return s


def run(s):
    kind = s["kind"]
    if not kind.endswith("train"):
        with torch.no_grad():
            if kind == "maxavg":
                return ComputeMaxAvgFunction.apply(s["f1"], s["f2"])
            if kind == "op":
                return (ComputeMaxAvgFunction.apply(s["f1"], s["f2"]),
                        ComputeSelfCompressionFunction.apply(s["f1"], s["f2"], s["a_u"], s["a_v"]))
            if kind == "separate":
                block = AlternateCorrBlockSepflow(s["fmap1"], s["fmap2"], None, radius=RADIUS)
                return block(None, sep=True, attention_weights=s["attention"])
            return s["block"](s["coords"]), s["block1d"](s["coords"])
    if kind in ("maxavg_train", "op_train"):
        leaves = [s["f1"], s["f2"]]
        out = ComputeMaxArgmaxAvgFunction.apply(s["f1"], s["f2"])
        if kind == "op_train":
            leaves += [s["a_u"], s["a_v"]]
            out = out + ComputeSelfCompressionFunction.apply(s["f1"], s["f2"], s["a_u"], s["a_v"])
    elif kind == "separate_train":
        # (the biases shift whole rows of a softmax: their gradients are zero but for rounding)
        leaves = [s["fmap1"], s["fmap2"]] + [m.weight for m in s["attention"]]
        block = AlternateCorrBlockSepflow(s["fmap1"], s["fmap2"], None, radius=RADIUS, support_backward=True)
        out = block(None, sep=True, attention_weights=s["attention"])
    else:
        leaves = [s["fmap1"], s["fmap2"], s["corr1"], s["corr2"]]
        block = AlternateCorrBlockSepflow(s["fmap1"], s["fmap2"], None, radius=RADIUS, support_backward=True)
        block1d = CorrBlock1D(s["corr1"], s["corr2"], radius=RADIUS)
        out = (block(s["coords"]),) + block1d(s["coords"])
    return [t.detach() for t in out], torch.autograd.grad(out, leaves, s["grads"])


def work(case):
    """Bytes: every input read once, every output written once.  Flops: the contractions of the definition (one is
    2 B N1 N2 C); the gradient of a maximum or average is a sum of selected rows or line means instead."""
    kind, B, H, W, C = case["kind"], case["B"], case["H"], case["W"], case["C"]
    K = case.get("K", 0)
    n = H * W
    feat, lines = B * n * C, B * n * (H + W)      # one feature map; one channel of both separated outputs together
    if kind.startswith("lookup"):
        win = 4 * ((2 * RADIUS + 1) ** 2 + 2 * (2 * RADIUS + 1)) * B * n
        floats = 2 * feat * (1 if kind == "lookup" else 2) + lines * (1 if kind == "lookup" else 2) + win
        flops = 4 * (2 * RADIUS + 2) ** 2 * 2 * B * n * C
        if kind == "lookup_train":
            floats, flops = floats + win, flops * 3
        return {"bytes": 4 * floats, "flops": flops}
    if kind.startswith("separate"):
        contraction = sum(2 * B * n * (H >> l) * (W >> l) * C for l in range(4))
        volume = 4 * (2 + K) * lines
        if kind == "separate":
            return {"bytes": 4 * (2 * feat + volume), "flops": 2 * contraction}
        return {"bytes": 4 * (4 * feat + 2 * volume), "flops": 5 * contraction}
    contraction = 2 * B * n * n * C
    floats = 2 * feat + 2 * lines
    flops = contraction
    if K:
        floats, flops = floats + 2 * K * lines, flops + contraction
    if kind.endswith("train"):
        floats += 2 * feat + (2 + 2 * K) * lines
        flops += 2 * 2 * lines * C * 2 + (3 * contraction if K else 0)
    return {"bytes": 4 * floats, "flops": flops}


def tolerance(case):
    """Sums of C products in 32 bits and, for gradients, of thousands of them: in another order they differ by 3e-7 to
    4e-7, single values by 6e-6.  Where the maximum over a line has two candidates that agree to the last bits of those
    sums, either one is right, and the gradient of that maximum goes to one feature row or the other: a few rows of a
    training step's feature gradients differ by whole terms (up to 2e-3 in all, single values by up to 0.5)."""
    if case["kind"] in ("maxavg_train", "op_train", "separate_train"):
        return {"rel": 8e-3, "max": 0.98}
    return {"rel": 2e-6, "max": 3e-5}


def exact(case, seed):
    """The outputs in 64 bits by plain torch: the volume of every image-1 row block formed whole, reduced and let go.
    None stands where the definition leaves a choice (the gradient of a maximum with two candidates that agree to the
    last bits goes to either) and for the lookups, whose gathers no dense form gives in reasonable time."""
    kind = case["kind"]
    if kind.startswith("lookup"):
        return None
    s = prepare(case, seed)
    train = kind.endswith("train")
    with torch.no_grad():
        if kind.startswith("separate"):
            outs = _exact_separate(s)
            return [outs, [None] * 4] if train else tuple(outs)
        f1, f2 = s["f1"].double(), s["f2"].double()
        outs = _exact_max_avg(f1, f2)
        if kind.startswith("maxavg"):
            return [outs, [None] * 2] if train else tuple(outs)
        comp = _exact_weighted(f1, f2, s["a_u"].double(), s["a_v"].double())
        if not train:
            return tuple(outs), tuple(comp)
        # (d_a_u = sum_u S g_cu and d_a_v = sum_v S g_cv: the same sums with the gradients as weights)
        d_v, d_u = _exact_weighted(f1, f2, s["grads"][3].double(), s["grads"][2].double())
        return [outs + comp, [None, None, d_u, d_v]]


def _volume_blocks(f1, f2):
    """(batch entry, image-1 rows, their volume (rows, W1, H2, W2)), at most about 2^27 entries at a time."""
    B, H1, W1, C = f1.shape
    _, H2, W2, _ = f2.shape
    rows = max(1, 2 ** 27 // (W1 * H2 * W2))
    for b in range(B):
        flat = f2[b].reshape(H2 * W2, C).t().contiguous()
        for i in range(0, H1, rows):
            part = f1[b, i:i + rows]
            yield b, slice(i, i + rows), (part.reshape(-1, C) @ flat).view(part.shape[0], W1, H2, W2)


def _exact_max_avg(f1, f2):
    B, H1, W1, _ = f1.shape
    out_u, out_v = f1.new_empty(B, H1, W1, 2, f2.shape[1]), f1.new_empty(B, H1, W1, 2, f2.shape[2])
    for b, rows, vol in _volume_blocks(f1, f2):
        out_u[b, rows] = torch.stack((vol.amax(3), vol.mean(3)), 2)
        out_v[b, rows] = torch.stack((vol.amax(2), vol.mean(2)), 2)
    return [out_u, out_v]


def _exact_weighted(f1, f2, over_v, over_u):
    """sum_v S over_v[k, v] and sum_u S over_u[k, u] for every image-1 pixel and channel k."""
    B, H1, W1, K, _ = over_v.shape
    out_u, out_v = f1.new_empty(B, H1, W1, K, f2.shape[1]), f1.new_empty(B, H1, W1, K, f2.shape[2])
    for b, rows, vol in _volume_blocks(f1, f2):
        for k in range(K):
            out_u[b, rows, :, k] = (vol * over_v[b, rows, :, k, None, :]).sum(3)
            out_v[b, rows, :, k] = (vol * over_u[b, rows, :, k, :, None]).sum(2)
    return [out_u, out_v]


def _exact_attention(conv, sep):
    """softmax over the displacement axis of the 3x3x3 convolution of sep (B,H1,W1,2,L): (B,H1,W1,K,L)."""
    x = torch.nn.functional.pad(sep.permute(0, 3, 4, 1, 2), (1,) * 6)
    w, bias = conv.weight.double(), conv.bias.double()
    L, H, W = x.shape[2] - 2, x.shape[3] - 2, x.shape[4] - 2
    z = bias.view(1, -1, 1, 1, 1).expand(x.shape[0], -1, L, H, W).clone()
    for d in range(27):
        t, i, j = d // 9, d // 3 % 3, d % 3
        for c in range(2):
            z += w[:, c, t, i, j].view(1, -1, 1, 1, 1) * x[:, c:c + 1, t:t + L, i:i + H, j:j + W]
    return z.softmax(2).permute(0, 3, 4, 1, 2).contiguous()


def _exact_separate(s):
    f1 = s["fmap1"].double().permute(0, 2, 3, 1).contiguous() / math.sqrt(s["fmap1"].shape[1])
    fmap2 = s["fmap2"].double()
    H, W = fmap2.shape[2:]
    levels = []
    for _ in range(4):
        f2 = fmap2.permute(0, 2, 3, 1).contiguous()
        sep = _exact_max_avg(f1, f2)
        over_v, over_u = (_exact_attention(conv, x) for conv, x in zip(s["attention"], sep[::-1]))
        comp = _exact_weighted(f1, f2, over_v, over_u)
        level = []
        for x, c, L in zip(sep[::-1], comp[::-1], (W, H)):
            v = torch.cat((x, c), 3).permute(0, 3, 4, 1, 2)
            level.append(torch.nn.functional.interpolate(v, (L, H, W), mode="trilinear", align_corners=True))
        levels.append(level)
        fmap2 = torch.nn.functional.avg_pool2d(fmap2, 2, 2)
    return [torch.cat([l[i] for l in levels], 1) for i in range(2)]
