"""The work this framework is timed on: networks and single layers called through the public modules.

A case is a dict of plain values.  listed() gives the fixed ones, draw(rng) another one of the same ranges, prepare(case,
seed) what a program holds before the call, run(state) one pass and work(case) what that pass cannot do without.

Inputs are synthetic scenes: one-voxel-thick room surfaces (a floor, walls, boxes) for the 3-D networks and layers, sphere
shells and planes for the single-layer batch, pen strokes for the 2-D network.  Points come in shuffled order, as a
voxelised point cloud does, and where the input layer merges points a share of them repeats a site."""
import math

import numpy as np
import torch

import sparseconvnet_amd as scn
from sparseconvnet_amd import synthetic

CLASSES = 20
SPATIAL = 4096


def listed():
    return [
        # One layer on a new scene: input layer, its rulebook, SubmanifoldConvolution 3^3, output layer.  Two objects of a
        # thousand voxels: nothing but latency, launches and the host.
        {"name": "single_2x1k", "kind": "single", "sites": 1000, "batch": 2, "n_in": 16, "n_out": 16},
        # The same on two samples of 40 000 voxels in 128^3, the size a dense 3-D network would still take.
        {"name": "single_2x40k", "kind": "single", "sites": 40000, "batch": 2, "n_in": 16, "n_out": 16},
        # Handwriting recognition: a 2-D network over a batch of pen strokes, one batch after the other.
        {"name": "vgg2d_eval_100", "kind": "vgg2d", "batch": 100, "train": False},
        # Its training step: forward with batch statistics, loss, backward.
        {"name": "vgg2d_train_100", "kind": "vgg2d", "batch": 100, "train": True},
        # The layers of a wide network at scene scale, one after the other on one level whose rulebook exists: from the
        # first layer's three channels to 256.
        {"name": "layers_1m", "kind": "layers", "sites": 1000000, "pairs": "3x32,32x32,64x64,128x128,256x256", "bf16": False,
         "train": False},
        # Wide layers with bf16 operands, at a size that is no multiple of anything.
        {"name": "layers_bf16_300k", "kind": "layers", "sites": 300007, "pairs": "32x64,64x64,128x128", "bf16": True,
         "train": False},
        # Two levels down and up again on a new scene: strided convolution, then transposed convolution and batch norm on one
        # branch, max pooling and two unpoolings on the other.
        {"name": "tree_1m", "kind": "tree", "sites": 1000000, "planes": 32},
        # Semantic segmentation of one small room by the small residual network, coordinates in host memory as a data
        # loader leaves them.
        {"name": "unet_20k", "kind": "unet", "sites": 20011, "batch": 1, "m": 16, "reps": 1, "levels": 7, "residual": True,
         "train": False, "bf16": False, "host": True},
        # Segmentation of a whole floor by the full-width network: 1.3 million points, a new scene each pass.
        {"name": "unet_1m", "kind": "unet", "sites": 1000000, "batch": 1, "m": 32, "reps": 2, "levels": 7, "residual": False,
         "train": False, "bf16": False, "host": False},
        # The same network serving a batch of four rooms with bf16 operands.
        {"name": "unet_bf16_4x200k", "kind": "unet", "sites": 200003, "batch": 4, "m": 32, "reps": 2, "levels": 7,
         "residual": False, "train": False, "bf16": True, "host": True},
        # Training step of the small residual network over a batch of eight crops.
        {"name": "unet_train_8x12k", "kind": "unet", "sites": 12345, "batch": 8, "m": 16, "reps": 1, "levels": 7,
         "residual": True, "train": True, "bf16": False, "host": True},
        # Training step of the full-width network on a scene of a million voxels.
        {"name": "unet_train_1m", "kind": "unet", "sites": 1000000, "batch": 1, "m": 32, "reps": 2, "levels": 7,
         "residual": False, "train": True, "bf16": False, "host": False},
    ]


def _between(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("single", "vgg2d", "layers", "tree", "unet", "unet", "unet"))
    if kind == "single":
        return {"kind": kind, "sites": _between(rng, 500, 40000), "batch": rng.randint(1, 4),
                "n_in": _between(rng, 1, 64), "n_out": _between(rng, 8, 64)}
    if kind == "vgg2d":
        return {"kind": kind, "batch": _between(rng, 8, 200), "train": rng.random() < 0.5}
    if kind == "layers":
        sites = _between(rng, 20000, 1000000)
        widths = [16, 32, 48, 64, 80, 96, 100, 128, 160, 192, 224, 256]
        pairs = ["%dx%d" % (rng.choice(widths), rng.choice(widths)) for _ in range(rng.randint(1, 2))]
        return {"kind": kind, "sites": sites, "pairs": ",".join(pairs), "bf16": rng.random() < 0.3, "train": rng.random() < 0.3}
    if kind == "tree":
        return {"kind": kind, "sites": _between(rng, 20000, 1000000), "planes": rng.choice((16, 20, 24, 32, 48, 64))}
    batch = rng.choice((1, 1, 2, 4, 8))
    train = rng.random() < 0.4
    return {"kind": kind, "sites": _between(rng, 5000, 1000000 // batch), "batch": batch, "m": rng.choice((8, 12, 16, 20, 24, 32)),
            "reps": rng.randint(1, 2), "levels": rng.randint(4, 7), "residual": rng.random() < 0.3 and not train, "train": train,
            "bf16": rng.random() < 0.25 and not train, "host": rng.random() < 0.5}


# ---- inputs ----------------------------------------------------------------------------------------------------------
def _room(sites, spatial, rng, gen):
    """Distinct voxels [sites, 3] of a room's surfaces on the GPU, shuffled: rectangles one voxel thick, sampled from the
    list of all their cells, scaled until there are enough."""
    n_boxes = max(4, min(50, sites // 4000))
    walls = rng.integers(2, 5)
    wall_h = rng.uniform(0.25, 0.4, walls)
    centre = rng.uniform(0.08, 0.92, (n_boxes, 2))
    extent = rng.uniform(0.03, 0.14, (n_boxes, 3)) * math.sqrt(50 / n_boxes)

    def rectangles(side):
        o, z0 = (spatial - side) // 2, max(1, (spatial - int(0.4 * side)) // 2)
        rects = [(2, z0, o, o, side, side)]  # axis it is normal to, position on it, corner and size on the other two
        for w in range(walls):
            rects.append((w % 2, o if w < 2 else o + side - 1, o, z0, side, max(2, int(wall_h[w] * side))))
        for b in range(n_boxes):
            s = np.maximum(2, (extent[b] * side).astype(np.int64))
            lo = [o + int(centre[b, 0] * side) - s[0] // 2, o + int(centre[b, 1] * side) - s[1] // 2, z0 + 1]
            for axis in range(3):
                u, v = [d for d in range(3) if d != axis]
                for pos in (lo[axis], lo[axis] + s[axis]):
                    rects.append((axis, pos, lo[u], lo[v], s[u] + 1, s[v] + 1))
        return torch.tensor(np.array(rects, dtype=np.int64)).cuda()

    side = max(8, int(math.sqrt(sites / 2.2)))
    while True:
        r = rectangles(side)
        area = r[:, 4] * r[:, 5]
        which = torch.repeat_interleave(torch.arange(len(r), device="cuda"), area)
        cell = torch.arange(len(which), device="cuda") - (area.cumsum(0) - area)[which]
        axis, pos, u0, v0, _, nv = r[which].unbind(1)
        u, v = u0 + cell // nv, v0 + cell % nv
        x = torch.where(axis == 0, pos, u)
        y = torch.where(axis == 1, pos, torch.where(axis == 0, u, v))
        z = torch.where(axis == 2, pos, v)
        key = ((x * spatial + y) * spatial + z)[(torch.stack((x, y, z)) >= 0).all(0) & (torch.stack((x, y, z)) < spatial).all(0)]
        key = torch.unique(key)
        if len(key) >= sites:
            break
        side = max(side + 1, int(side * math.sqrt(1.01 * sites / len(key))))
    key = key[:sites][torch.randperm(sites, device="cuda", generator=gen)]
    return torch.stack((key // (spatial * spatial), key // spatial % spatial, key % spatial), 1)


def _rooms(sites, batch, spatial, seed, repeated):
    """Coordinates [points, 4] of `batch` rooms on the GPU; `repeated` of the sites have a second point."""
    rng = np.random.default_rng([seed, 77])
    gen = torch.Generator(device="cuda").manual_seed(seed)
    out = []
    for b in range(batch):
        p = _room(sites, spatial, rng, gen)
        if repeated:
            p = torch.cat((p, p[:int(repeated * sites)]))
            p = p[torch.randperm(len(p), device="cuda", generator=gen)]
        out.append(torch.cat((p, torch.full((len(p), 1), b, device="cuda")), 1))
    return torch.cat(out), gen


def _statistics(model, gen):
    """Running statistics as training leaves them: of the size of the values, not 0 and 1."""
    for bn in model.modules():
        if isinstance(bn, scn.BatchNormalization):
            bn.running_mean.normal_(0, 0.1, generator=gen)
            bn.running_var.uniform_(0.5, 1.5, generator=gen)


def _vgg2d():
    return scn.Sequential().add(scn.SparseVggNet(2, 1, [['C', 8], ['C', 8], ['MP', 3, 2], ['C', 16], ['C', 16], ['MP', 3, 2],
                                                        ['C', 24], ['C', 24], ['MP', 3, 2]])).add(
        scn.SubmanifoldConvolution(2, 24, 32, 3, False)).add(scn.BatchNormReLU(32)).add(scn.SparseToDense(2, 32))


def prepare(case, seed):
    torch.manual_seed(seed)
    kind = case["kind"]
    s = {"kind": kind, "train": case.get("train", False), "bf16": case.get("bf16", False)}
    if kind == "single":
        spatial = max(16, min(128, int(0.64 * math.sqrt(case["sites"]))))
        coords = np.concatenate([synthetic.shells_and_planes(seed * 8 + b, spatial, case["sites"], b) for b in range(case["batch"])])
        s["coords"] = torch.as_tensor(coords).cuda()
        s["features"] = torch.randn((len(coords), case["n_in"]), device="cuda")
        s["input"] = scn.InputLayer(3, spatial, mode=4)
        s["model"] = scn.Sequential().add(scn.SubmanifoldConvolution(3, case["n_in"], case["n_out"], 3, False)).add(
            scn.OutputLayer(3)).cuda().eval()
    elif kind == "vgg2d":
        coords = synthetic.strokes2d(seed=seed * 1000, batch=case["batch"])
        s["coords"] = torch.as_tensor(coords).cuda()
        s["features"] = torch.ones((len(coords), 1), device="cuda")
        s["input"] = scn.InputLayer(2, 71, mode=3)
        s["model"] = _vgg2d().cuda().train(s["train"])
        s["linear"] = torch.nn.Linear(32 * 8 * 8, 183).cuda()  # as many classes as the characters of the reference's data set
        s["labels"] = torch.randint(183, (case["batch"],), device="cuda")
    elif kind == "layers":
        coords, gen = _rooms(case["sites"], 1, SPATIAL, seed, 0)
        pairs = [tuple(int(v) for v in p.split("x")) for p in case["pairs"].split(",")]
        level = scn.InputLayer(3, SPATIAL, mode=0)([coords, torch.zeros((len(coords), 1), device="cuda")])
        level.metadata.setBf16(s["bf16"])
        s["layers"] = []
        for n_in, n_out in pairs:
            x = torch.randn((len(coords), n_in), device="cuda", generator=gen)
            conv = scn.SubmanifoldConvolution(3, n_in, n_out, 3, False).cuda().train(s["train"])
            grad = torch.randn((len(coords), n_out), device="cuda", generator=gen) if s["train"] else None
            s["layers"].append((conv, scn.SparseConvNetTensor(x.requires_grad_(s["train"]), level.metadata, level.spatial_size), grad))
    elif kind == "tree":
        n = case["planes"]
        s["coords"], gen = _rooms(case["sites"], 1, 4094, seed, 0)
        s["features"] = torch.randn((case["sites"], n), device="cuda", generator=gen)
        s["input"] = scn.InputLayer(3, 4094, mode=0)
        s["down"] = scn.Convolution(3, n, 2 * n, 2, 2, False).cuda().eval()
        s["pool"] = scn.Sequential().add(scn.MaxPooling(3, 3, 2)).add(scn.UnPooling(3, 3, 2)).add(scn.UnPooling(3, 2, 2))
        s["model"] = scn.Sequential().add(scn.Deconvolution(3, 2 * n, n, 2, 2, False)).add(scn.BatchNormReLU(n)).cuda().eval()
    else:
        coords, gen = _rooms(case["sites"], case["batch"], SPATIAL, seed, 0.3)
        m = case["m"]
        s["features"] = torch.rand((len(coords), 3), device="cuda", generator=gen) * 2 - 1
        s["coords"] = coords.cpu() if case["host"] else coords
        s["input"] = scn.InputLayer(3, SPATIAL, mode=4)
        s["model"] = scn.Sequential().add(scn.SubmanifoldConvolution(3, 3, m, 3, False)).add(
            scn.UNet(3, case["reps"], [m * (i + 1) for i in range(case["levels"])], case["residual"])).add(
            scn.BatchNormReLU(m)).add(scn.OutputLayer(3)).cuda().train(s["train"])
        s["linear"] = torch.nn.Linear(m, CLASSES).cuda()
        s["labels"] = torch.randint(CLASSES, (len(coords),), device="cuda", generator=gen)
    if "model" in s and not s["train"]:
        _statistics(s["model"], torch.Generator(device="cuda").manual_seed(seed + 1))
    return s


# ---- one pass ---------------------------------------------------------------------------------------------------------
def _head(s, y):
    return s["linear"](y.flatten(1)) if "linear" in s else y


def _scene(s):
    x = s["input"]([s["coords"], s["features"]])
    if s["bf16"]:
        x.metadata.setBf16(True)
    return x


def _train(s):
    modules = (s["model"], s["linear"])
    for module in modules:
        module.zero_grad(set_to_none=True)
    y = _head(s, s["model"](_scene(s)))
    loss = torch.nn.functional.cross_entropy(y, s["labels"])
    loss.backward()
    return {"logits": y.detach(), "loss": loss.detach(),
            "gradients": torch.cat([p.grad.flatten() for module in modules for p in module.parameters()]),
            "statistics": torch.cat([b.flatten() for module in modules for b in module.buffers()])}


def _layers(s):
    if not s["train"]:
        with torch.no_grad():
            return [conv(x).features for conv, x, _ in s["layers"]]
    out = []
    for conv, x, grad in s["layers"]:
        x.features.grad = conv.weight.grad = None
        y = conv(x).features
        y.backward(grad)
        out += [y.detach(), x.features.grad, conv.weight.grad]
    return out


def run(s):
    if s["kind"] == "layers":
        return _layers(s)
    if s["train"]:
        return _train(s)
    with torch.no_grad():
        x = _scene(s)
        if s["kind"] != "tree":
            return _head(s, s["model"](x))
        h = s["down"](x)
        return [s["pool"](h).features, s["model"](h).features]


# ---- what a pass cannot do without --------------------------------------------------------------------------------------
#: Neighbours (itself included) of a voxel of the room surfaces in its 3^3 box, and the share of sites left per halving.
RULES, SHRINK = 10.8, 0.246


def _conv(rows_in, rows_out, rules, taps, n_in, n_out):
    """Bytes and operations of one convolution: rows in, weights and rows out once."""
    return np.array([4.0 * (rows_in * n_in + rows_out * n_out + taps * n_in * n_out), 2.0 * rules * n_in * n_out])


def _unet_work(case):
    sites, total = float(case["sites"] * case["batch"]), np.zeros(2)
    planes = [case["m"] * (i + 1) for i in range(case["levels"])]
    for i, p in enumerate(planes):
        n = sites * SHRINK ** i

        def subm(n_in):
            return _conv(n, n, RULES * n, 27, n_in, p)
        unit = 2 if case["residual"] else 1
        total += unit * case["reps"] * subm(p) + (subm(3) if i == 0 else 0)
        if i + 1 < len(planes):
            q, c = planes[i + 1], n * SHRINK
            total += _conv(n, c, n, 8, p, q) + _conv(c, n, n, 8, q, p)
            total += subm(2 * p) + (unit * case["reps"] - 1) * subm(p)
            if case["residual"]:
                total += _conv(n, n, n, 1, 2 * p, p)
    points = 1.3 * sites
    total += np.array([points * (32 + 12 + 4 * case["m"] + 4 * CLASSES), 2 * points * case["m"] * CLASSES])
    return total


def work(case):
    kind = case["kind"]
    if kind == "single":
        n = case["sites"] * case["batch"]
        w = _conv(n, n, 11.0 * n, 27, case["n_in"], case["n_out"]) + np.array([32.0 * n, 0])
    elif kind == "vgg2d":
        n, w = 165.0 * case["batch"], np.zeros(2)  # pixels of a sample; the pooled levels keep about 0.75 and 0.4 of them
        for rows, n_in, n_out in ((n, 1, 8), (n, 8, 8), (0.75 * n, 8, 16), (0.75 * n, 16, 16), (0.4 * n, 16, 24), (0.4 * n, 24, 24),
                                  (0.2 * n, 24, 32)):
            w += _conv(rows, rows, 4.0 * rows, 9, n_in, n_out)
        w += _conv(case["batch"], case["batch"], case["batch"], 1, 2048, 183)
    elif kind == "layers":
        n, w = case["sites"], np.zeros(2)
        for pair in case["pairs"].split(","):
            w += _conv(n, n, RULES * n, 27, *(int(v) for v in pair.split("x")))
    elif kind == "tree":
        n, p = case["sites"], case["planes"]
        c = SHRINK * n
        w = _conv(n, c, n, 8, p, 2 * p) + _conv(c, n, n, 8, 2 * p, p) + np.array([32.0 * n + 4.0 * 2 * p * (3 * c + 2 * SHRINK * c + n), 0])
    else:
        w = _unet_work(case)
    if case.get("train"):
        w = 3 * w  # the two gradients of every layer are as much again each
    return {"bytes": float(w[0]), "flops": float(w[1])}


def tolerance(case):
    """About four times what the same pass on the mirrored scene with mirrored filters (the same sums in another order) and, for
    the layers, the sums in 64 bits differ by: fp32 layers up to 1.0e-6 (1.6e-5 at one value), bf16 operands 2.4e-3.  Through
    a network's training step a value on the edge of a ReLU falls to one side or the other, so that its gradients differ by
    more than their sums do: 1.6e-3 (0.11) over a million sites, 4e-4 (0.04) over a hundred thousand."""
    if case.get("bf16"):
        return {"rel": 5e-3, "max": 0.06}
    if case.get("train") and case["kind"] != "layers":
        return {"rel": 6e-3, "max": 0.4} if case["kind"] == "unet" else {"rel": 2e-3, "max": 0.15}
    return {"rel": 4e-6, "max": 7e-5}
