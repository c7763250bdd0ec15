"""What this framework is used for, as cases that can be timed.

A case is a plain dictionary; its ``kind`` names the call:

* ``layer``   one submanifold 3x3x3 convolution over a kept kernel map, with bias and ReLU fused (what a folded
              convolution + norm + activation of an inference network is);
* ``updown``  a 2x2x2 stride-2 convolution and the transposed one back over the same kept map;
* ``maps``    the nine kernel maps of a four-level U-Net on a new cloud;
* ``points``  raw points of one or several scans -> voxels -> one collated batch;
* ``net``     inference of the sparse residual U-Net on a new cloud (its maps are built in the pass);
* ``train``   one training step of that network (forward, cross-entropy, backward, SGD with momentum) on a new cloud.

``cloud`` / ``size`` / ``batch`` describe the coordinates: ``lidar`` is the 64-ring scan of ``synth.lidar_cloud`` (size =
azimuth steps), ``surface`` the sphere and plane of ``synth.sphere_plane_cloud`` (size = points on the sphere), ``rooms``
the indoor scenes of ``synth.indoor_batch`` (size = points on the walls of a room), ``dense`` a random cloud (size =
points thrown into a cube of 2.17 times as many cells, the filling of a decoder's deep levels; single layers only).
"""
import functools
import math

import numpy as np
import torch

import pcengine_amd as pe
from pcengine_amd import nets, synth
from pcengine_amd.spconv import prebuild_maps
from pcengine_amd.utils import sparse_collate, sparse_quantize

DEVICE = "cuda:0"
DTYPES = {"f16": torch.float16, "f32": torch.float32}
BASE = dict(stem=32, enc=(32, 64, 128, 256), dec=(256, 128, 96, 96))
WIDE = dict(stem=64, enc=(64, 128, 256, 512), dec=(512, 256, 192, 192))
CLASSES = 20
LEARNING_RATE, MOMENTUM = 0.1, 0.9
LOSS_SCALE = 8192.0      # static loss scale of the fp16 training step: the mean over 10^5 rows is below fp16's range


def listed():
    return [
        # a small object scan through a narrow fp32 layer: the smallest call, launch and host time count
        dict(name="layer_surface_f32_c16", kind="layer", cloud="surface", size=21000, batch=1, dtype="f32", c_in=16, c_out=16),
        # the first level of a driving network: one scan, 150k voxels, few neighbours per voxel
        dict(name="layer_lidar_f16_c64", kind="layer", cloud="lidar", size=2048, batch=1, dtype="f16", c_in=64, c_out=64),
        # the same layer on a batch of eight scans: 1.2M voxels, more than the last-level cache holds
        dict(name="layer_lidar8_f16_c64", kind="layer", cloud="lidar", size=2048, batch=8, dtype="f16", c_in=64, c_out=64),
        # a deep layer of a decoder: wide rows, nine neighbours per voxel, matrix-core work
        dict(name="layer_dense_f16_c256", kind="layer", cloud="dense", size=90000, batch=1, dtype="f16", c_in=256, c_out=256),
        # one resolution step of the encoder and its inverse in the decoder
        dict(name="updown_lidar_f16_64_128", kind="updown", cloud="lidar", size=2048, batch=1, dtype="f16", c_in=64, c_out=128),
        # the maps of a network on a scan that was just received
        dict(name="maps_lidar", kind="maps", cloud="lidar", size=1344, batch=1),
        # the front end: four raw scans to one batch of voxels
        dict(name="points_lidar4", kind="points", cloud="lidar", size=2048, batch=4, dtype="f32", voxel=0.1),
        # interactive inference on a small object scan: latency
        dict(name="net_surface_f16", kind="net", cloud="surface", size=21000, batch=1, dtype="f16", wide=False),
        # inference on one driving scan, 100k voxels
        dict(name="net_lidar_f16", kind="net", cloud="lidar", size=1344, batch=1, dtype="f16", wide=False),
        # offline segmentation of eight indoor scenes with the wide network, 954k voxels: the largest
        dict(name="net_rooms8_f16_wide", kind="net", cloud="rooms", size=120000, batch=8, dtype="f16", wide=True),
        # a training step in mixed precision (fp16 features, fp32 parameters) on one driving scan
        dict(name="train_lidar_f16", kind="train", cloud="lidar", size=1344, batch=1, dtype="f16", wide=False),
        # a training step in full precision on a small object scan
        dict(name="train_surface_f32", kind="train", cloud="surface", size=21000, batch=1, dtype="f32", wide=False),
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread evenly over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_cloud(rng, most, kinds=("lidar", "lidar", "surface", "rooms")):
    """A cloud of roughly 2 000 to `most` voxels."""
    cloud = rng.choice(kinds)
    n = _log(rng, 2000, most)
    if cloud == "lidar":              # about 74 voxels per azimuth step and scan
        batch = rng.randint(1, max(1, min(8, n // 20000)))
        return dict(cloud=cloud, size=max(24, n // (74 * batch)), batch=batch)
    if cloud == "rooms":              # about 120 000 voxels in a fully sampled room
        batch = rng.randint(1, max(1, min(8, n // 20000)))
        return dict(cloud=cloud, size=max(1000, min(120000, n // batch)), batch=batch)
    return dict(cloud=cloud, size=min(n, 110000), batch=1)


def draw(rng):
    kind = rng.choice(("layer", "layer", "layer", "layer", "updown", "maps", "points", "net", "net", "train"))
    dtype = rng.choice(("f16", "f16", "f16", "f32"))
    if kind == "points":
        return dict(kind=kind, cloud="lidar", size=_log(rng, 64, 2048), batch=rng.randint(1, 8), dtype=rng.choice(("f32", "f64")),
                    voxel=rng.choice((0.05, 0.1, 0.2)))
    if kind == "maps":
        return dict(kind=kind, **_draw_cloud(rng, 1000000))
    if kind == "net":
        wide = rng.random() < 0.3
        return dict(kind=kind, **_draw_cloud(rng, (400000 if wide else 1000000) if dtype == "f16" else 40000), dtype=dtype, wide=wide)
    if kind == "train":
        return dict(kind=kind, **_draw_cloud(rng, 100000 if dtype == "f16" else 20000), dtype=dtype, wide=False)
    widths = (16, 32, 48, 64, 80, 96, 128, 160, 192, 256, 384)
    c_in, c_out = rng.choice(widths), rng.choice(widths)
    if rng.random() < 0.5:            # most layers of a network keep their width
        c_out = c_in
    most = 1000000 if c_in * c_out <= 64 * 128 else 300000 if c_in * c_out <= 192 * 192 else 100000
    return dict(kind=kind, **_draw_cloud(rng, most if dtype == "f16" else most // 4, ("lidar", "lidar", "surface", "rooms", "dense")),
                dtype=dtype, c_in=c_in, c_out=c_out)


# ---- inputs -----------------------------------------------------------------------------------------------------

@functools.lru_cache(maxsize=4)
def _scenes(cloud, size, batch, voxel):
    """The scenes of a batch as int64 [N, 3] voxel coordinates."""
    if cloud == "lidar":
        return [synth.lidar_cloud(seed=2 + b, azimuths=size, n_ground=size * 10, voxel=voxel)[:, 1:] for b in range(batch)]
    if cloud == "rooms":
        c = synth.indoor_batch(scenes=batch, n_room=size, n_box=max(20, size // 48))
        return [c[c[:, 0] == b, 1:] for b in range(batch)]
    if cloud == "surface":
        return [synth.sphere_plane_cloud(n_sphere=size, n_plane=size // 3)[:, 1:]]
    return [synth.random_cloud(seed=7, n=size, extent=round((2.17 * size) ** (1 / 3)))[:, 1:]]


def _placed(case, rng):
    """The case's scenes, each seen from another side and at another place: x and y exchanged or mirrored, shifted by
    multiples of 16 voxels.  The rows, and the voxels of every level of a network, stay as many whatever the seed.
    Returns the scenes and the bound of their coordinates."""
    scenes = _scenes(case["cloud"], case["size"], case["batch"], case.get("voxel", 0.1))
    top = np.max([c.max(axis=0) for c in scenes], axis=0)
    side, height = (int(-(-(v + 1) // 16) * 16) for v in (max(top[0], top[1]), top[2]))
    out = []
    for c in scenes:
        xy = c[:, :2]
        if rng.integers(2):
            xy = xy[:, ::-1]
        xy = np.where(rng.integers(2, size=2), side - 1 - xy, xy) + 16 * rng.integers(4, size=2)
        out.append(np.concatenate([xy, c[:, 2:]], axis=1))
    return out, [side + 47, side + 47, height - 1]


def _coords(case, seed):
    """int32 [N, 4] voxel coordinates of the case, sorted by (batch, x, y, z) as the front end leaves them, and the
    bound of the three last columns."""
    scenes, cmax = _placed(case, np.random.default_rng(seed))
    rows = []
    for b, c in enumerate(scenes):
        c = c[np.argsort((c[:, 0] * 4096 + c[:, 1]) * 4096 + c[:, 2])]
        rows.append(np.concatenate([np.full((len(c), 1), b), c], axis=1))
    return np.concatenate(rows, axis=0).astype(np.int32), cmax


def _points(case, seed):
    """Raw points of every scan: one in each of its voxels, and a second one in a seventh of them, in random order (the
    share of points that fall into a voxel with another one in a 64-ring scan at 0.1 m)."""
    rng = np.random.default_rng(seed)
    out = []
    for c in _placed(case, rng)[0]:
        c = np.concatenate([c, c[rng.permutation(len(c))[:len(c) // 7]]], axis=0)
        out.append((rng.permutation(c) + rng.uniform(0.02, 0.98, size=c.shape)) * case["voxel"])
    return out


def _network(case, gen):
    """The U-Net with random kernels scaled so that features stay near one, and norms as after training."""
    model = nets.SparseResUNet(4, CLASSES, **(WIDE if case["wide"] else BASE)).to(DEVICE)
    with torch.no_grad():
        for m in model.modules():
            if isinstance(m, pe.conv3d):
                fan = m.in_channels * {27: 8, 8: 2, 1: 1}[m.kernel_volume]
                m.kernel.normal_(generator=gen).mul_(fan ** -0.5)
                if m.bias is not None:
                    m.bias.normal_(generator=gen).mul_(0.1)
            elif isinstance(m, pe.BatchNorm):
                m.weight.uniform_(0.8, 1.2, generator=gen)
                m.bias.normal_(generator=gen).mul_(0.1)
                m.running_mean.normal_(generator=gen).mul_(0.1)
                m.running_var.uniform_(0.5, 1.5, generator=gen)
    return model


def _in_one(tensors):
    """Moves the tensors into one buffer, each on a 256-byte boundary, and returns it: the flat form in which a program
    broadcasts, checkpoints or averages its weights."""
    sizes = [-(-t.numel() // 64) * 64 for t in tensors]
    flat = torch.zeros(sum(sizes), device=DEVICE)
    for t, piece in zip(tensors, flat.split(sizes)):
        t.data = piece[:t.numel()].copy_(t.detach().reshape(-1)).view(t.shape)
    return flat


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    state = dict(case=case)
    if case["kind"] == "points":
        dtype = torch.float64 if case["dtype"] == "f64" else torch.float32
        clouds = _points(case, seed)
        state["points"] = [torch.as_tensor(c, dtype=dtype, device=DEVICE) for c in clouds]
        state["values"] = [torch.rand((len(c), 4), generator=gen, device=DEVICE) for c in clouds]
        return state
    coords, state["cmax"] = _coords(case, seed)
    state["coords"] = torch.as_tensor(coords, device=DEVICE)
    n = len(coords)
    if case["kind"] == "maps":
        state["feats"] = torch.zeros((n, 1), device=DEVICE)
        return state
    dtype = DTYPES[case["dtype"]]
    if case["kind"] in ("layer", "updown"):
        c_in, c_out = case["c_in"], case["c_out"]
        down = case["kind"] == "updown"
        pairs = 2 if down else 8
        layers = [pe.conv3d(c_in, c_out, 2 if down else 3, 2 if down else 1, bias=True)]
        if down:
            layers.append(pe.conv3d(c_out, c_in, 2, 2, bias=True, transposed=True))
        for m in layers:
            m.to(DEVICE)
            with torch.no_grad():
                m.kernel.normal_(generator=gen).mul_((m.in_channels * pairs) ** -0.5)
                m.bias.normal_(generator=gen).mul_(0.1)
            m.to(dtype).eval()
        feats = torch.randn((n, c_in), generator=gen, device=DEVICE).to(dtype)
        x = pe.spTensor(feats, state["coords"], None, [0, 0, 0], state["cmax"], batchsize=case["batch"])
        prebuild_maps(x, [(2, 2, 0) if down else (3, 1, 0)])
        state.update(layers=layers, x=x)
        return state
    model = _network(case, gen)
    # the values of a point cloud: where the voxel is in the box, and an intensity
    bound = torch.tensor(state["cmax"], device=DEVICE) + 1
    place = state["coords"][:, 1:] / bound * 2 - 1
    state["feats"] = torch.cat([place, torch.randn((n, 1), generator=gen, device=DEVICE)], dim=1).to(dtype)
    if case["kind"] == "net":
        state["model"] = model.eval().fuse_bn().to(dtype).use_planner()
    else:
        state["model"] = model.train()
        state["weights"] = _in_one(list(model.parameters()))
        state["stats"] = _in_one([b for b in model.buffers() if b.is_floating_point()])
        # classes that lie in space as those of a scene do: bands of height and distance
        state["target"] = ((place[:, 2] * 5 + place[:, :2].norm(dim=1) * 2.5).floor().long() % CLASSES).contiguous()
        state["scale"] = LOSS_SCALE if dtype == torch.float16 else 1.0
        # the loss scale is taken out again by the learning rate
        state["optimizer"] = torch.optim.SGD(model.parameters(), lr=LEARNING_RATE / state["scale"], momentum=MOMENTUM)
    return state


# ---- one pass ---------------------------------------------------------------------------------------------------

UNET_MAPS = [(3, 1, 0)] + [(2, 2, 0), (3, 1, 0)] * 4


def _run_points(state):
    samples, inverse = [], []
    for pts, values in zip(state["points"], state["values"]):
        coords, first, inv = sparse_quantize(pts, state["case"]["voxel"], return_index=True, return_inverse=True)
        samples.append(pe.spTensor(values[first], coords))
        inverse.append(inv)
    batch = sparse_collate(samples)
    return dict(coords=batch.coords, feats=batch.feats, inverse=inverse, upper=torch.tensor(batch.coords_max))


def _run_maps(state):
    x = pe.spTensor(state["feats"], state["coords"], None, [0, 0, 0], state["cmax"], batchsize=state["case"]["batch"])
    prebuild_maps(x, UNET_MAPS)
    out = []
    for km in x.kmaps.values():       # the six entries of a kernel map, and the coordinates of the level it leads to
        imap, omap, kpos, qkpos, qsum, _ = [km[i] for i in range(6)]
        out.append([imap, omap, kpos, qkpos, qsum, km.out_coords])
    return out


def _run_train(state):
    model = state["model"]
    model.zero_grad(set_to_none=True)
    x = pe.spTensor(state["feats"], state["coords"], None, [0, 0, 0], state["cmax"], batchsize=state["case"]["batch"])
    logits = model(x).feats.float()
    loss = torch.nn.functional.cross_entropy(logits, state["target"])
    (loss * state["scale"]).backward()
    state["optimizer"].step()
    return dict(loss=loss.detach(), logits=logits.detach(), weights=state["weights"], stats=state["stats"])


def run(state):
    kind = state["case"]["kind"]
    if kind == "points":
        return _run_points(state)
    if kind == "maps":
        return _run_maps(state)
    if kind == "train":
        return _run_train(state)
    with torch.no_grad():
        if kind == "layer":
            return state["layers"][0](state["x"], act="relu").feats
        if kind == "updown":
            down = state["layers"][0](state["x"], act="relu")
            return dict(down=down.feats, up=state["layers"][1](down, act="relu").feats)
        x = pe.spTensor(state["feats"], state["coords"], None, [0, 0, 0], state["cmax"], batchsize=state["case"]["batch"])
        return state["model"](x).feats


# ---- what a pass cannot do without --------------------------------------------------------------------------------

def _keys(c):
    c = c.long()
    return ((c[:, 0] * 4096 + c[:, 1]) * 4096 + c[:, 2]) * 4096 + c[:, 3]


def _pairs(coords):
    """Neighbour pairs of a submanifold 3x3x3 map, without the centre ones."""
    keys = _keys(coords + torch.tensor([0, 1, 1, 1], device=coords.device))
    total = 0
    for k in range(13):
        dx, dy, dz = k // 9 - 1, k // 3 % 3 - 1, k % 3 - 1
        want = keys + (dx * 4096 + dy) * 4096 + dz
        at = torch.searchsorted(keys, want).clamp_(max=len(keys) - 1)
        total += 2 * int((keys[at] == want).sum())
    return total


def _levels(case):
    """[(rows, pairs of the 3x3x3 map)] of the levels the case visits; every row has one pair to the level below."""
    c = torch.as_tensor(_coords(case, 0)[0], device=DEVICE if torch.cuda.is_available() else "cpu")
    out = [(len(c), _pairs(c))]
    for _ in range(4 if case["kind"] in ("maps", "net", "train") else case["kind"] == "updown"):
        c = torch.unique(torch.cat([c[:, :1], c[:, 1:] // 2], dim=1), dim=0)
        out.append((len(c), _pairs(c)))
    return out


def work(case):
    """Every array of a call read or written once, layer by layer for a network: rows in, rows out, a residual where a
    block has one, kernel, pair list (8 bytes a pair).  A multiply-accumulate counts as two operations."""
    kind = case["kind"]
    if kind == "points":
        size = 8 if case["dtype"] == "f64" else 4
        voxels = sum(len(c) for c in _scenes(case["cloud"], case["size"], case["batch"], case["voxel"]))
        points = voxels + voxels // 7
        return {"bytes": points * (3 * size + 8) + voxels * (16 + 2 * 16), "flops": 6 * points}
    levels = _levels(case)
    if kind == "maps":
        size = sum(16 * n for n, _ in levels) + sum(8 * m for _, m in levels) + sum(8 * n for n, _ in levels[:-1])
        return {"bytes": size, "flops": 27 * sum(n for n, _ in levels)}
    e = 2 if case["dtype"] == "f16" else 4
    total = [0, 0]

    def layer(n_in, n_out, pairs, kv, c_in, c_out, centre, residual=False):
        total[0] += e * (n_in * c_in + n_out * c_out * (2 if residual else 1) + kv * c_in * c_out) + 8 * pairs
        total[1] += 2 * (pairs + (n_out if centre else 0)) * c_in * c_out

    def block(n, m, c_in, c_out):
        if c_in != c_out:
            layer(n, n, 0, 1, c_in, c_out, True)
        layer(n, n, m, 27, c_in, c_out, True)
        layer(n, n, m, 27, c_out, c_out, True, True)

    if kind == "layer":
        layer(levels[0][0], levels[0][0], levels[0][1], 27, case["c_in"], case["c_out"], True)
    elif kind == "updown":
        n, n2 = levels[0][0], levels[1][0]
        layer(n, n2, n, 8, case["c_in"], case["c_out"], False)
        layer(n2, n, n, 8, case["c_out"], case["c_in"], False)
    else:
        w = WIDE if case["wide"] else BASE
        n, m = levels[0]
        layer(n, n, m, 27, 4, w["stem"], True)
        layer(n, n, m, 27, w["stem"], w["stem"], True)
        c, skips = w["stem"], [w["stem"]]
        for l, ce in enumerate(w["enc"]):
            layer(levels[l][0], levels[l + 1][0], levels[l][0], 8, c, c, False)
            block(*levels[l + 1], c, ce)
            block(*levels[l + 1], ce, ce)
            c = ce
            skips.append(c)
        skips.pop()
        for l, cd in zip((3, 2, 1, 0), w["dec"]):
            layer(levels[l + 1][0], levels[l][0], levels[l][0], 8, c, cd, False)
            block(*levels[l], cd + skips.pop(), cd)
            block(*levels[l], cd, cd)
            c = cd
        layer(n, n, 0, 1, c, CLASSES, True)
        maps = sum(16 * r + 8 * p for r, p in levels)
        total[0] += maps
        if kind == "train":           # the gradient of the rows and of the kernel: each as much as the forward layer
            total = [3 * total[0], 3 * total[1]]
    return {"bytes": total[0], "flops": total[1]}


def tolerance(case):
    """Four times what the calls show against themselves with every layer in another dataflow (other orders of summation,
    other roundings of partial sums) or in a wider type: layers 5e-4 in fp16 and 5e-7 in fp32, the fifty layers of a
    network 1.6e-3 and 2.5e-6, a training step 3.4e-3 and 5.5e-6 (its logits; its weights move less)."""
    kind = case["kind"]
    if kind in ("points", "maps"):
        return "exact"
    half = case["dtype"] == "f16"
    if kind in ("layer", "updown"):
        return {"rel": 2e-3, "max": 0.016} if half else {"rel": 2e-6, "max": 2.5e-5}
    if kind == "net":
        return {"rel": 6.5e-3, "max": 0.35} if half else {"rel": 1e-5, "max": 2e-4}
    return {"rel": 1.4e-2, "max": 0.4} if half else {"rel": 2.5e-5, "max": 3e-3}
