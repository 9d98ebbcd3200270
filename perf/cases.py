"""What a program that uses this framework has it do, as cases that can be timed and compared.

A case is a dict of plain values; its ``kind`` says what one pass is:

``step``    the voxel operators of one layer, forward and backward, on a ``ScatterData`` the
            program already holds (every layer of a voxel encoder after the first)
``centre``  the mean of the raw points of every voxel, forward only (cluster centres: few
            channels, no gradient), on a ``ScatterData`` the program already holds
``frame``   a frame from its points on: ``ScatterData.from_points`` and then one layer's
            forward and backward
``iter``    a training iteration that gets ``unq_inv`` / ``unq_cnts``: ``ScatterData(...)`` and
            then one layer's forward and backward
``ranks``   ``ingroup_inds``: the rank of every point inside its voxel
``pool``    ``dynamic_point_pool``: the points inside every box
``hash``    ``GridHash`` of a frame's voxel coordinates, probed with another frame's

The voxels (``keys``) are those of LiDAR-like sweeps (range density ~ 1/r^2 over 2-75 m) in
0.2 m cubes (``sweep``) or 0.2 m columns (``pillars``), of uniform points in 0.32 m columns
(``uniform``), of a Zipf(1.2) draw over few ids (``zipf``), or groups of a few to a few hundred
rows, delivered group by group (``groups``) or in any order (``clusters``).
"""
import math

import numpy as np
import torch

import torchex_amd as T

_DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
_BYTES = {"f32": 4, "f16": 2, "bf16": 2}
_RANGE = [-75.0, -75.0, -2.0, 75.0, 75.0, 4.0]   # metres; sweeps and uniform points lie inside
_CUBE = 0.2       # voxel edge of a sweep
_COLUMN = 0.32    # column edge of the uniform box


def listed():
    return [
        # points gathered per instance in a detector's second stage: a few thousand rows
        {"name": "small_step_f32", "kind": "step", "keys": "clusters", "points": 3000, "groups": 120,
         "channels": 128, "dtype": "f32", "ops": "sum,max"},
        # an encoder layer over a full sweep in fp32, the benchmark's own step
        {"name": "sweep_step_f32", "kind": "step", "keys": "sweep", "points": 1_000_000, "groups": 0,
         "channels": 128, "dtype": "f32", "ops": "mean,max"},
        # the same under mixed precision
        {"name": "sweep_step_f16", "kind": "step", "keys": "sweep", "points": 1_000_000, "groups": 0,
         "channels": 128, "dtype": "f16", "ops": "mean,max"},
        # columns over the full height: heavy-tailed occupancy
        {"name": "pillars_step_bf16", "kind": "step", "keys": "pillars", "points": 1_000_000, "groups": 0,
         "channels": 128, "dtype": "bf16", "ops": "mean,max"},
        # few voxels that own very many rows each
        {"name": "zipf_step_f32", "kind": "step", "keys": "zipf", "points": 2_000_000, "groups": 1024,
         "channels": 16, "dtype": "f32", "ops": "mean,max"},
        # features with the offset to the centre appended: a channel count that no vector divides
        {"name": "odd_step_f32", "kind": "step", "keys": "uniform", "points": 300_007, "groups": 0,
         "channels": 67, "dtype": "f32", "ops": "mean,max"},
        # voxel centres of a sweep
        {"name": "centre_f32", "kind": "centre", "keys": "sweep", "points": 1_000_000, "groups": 0,
         "channels": 3, "dtype": "f32", "ops": "mean"},
        # a frame of ordinary size from its points to the first layer's gradients
        {"name": "frame_bf16", "kind": "frame", "keys": "sweep", "points": 200_000, "groups": 0,
         "channels": 64, "dtype": "bf16", "ops": "mean,max"},
        # a batch of four sweeps, its index data prepared in the iteration
        {"name": "iter_4sweeps_f32", "kind": "iter", "keys": "sweep", "points": 4_000_000, "groups": 4,
         "channels": 32, "dtype": "f32", "ops": "mean,max"},
        # ranks of a sweep's points inside their voxels (to cap or pad voxels)
        {"name": "ranks_sweep", "kind": "ranks", "keys": "sweep", "points": 1_000_000, "groups": 0},
        # points of a frame inside a detector's proposals
        {"name": "pool_200boxes", "kind": "pool", "points": 200_000, "boxes": 200, "cap": 512},
        # voxel coordinates of one frame looked up in those of another
        {"name": "hash_frame", "kind": "hash", "points": 300_000, "probes": 300_000},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step"] * 6 + ["centre", "frame", "frame", "iter", "ranks", "pool", "hash"])
    if kind == "pool":
        return {"kind": kind, "points": _log_int(rng, 5_000, 300_000), "boxes": _log_int(rng, 3, 300),
                "cap": rng.choice([64, 128, 512])}
    if kind == "hash":
        return {"kind": kind, "points": _log_int(rng, 5_000, 500_000), "probes": _log_int(rng, 5_000, 1_000_000)}
    case = {"kind": kind, "groups": 0}
    if kind == "step":
        case["keys"] = rng.choice(["sweep", "pillars", "uniform", "zipf", "groups", "clusters"])
    elif kind == "frame":
        case["keys"] = rng.choice(["sweep", "pillars", "uniform"])
    elif kind == "ranks":
        case["keys"] = rng.choice(["sweep", "pillars", "clusters"])
    else:
        case["keys"] = rng.choice(["sweep", "pillars"])
    if kind == "ranks":
        case["points"] = _log_int(rng, 3_000, 2_000_000)
    else:
        case["dtype"] = rng.choice(["f32", "f16", "bf16"]) if kind != "centre" else "f32"
        case["channels"] = rng.choice([16, 32, 64, 128, 256, 10, 13, 35, 67, 131]) if kind != "centre" \
            else rng.choice([3, 4])
        if case["keys"] == "zipf":
            case["channels"] = rng.choice([13, 16, 32])
        most = min(4_000_000 if kind == "iter" else 2_000_000,
                   500_000_000 // (case["channels"] * _BYTES[case["dtype"]]))
        least = 20_000 if case["keys"] == "zipf" or kind in ("frame", "centre", "iter") else 1_000
        case["points"] = _log_int(rng, least, most)
        case["ops"] = "mean" if kind == "centre" else rng.choice(["mean,max", "mean,max", "sum,max"])
    if kind == "iter":
        case["groups"] = rng.randint(1, 4)
    elif case["keys"] == "zipf":
        case["groups"] = rng.choice([64, 300, 1024])
    elif case["keys"] in ("groups", "clusters"):
        case["groups"] = max(1, case["points"] // rng.choice([5, 25, 100, 400]))
    return case


# ------------------------------------------------------------------- inputs --

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _sweep_points(n, g):
    """[n, 3] points with range density ~ 1/r^2 on [2 m, 75 m], uniform azimuth and height."""
    u = torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
    r = 1.0 / (0.5 - u * (0.5 - 1.0 / 75.0))
    th = torch.rand(n, generator=g, device="cuda", dtype=torch.float64) * (2.0 * math.pi)
    z = torch.rand(n, generator=g, device="cuda", dtype=torch.float64) * 5.99 - 1.995
    return torch.stack([(r * torch.cos(th)).clamp(-74.99, 74.99), (r * torch.sin(th)).clamp(-74.99, 74.99), z],
                       dim=1).float()


def _uniform_points(n, g):
    p = torch.rand((n, 3), generator=g, device="cuda")
    p[:, :2] = p[:, :2] * 149.9 - 74.95
    p[:, 2] = p[:, 2] * 5.99 - 1.995
    return p


def _voxel_size(keys):
    return {"sweep": [_CUBE] * 3, "pillars": [_CUBE, _CUBE, 6.0], "uniform": [_COLUMN, _COLUMN, 6.0]}[keys]


def _cells(points, keys):
    """Linear voxel ids, x-major."""
    size = torch.tensor(_voxel_size(keys), device="cuda")
    lo = torch.tensor(_RANGE[:3], device="cuda")
    c = torch.div(points - lo, size, rounding_mode="floor").long()
    ny, nz = (int(math.ceil((_RANGE[3 + a] - _RANGE[a]) / _voxel_size(keys)[a] - 1e-6)) for a in (1, 2))
    return (c[:, 0] * ny + c[:, 1]) * nz + c[:, 2]


def _frame_points(keys, n, g, voxels):
    """Points of one frame that occupy ``voxels`` voxels whatever the seed: the few emptiest
    voxels beyond that many give their points to places where others lie."""
    p = _uniform_points(n, g) if keys == "uniform" else _sweep_points(n, g)
    _, inv, cnt = torch.unique(_cells(p, keys), return_inverse=True, return_counts=True)
    over = cnt.numel() - voxels
    if over > 0:
        order = torch.argsort(cnt + torch.rand(cnt.numel(), generator=g, device="cuda"))
        gone = torch.zeros(cnt.numel(), dtype=torch.bool, device="cuda")
        gone[order[:over]] = True
        gone = gone[inv]
        stay = p[~gone]
        p[gone] = stay[torch.randint(stay.shape[0], (int(gone.sum()),), generator=g, device="cuda")]
    return p


def _edges(weights):
    """Cumulative shares (on the host: the same to the last bit every time)."""
    return torch.from_numpy(np.cumsum(weights / weights.sum())).cuda()


def _ids(case, g):
    """(unq_inv, unq_cnts) as ``torch.unique`` returns them, rows in the order they arrive."""
    n, keys, groups = case["points"], case["keys"], case["groups"]
    if keys in ("sweep", "pillars", "uniform"):
        if case["kind"] == "iter":   # several sweeps, the sample's index folded into the voxel id
            parts = [_cells(_frame_points(keys, n // groups, g, _frame_voxels(keys, n // groups)), keys) +
                     b * (750 * 750 * 30) for b in range(groups)]
            k = torch.cat(parts)
        else:
            k = _cells(_frame_points(keys, n, g, _frame_voxels(keys, n)), keys)
    else:
        if keys == "zipf":
            w = np.arange(1, groups + 1, dtype=np.float64) ** -1.2
        else:   # group sizes between a tenth of the mean and twice the mean
            w = torch.rand(groups, generator=g, device="cuda", dtype=torch.float64).cpu().numpy() * 1.9 + 0.1
        k = torch.searchsorted(_edges(w), torch.rand(n, generator=g, device="cuda", dtype=torch.float64))
        k = k.clamp_(max=groups - 1)
        # no group is empty
        k[torch.randperm(n, generator=g, device="cuda")[:groups]] = torch.arange(groups, device="cuda")
        if keys == "groups":
            k = torch.sort(k)[0]
    _, inv, cnt = torch.unique(k, return_inverse=True, return_counts=True)
    return inv, cnt


def _rows(case):
    """Feature rows of a case (an ``iter`` case has a whole number of sweeps)."""
    n = case["points"]
    return n // case["groups"] * case["groups"] if case["kind"] == "iter" else n


def _inside(case):
    """Points inside every box of a ``pool`` case: few boxes hold many."""
    w = np.arange(1, case["boxes"] + 1, dtype=np.float64) ** -0.7
    return np.floor(0.15 * case["points"] * w / w.sum()).astype(np.int64)


def _boxes_and_points(case, g):
    """Boxes that do not touch, points inside them, and the rest of a sweep, whose points
    above or beside a box stay outside it."""
    b, n, inside = case["boxes"], case["points"], _inside(case)

    def u(*shape):
        return torch.rand(shape, generator=g, device="cuda")
    spot = torch.randperm(17 * 18, generator=g, device="cuda")[:b]
    rois = torch.zeros((b, 7), device="cuda")
    rois[:, 0] = (spot // 18 - 8).float() * 8.2 + u(b) - 0.5
    rois[:, 1] = (spot % 18 - 8.5).float() * 8.2 + u(b) - 0.5
    rois[:, 2] = u(b) - 1.5
    rois[:, 3:6] = u(b, 3) * torch.tensor([3.5, 3.5, 2.0], device="cuda") + 1.0
    rois[:, 6] = u(b) * 6.283
    rest = _sweep_points(n - int(inside.sum()), g)
    rest[:, 2] = rest[:, 2] * 0.1 + 3.5       # above every box
    box = rois[torch.from_numpy(np.repeat(np.arange(b), inside)).cuda()]
    m = box.shape[0]
    # a box's length lies along its heading turned by a quarter
    along, across = (u(m) - 0.5) * 0.98 * box[:, 4], (u(m) - 0.5) * 0.98 * box[:, 3]
    turn = box[:, 6] + 0.5 * math.pi
    mine = torch.stack([box[:, 0] + along * torch.cos(turn) + across * torch.sin(turn),
                        box[:, 1] - along * torch.sin(turn) + across * torch.cos(turn),
                        box[:, 2] + (u(m) * 0.98 + 0.01) * box[:, 5]], dim=1)
    pts = torch.cat([mine, rest])[torch.randperm(n, generator=g, device="cuda")]
    return rois, pts.contiguous()


def prepare(case, seed):
    g = _generator(seed)
    kind, n = case["kind"], case["points"]
    state = {"case": case}
    if kind == "pool":
        state["rois"], state["pts"] = _boxes_and_points(case, g)
        return state
    if kind == "hash":
        size, lo = torch.tensor([_CUBE] * 3, device="cuda"), torch.tensor(_RANGE[:3], device="cuda")

        def coors(count):
            return torch.div(_sweep_points(count, g) - lo, size, rounding_mode="floor").int()
        built = coors(n)
        state.update(coors=built, probes=torch.minimum(coors(case["probes"]), built.amax(0)))
        return state
    if kind == "ranks":
        state["inv"] = _ids(case, g)[0]
        return state
    dt, c, rows = _DTYPES[case["dtype"]], case["channels"], _rows(case)
    if kind == "centre":
        state["feats"] = torch.rand((n, c), generator=g, device="cuda") * 150.0 - 75.0
        state["data"] = T.ScatterData(*_ids(case, g))
        return state
    state["feats"] = torch.randn((rows, c), generator=g, device="cuda").to(dt).requires_grad_(True)
    if kind == "frame":
        xyz = _frame_points(case["keys"], n, g, _voxels(case))
        state["points"] = torch.cat([xyz, torch.rand((n, 1), generator=g, device="cuda")], dim=1)
    elif kind == "iter":
        state["inv"], state["cnt"] = _ids(case, g)
    else:
        state["data"] = T.ScatterData(*_ids(case, g))
    for op in case["ops"].split(","):   # the gradients that reach the layer's outputs
        state["g_" + op] = torch.randn((_voxels(case), c), generator=g, device="cuda").to(dt)
    return state


# ---------------------------------------------------------------- one pass --

def _layer(state, data, out):
    feats = state["feats"]
    for op in state["case"]["ops"].split(","):
        if op == "max":
            y, out["arg"] = T.scatter_max(feats, data)
        else:
            y = (T.scatter_mean if op == "mean" else T.scatter_sum)(feats, data)
        out[op] = y.detach()
        out["grad_" + op] = torch.autograd.grad(y, feats, state["g_" + op])[0]
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "step":
        return _layer(state, state["data"], {})
    if kind == "centre":
        return {"mean": T.scatter_mean(state["feats"], state["data"])}
    if kind == "frame":
        data = T.ScatterData.from_points(state["points"], _voxel_size(case["keys"]), _RANGE)
        return _layer(state, data, {"coors": data.coors, "inv": data.unq_inv, "counts": data.unq_cnts,
                                    "keys": data.unq_keys})
    if kind == "iter":
        data = T.ScatterData(state["inv"], state["cnt"])
        return _layer(state, data, {})
    if kind == "ranks":
        return T.ingroup_inds(state["inv"])
    if kind == "pool":
        idx, roi, feats = T.dynamic_point_pool(state["rois"], state["pts"], [0.5, 0.5, 0.2], case["cap"])
        return {"pts_idx": idx, "roi_idx": roi, "feats": feats}
    return T.GridHash(state["coors"]).probe(state["probes"])


# ------------------------------------------------------------ work, tolerance --

def _frame_voxels(keys, n):
    """Voxels that n points of one frame occupy: a little under the number to be expected."""
    if keys == "uniform":
        cells = math.ceil(150.0 / _COLUMN) ** 2
        u = cells * -math.expm1(-n / cells)
    else:
        nz = 30 if keys == "sweep" else 1
        r = np.linspace(2.0, 75.0, 20001)
        p = (_CUBE * _CUBE / nz) / (2.0 * math.pi * (0.5 - 1.0 / 75.0)) * r ** -3   # of one cell at range r
        per_ring = 2.0 * math.pi * r / (_CUBE * _CUBE) * nz * -np.expm1(-n * p)
        u = float(per_ring.sum() * (r[1] - r[0]))
    return int(0.99 * u - 3.0 * math.sqrt(u))


def _voxels(case):
    """Voxels of a case."""
    n, groups, keys = case["points"], case["groups"], case["keys"]
    if keys in ("groups", "clusters", "zipf"):
        return groups
    if case["kind"] == "iter":
        return groups * _frame_voxels(keys, n // groups)
    return _frame_voxels(keys, n)


def work(case):
    kind, n = case["kind"], case["points"]
    if kind == "ranks":
        return {"bytes": 16.0 * n, "flops": 0.0}                    # int64 ids in, int64 ranks out
    if kind == "pool":
        hits = int(np.minimum(_inside(case), case["cap"]).sum())    # two int64 and 13 floats each
        return {"bytes": 12.0 * n + 28.0 * case["boxes"] + 68.0 * hits, "flops": 0.0}
    if kind == "hash":
        # coordinates in, one (key, value) pair per voxel and one per probe, the answers
        return {"bytes": 12.0 * n + 8.0 * _frame_voxels("sweep", n) + (12.0 + 8.0 + 4.0) * case["probes"], "flops": 0.0}
    u = _voxels(case)
    e, c = _BYTES[case["dtype"]], case["channels"]
    rows, cells = float(n) * c, u * c
    total, flops = 0.0, 0.0
    for op in case["ops"].split(","):
        extra = 4 * cells if op == "max" else (8 * u if op == "mean" else 0)
        one = rows * e + 4 * n + cells * e + extra                  # either direction
        total += one if kind == "centre" else 2 * one
        flops += rows
    if kind == "frame":
        total += (16 + 12 + 4) * n + (4 + 8) * u                    # points; coordinates, ids; keys, counts
    if kind == "iter":
        total += 8 * n + 8 * u                                      # int64 ids, counts
    return {"bytes": total, "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if kind in ("ranks", "hash"):
        return "exact"
    if kind == "pool":
        return {"rel": 4e-7, "max": 4e-6}   # fp32 coordinates turned into a box's frame
    # four times what sums and means differ by from the same in 64 bits (measured: rel 1.0e-7 /
    # 2e-4 / 1.6e-3 and max 7e-7 / 4.9e-4 / 3.9e-3); ids, counts and arg are exact
    return {"f32": {"rel": 4e-7, "max": 3e-6}, "f16": {"rel": 8e-4, "max": 2e-3},
            "bf16": {"rel": 6.5e-3, "max": 1.6e-2}}[case["dtype"]]
