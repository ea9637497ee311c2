"""Timed workloads of brook_amd, each through the package's public entry points.

A case is a dict of plain values; `listed()` names the fixed ones and `draw()` takes others of the
same ranges. The kinds and what they stand for:

  skeletonize     one label volume in, packed skeletons out: an interactive crop of a few objects, a
                  served request, a large block of a segmentation, a stack of thin supervoxels
  batch           many mixed-shape volumes in one `skeletonize_batch` call
  components      `device.connected_components` of a dense segmentation (every voxel labelled)
  edt             `device.edt` of a dense segmentation
  merge           `packed.merge_fragments` of the skeletons of overlapping chunks
  postprocess     `device_post.postprocess` of merged skeletons (dust, loops, joins, ticks)
"""
import math

import numpy as np
import torch

import brook_amd
from brook_amd import device, device_post, packed, synth

PARAMS = dict(scale=1.5, const=300, pdrf_scale=100000, pdrf_exponent=4)
DTYPES = {"uint8": np.uint8, "uint16": np.uint16, "uint32": np.uint32, "uint64": np.uint64}
# torch's integer types of the same width: the ids of a case stay below their signed limits
TENSOR = {"uint8": torch.uint8, "uint16": torch.int16, "uint32": torch.int32, "uint64": torch.int64}


def _volume(name, source, shape, labels, dtype="uint32", layout="device F", aniso="8 8 40", **options):
    return dict(name=name, kind="skeletonize", source=source, sx=shape[0], sy=shape[1], sz=shape[2], labels=labels,
                dtype=dtype, layout=layout, aniso=aniso, dust=options.pop("dust", 1000),
                fix_branching=options.pop("fix_branching", True), fill_holes=options.pop("fill_holes", False), **options)


def listed():
    return [
        # a proofreader's crop around a few objects: launches and host round trips
        _volume("crop_48", "tubes", (48, 41, 37), 3, "uint8", "device C", "16 16 40", dust=100),
        # the small reference workload, from host memory in numpy's own order
        _volume("host_tubes_128", "tubes", (128, 128, 128), 20, "uint32", "host C", "16 16 40"),
        # a served request: the middle of the serving stream's sizes, ragged
        _volume("request_317", "tubes", (317, 254, 391), 27, "uint32", "device F", "16 16 40"),
        # the headline workload: thick branching objects filling 40 % of the volume
        _volume("trees_512", "trees", (512, 512, 512), 200, "uint32", "device F", "8 8 40"),
        # the same objects traced by parent walks
        _volume("parents_300", "trees", (300, 256, 271), 45, "uint16", "device F", "8 8 40", fix_branching=False),
        # thousands of thin fragments with 64-bit ids in flat voxels
        _volume("cells_512", "cells", (512, 480, 250), 590, "uint64", "device F", "4 4 40"),
        # a noisy segmentation: single-voxel holes filled first
        _volume("holes_200", "trees", (200, 184, 168), 16, "uint32", "device F", "8 8 40", fill_holes=True),
        # a queue of small volumes in one call
        dict(name="batch_24", kind="batch", count=24, low=64, high=220, dtype="uint32"),
        # stages called on their own, on a dense segmentation
        dict(name="components_400", kind="components", sx=401, sy=512, sz=300, cell=23, dtype="uint32"),
        dict(name="edt_450", kind="edt", sx=450, sy=387, sz=256, cell=31, dtype="uint16", aniso="4 4 40", border=True),
        # chunked results put together, and the cleaning of what comes out
        dict(name="merge_8", kind="merge", labels=180, branches=14, length=90, fragments=8),
        dict(name="postprocess_150", kind="postprocess", labels=150, branches=14, length=90),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["crop", "tubes", "tubes", "trees", "trees", "cells", "batch", "components", "edt", "merge",
                       "postprocess"])
    if kind in ("crop", "tubes", "trees", "cells"):
        low, high = {"crop": (30, 90), "tubes": (90, 420), "trees": (90, 400), "cells": (120, 480)}[kind]
        shape = tuple(_log(rng, low, high) for _ in range(3))
        voxels = shape[0] * shape[1] * shape[2]
        if kind == "crop":
            labels, dtype, dust = rng.randint(1, 6), rng.choice(["uint8", "uint16"]), 100
        elif kind == "tubes":
            labels, dtype, dust = rng.randint(5, 50), rng.choice(["uint16", "uint32", "uint64"]), 1000
        elif kind == "trees":  # the voxels per object of the 512^3 workload
            labels, dtype, dust = max(2, voxels // 670000), rng.choice(["uint16", "uint32"]), 1000
        else:  # the voxels per cell of the 1024 x 1024 x 512 workload
            labels, dtype, dust = max(4, voxels // 105000), "uint64", 1000
        aniso = {"crop": "16 16 40", "tubes": "16 16 40", "trees": "8 8 40", "cells": "4 4 40"}[kind]
        c = _volume("", "tubes" if kind == "crop" else kind, shape, labels, dtype,
                    rng.choice(["device F", "device F", "device C", "host C", "host F"]), aniso, dust=dust,
                    fix_branching=rng.random() < 0.75, fill_holes=kind == "trees" and voxels < 8e6 and rng.random() < 0.5)
        del c["name"]
        return c
    if kind == "batch":
        return dict(kind="batch", count=rng.randint(4, 32), low=48, high=_log(rng, 120, 240),
                    dtype=rng.choice(["uint16", "uint32"]))
    if kind in ("components", "edt"):
        c = dict(kind=kind, sx=_log(rng, 60, 500), sy=_log(rng, 60, 500), sz=_log(rng, 40, 320), cell=rng.randint(9, 50),
                 dtype=rng.choice(["uint8", "uint16", "uint32", "uint64"]))
        if kind == "edt":
            c.update(aniso=rng.choice(["1 1 1", "4 4 40", "16 16 40"]), border=rng.random() < 0.5)
        return c
    c = dict(kind=kind, labels=_log(rng, 4, 250), branches=rng.randint(2, 16), length=_log(rng, 20, 140))
    if kind == "merge":
        c["fragments"] = rng.randint(2, 12)
    return c


# ---- inputs ------------------------------------------------------------------------------------

def _to_device(vol, dtype, order):
    """A device tensor of vol's shape with Fortran or C strides."""
    flat = torch.from_numpy(np.ravel(vol.astype(DTYPES[dtype], copy=False), order=order).view(
        {1: np.uint8, 2: np.int16, 4: np.int32, 8: np.int64}[np.dtype(DTYPES[dtype]).itemsize])).cuda()
    if order == "C":
        return flat.view(vol.shape)
    return flat.view(vol.shape[::-1]).permute(2, 1, 0)


def _labels(case, seed):
    shape = (case["sx"], case["sy"], case["sz"])
    if case["source"] == "cells":
        vol = synth.cells(shape, case["labels"], seed, _aniso(case))[0]
    else:
        vol = synth.volume(case["source"], shape, case["labels"], seed)
    if case["fill_holes"]:  # single voxels lost, mostly inside objects
        vol[np.random.default_rng(seed).random(vol.shape, np.float32) < 0.001] = 0
    return vol


def _dense(case, seed):
    """A dense segmentation on the GPU: Voronoi cells of jittered seeds, ids drawn with repeats so
    that a value can name several components, in Fortran order."""
    g = torch.Generator("cuda").manual_seed(seed)
    size = (case["sz"], case["sy"], case["sx"])
    pitch = case["cell"]
    grid = [s // pitch + 3 for s in size]  # one cell of margin on each side
    seeds = torch.rand((3, *grid), generator=g, device="cuda") * pitch
    top = 250 if case["dtype"] == "uint8" else 30000
    ids = torch.randint(1, top, grid, generator=g, device="cuda", dtype=torch.int32)
    out = torch.empty(size, dtype=TENSOR[case["dtype"]], device="cuda")
    y = torch.arange(size[1], device="cuda")[:, None]
    x = torch.arange(size[2], device="cuda")[None, :]
    cy, cx = y // pitch + 1, x // pitch + 1
    slab = 32
    for z0 in range(0, size[0], slab):
        z = torch.arange(z0, min(z0 + slab, size[0]), device="cuda")[:, None, None]
        cz = z // pitch + 1
        best = torch.full((z.shape[0], size[1], size[2]), float("inf"), device="cuda")
        label = torch.zeros(best.shape, dtype=torch.int32, device="cuda")
        for dz in (-1, 0, 1):
            for dy in (-1, 0, 1):
                for dx in (-1, 0, 1):
                    at = (cz + dz, cy + dy, cx + dx)
                    d = ((seeds[0][at] + (cz + dz - 1) * pitch - z).square() + (seeds[1][at] + (cy + dy - 1) * pitch - y).square()
                         + (seeds[2][at] + (cx + dx - 1) * pitch - x).square())
                    nearer = d < best
                    best = torch.where(nearer, d, best)
                    label = torch.where(nearer, ids[at], label)
        out[z0:z0 + slab] = label.to(out.dtype)
    return out.permute(2, 1, 0)


def _aniso(case):
    return tuple(float(a) for a in case["aniso"].split())


def _skeletons(case, seed):
    """Branching lattice skeletons as `skeletonize` gives them (vertices unique within a label): per
    label a tree of direction-keeping walks, each branch off an earlier vertex, some branches short
    (ticks), a few closed into loops, a few cut (pieces to join). Host PackedSkeletons."""
    rng = np.random.default_rng(seed)
    aniso = np.array((16.0, 16.0, 40.0), np.float32)
    labels, v_off, e_off, verts, edges, radii = [], [0], [0], [], [], []
    for label in range(1, case["labels"] + 1):
        points = [rng.integers(0, 2000, (1, 3))]
        links, count = [], 1
        for b in range(case["branches"]):
            n = int(rng.integers(3, 8)) if b and rng.random() < 0.3 else max(4, int(case["length"] * rng.uniform(0.4, 1.6)))
            heading = rng.normal(size=3)
            steps = np.clip(np.rint(1.1 * heading / np.abs(heading).max() + rng.uniform(-0.7, 0.7, (n, 3))), -1, 1).astype(np.int64)
            steps[~steps.any(1), 0] = 1
            start = int(rng.integers(0, count))
            whole = np.concatenate(points)
            points.append(whole[start] + np.cumsum(steps, 0))
            chain = np.concatenate([[start], np.arange(count, count + n)])
            links.append(np.stack([chain[:-1], chain[1:]], 1))
            if b and rng.random() < 0.1:  # the branch meets the tree again
                links.append([[count + n - 1, int(np.abs(whole - points[-1][-1]).sum(1).argmin())]])
            count += n
        p, e = np.concatenate(points), np.concatenate(links)
        _, first, where = np.unique(p, axis=0, return_index=True, return_inverse=True)
        p, e = p[first], where.reshape(-1)[e]
        e = np.sort(e[rng.random(len(e)) >= 0.004], 1)
        e = np.unique(e[e[:, 0] != e[:, 1]], axis=0)
        labels.append(label)
        v_off.append(v_off[-1] + len(p))
        e_off.append(e_off[-1] + len(e))
        verts.append(p.astype(np.float32) * aniso)
        edges.append(e.astype(np.uint32))
        radii.append(rng.uniform(16, 300, len(p)).astype(np.float32))
    return packed.PackedSkeletons(np.asarray(labels, np.int64), np.asarray(v_off, np.int64), np.asarray(e_off, np.int64),
                                  np.concatenate(verts), np.concatenate(edges), np.concatenate(radii),
                                  tuple(float(a) for a in aniso))


def _fragments(case, seed):
    """(parts, origins) on the host: every part holds each skeleton's vertices in a frame of its own and a run
    of its edges that overlaps the next part's, as chunks with a shared border give them."""
    whole, rng, k = _skeletons(case, seed), np.random.default_rng(seed + 1), case["fragments"]
    parts, origins = [], []
    for f in range(k):
        pieces = []
        for s in range(len(whole)):
            e = whole.edges[whole.e_off[s]:whole.e_off[s + 1]]
            lo, hi = len(e) * f // k, min(len(e), len(e) * (f + 1) // k + 5)
            pieces.append(e[lo:hi])
        origin = np.asarray(whole.anisotropy, np.float32) * rng.integers(0, 64, 3)
        parts.append(packed.PackedSkeletons(whole.labels, whole.v_off,
                                            np.concatenate([[0], np.cumsum([len(p) for p in pieces])]).astype(np.int64),
                                            whole.vertices - origin.astype(np.float32), np.concatenate(pieces), whole.radii,
                                            whole.anisotropy))
        origins.append(tuple(float(o) for o in origin))
    return parts, origins


def _batch_shapes(case):
    """Edges spread over the range, the same for every seed (their contents differ)."""
    rng = np.random.default_rng(case["count"] * 1000 + case["high"])
    return [tuple(int(round(math.exp(rng.uniform(math.log(case["low"]), math.log(case["high"]))))) for _ in range(3)) +
            (int(rng.integers(1, 31)),) for _ in range(case["count"])]


def _sizes(case):
    """Room for a result: skeletons, vertices, edges. More than the workloads of a case ever need."""
    if case["kind"] == "skeletonize":
        voxels, labels = case["sx"] * case["sy"] * case["sz"], case["labels"]
    elif case["kind"] == "batch":
        shapes = _batch_shapes(case)
        voxels, labels = sum(a * b * c for a, b, c, _ in shapes), sum(s[3] for s in shapes)
    else:
        top = int(case["labels"] * (2 + case["branches"] * (1.6 * case["length"] + 2)))
        return case["labels"], top, 2 * top
    top = labels * 1000 + voxels // 100
    return 8 * labels + 64, top, top


def _components_room(case):
    cells = 1.0
    for s in ("sx", "sy", "sz"):
        cells *= case[s] / case["cell"] + 3
    return int(3 * cells) + 64


class _Results:
    """The arrays a program keeps its results in, one set per input: what a pass gives is copied to
    their front, zeros follow."""

    def __init__(self, empty, **rooms):
        self.arrays = {k: empty(shape, dtype) for k, (shape, dtype) in rooms.items()}
        self.used = dict.fromkeys(rooms, 0)

    def take(self, **values):
        for k, v in values.items():
            n, a = len(v), self.arrays[k]
            if n > len(a):
                raise ValueError(f"{k}: {n} entries for {len(a)}")
            a[:n] = v
            if n < self.used[k]:
                a[n:self.used[k]] = 0
            self.used[k] = n
        return self.arrays


def _results(case):
    kind = case["kind"]
    if kind == "components":
        n = _components_room(case)
        return _Results(np.zeros, mapping=((n + 1,), np.int64), roots=((n,), np.int64))
    if kind == "edt":
        return None
    labels, vertices, edges = _sizes(case)
    rooms = dict(labels=((labels,), np.int64), v_off=((labels + 1,), np.int64), e_off=((labels + 1,), np.int64),
                 vertices=((vertices, 3), np.float32), edges=((edges, 2), np.uint32), radii=((vertices,), np.float32))
    if kind == "batch":
        rooms.update(sample=((labels,), np.int64), s_off=((case["count"] + 1,), np.int64))
    if kind in ("merge", "postprocess"):  # results that stay on the GPU
        types = {np.float32: torch.float32, np.uint32: torch.int64}
        on_gpu = {k: (rooms[k][0], types[rooms[k][1]]) for k in ("vertices", "edges", "radii")}
        return (_Results(np.zeros, **{k: rooms[k] for k in ("labels", "v_off", "e_off")}),
                _Results(lambda shape, dtype: torch.zeros(shape, dtype=dtype, device="cuda"), **on_gpu))
    return _Results(np.zeros, **rooms)


def prepare(case, seed):
    kind, results = case["kind"], _results(case)
    if kind == "skeletonize":
        x, layout = _labels(case, seed), case["layout"].split()
        if layout[0] == "host":
            x = np.asarray(x.astype(DTYPES[case["dtype"]], copy=False), order=layout[1])
        else:
            x = _to_device(x, case["dtype"], layout[1])
    elif kind == "batch":
        x = [_to_device(synth.volume("tubes", s[:3], s[3], seed * 1000 + i), case["dtype"], "F")
             for i, s in enumerate(_batch_shapes(case))]
    elif kind in ("components", "edt"):
        x = _dense(case, seed)
    elif kind == "merge":
        parts, origins = _fragments(case, seed)
        x = [p.to_device("cuda") for p in parts], origins
    else:
        x = _skeletons(case, seed).to_device("cuda")
    return case, x, results


# ---- one pass ----------------------------------------------------------------------------------

def _arrays(p, *more):
    return {k: getattr(p, k) for k in ("labels", "v_off", "e_off", "vertices", "edges", "radii") + more}


def _on_gpu(results, p):
    a = _arrays(p)
    return {**results[0].take(**{k: a[k] for k in results[0].arrays}), **results[1].take(**{k: a[k] for k in results[1].arrays})}


def run(state):
    case, x, results = state
    kind = case["kind"]
    if kind == "skeletonize":
        return results.take(**_arrays(brook_amd.skeletonize(
            x, PARAMS, _aniso(case), dust_threshold=case["dust"], output="packed", progress=False,
            fix_branching=case["fix_branching"], fill_holes=case["fill_holes"])))
    if kind == "batch":
        return results.take(**_arrays(brook_amd.skeletonize_batch(x, PARAMS, (16, 16, 40), dust_threshold=1000,
                                                                  output="packed"), "sample", "s_off"))
    if kind == "components":
        ids, mapping, roots = device.connected_components(x)
        signed = {1: torch.uint8, 2: torch.int16, 4: torch.int32}[ids.element_size()]
        return dict(results.take(mapping=mapping, roots=roots), ids=ids.view(signed).permute(2, 1, 0))
    if kind == "edt":
        return device.edt(x, _aniso(case), case["border"]).permute(2, 1, 0)
    if kind == "merge":
        return _on_gpu(results, packed.merge_fragments(x[0], x[1], on_device=True))
    return _on_gpu(results, device_post.postprocess(x, 1500.0, 3500.0))


# ---- what a pass cannot do without ---------------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "skeletonize":  # the labels in; the skeletons out are a thousandth of that
        return dict(bytes=case["sx"] * case["sy"] * case["sz"] * np.dtype(DTYPES[case["dtype"]]).itemsize, flops=0)
    if kind == "batch":
        return dict(bytes=sum(a * b * c for a, b, c, _ in _batch_shapes(case)) * np.dtype(DTYPES[case["dtype"]]).itemsize, flops=0)
    if kind in ("components", "edt"):
        voxels = case["sx"] * case["sy"] * case["sz"]
        cells = 1.0
        for s in ("sx", "sy", "sz"):
            cells *= case[s] / case["cell"] + 1
        out = 4 if kind == "edt" else 1 if cells < 250 else 2 if cells < 65000 else 4
        return dict(bytes=voxels * (np.dtype(DTYPES[case["dtype"]]).itemsize + out), flops=0)
    # vertices, radii and edges in once, and out once
    vertices = case["labels"] * (1 + case["branches"] * (0.7 * case["length"] + 0.3 * 5))
    if kind == "merge":
        return dict(bytes=vertices * (case["fragments"] * 16 + 16 + 8 + 16 + 16), flops=0)
    return dict(bytes=vertices * (16 + 16 + 16 + 16), flops=0)


def tolerance(case):
    # Distances are float32 results of one rounding of an exact sum and one of its root: 6e-8 in all,
    # and at most an ulp at a value. Every other output is a choice (ids, paths, orders) or a copied
    # value: a path that differs in one vertex is another skeleton.
    return {"rel": 2e-7, "max": 5e-7} if case["kind"] == "edt" else "exact"


# ---- the same in 64 bits ---------------------------------------------------------------------------

def _exact_edt(labels, aniso, border):
    """Multi-label squared distances, one axis after another: within each run of one label the lower
    envelope of the parabolas of its positions and of the walls at its ends (none at the volume's faces
    unless `border`), by trying every offset as long as a run is that long."""
    d = torch.zeros(labels.shape, dtype=torch.float64, device=labels.device)
    for axis in (2, 1, 0):  # tensor axes of x, y, z: labels come as (z, y, x)
        w = float(aniso[2 - axis])
        l, f = labels.movedim(axis, 0), d.movedim(axis, 0)
        n = l.shape[0]
        inf = torch.full_like(f[0], float("inf"))
        # steps to the wall on either side
        up, down = torch.empty_like(f), torch.empty_like(f)
        run = inf if not border else torch.zeros_like(inf)
        for i in range(n):
            run = run + 1 if i == 0 else torch.where(l[i] == l[i - 1], run + 1, torch.ones_like(run))
            up[i] = run
        run = inf if not border else torch.zeros_like(inf)
        for i in range(n - 1, -1, -1):
            run = run + 1 if i == n - 1 else torch.where(l[i] == l[i + 1], run + 1, torch.ones_like(run))
            down[i] = run
        wall = (w * torch.minimum(up, down)).square()
        best = wall if axis == 2 else torch.minimum(f, wall)
        if axis != 2:
            same = torch.ones((n, *l.shape[1:]), dtype=torch.bool, device=l.device)
            for k in range(1, n):  # same[i]: positions i..i+k hold one label
                same = same[:-1] & (l[k:] == l[k - 1:-1])
                if not bool(same.any()):
                    break
                step = (w * k) ** 2
                best[:-k] = torch.minimum(best[:-k], torch.where(same, f[k:] + step, float("inf")))
                best[k:] = torch.minimum(best[k:], torch.where(same, f[:-k] + step, float("inf")))
        d = best.movedim(0, axis).contiguous()
    return torch.where(labels == 0, 0.0, d.sqrt())


def _exact_merge(parts, origins):
    labels, verts, radii, edges, base = [], [], [], [], 0
    for p, o in zip(parts, origins):
        labels.append(np.repeat(p.labels, np.diff(p.v_off)))
        verts.append((p.vertices + np.asarray(o, np.float32)).astype(np.float64))  # positions meet in float32, as stored
        radii.append(p.radii.astype(np.float64))
        edges.append(p.edges.astype(np.int64) + np.repeat(p.v_off[:-1], np.diff(p.e_off))[:, None] + base)
        base += len(p.vertices)
    labels, verts, radii, edges = (np.concatenate(a) for a in (labels, verts, radii, edges))
    key = np.column_stack([labels.astype(np.float64), verts])
    order = np.lexsort((np.arange(len(key)), key[:, 3], key[:, 2], key[:, 1], key[:, 0]))
    head = np.ones(len(key), bool)
    head[1:] = (key[order[1:]] != key[order[:-1]]).any(1)
    rank = np.empty(len(key), np.int64)
    rank[order] = np.cumsum(head) - 1
    kept = order[head]
    e = np.sort(rank[edges], 1)
    used = np.zeros(len(kept), bool)
    used[e[e[:, 0] != e[:, 1]]] = True
    return verts[kept][used], radii[kept][used]


def exact(case, seed):
    kind = case["kind"]
    if kind == "edt":
        labels = _dense(case, seed).permute(2, 1, 0)
        return _exact_edt(labels, _aniso(case), case["border"])
    if kind == "merge":
        vertices, radii = _exact_merge(*_fragments(case, seed))
        room = _sizes(case)[1]
        out = dict(labels=None, v_off=None, e_off=None, vertices=np.zeros((room, 3)), edges=None, radii=np.zeros(room))
        out["vertices"][:len(vertices)], out["radii"][:len(radii)] = vertices, radii
        return out
    # A skeleton is a sequence of choices by float32 distances (64-bit ones choose other paths), and
    # ids have no rounding: no 64-bit value to be near to.
    return None
