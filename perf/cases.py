"""The work that users of this engine have it do, as timed cases.

`listed()` holds the named cases, `draw(rng)` gives another of the same
ranges.  `prepare(case, seed)` makes what a program holds before the call
(inputs on the GPU, the context it keeps), `run(state)` is one pass through
the public entry points, `work(case)` the bytes and operations a pass cannot
do without, and `exact(case, seed)` the pass's computed numbers in 64 bits.

A remeshing program takes patch after patch: for each it rasterizes the
density, moves the sites by Lloyd's iteration (the bulk of the time),
triangulates them and lifts them back to the surface.  The kinds of case are
those stages; their sizes are the ones of cvtamd.workloads, bench.py and the
tests (512^2 to 4096^2 grids at about 256 pixels per site, 11858-face patch
meshes, 16384 to 1 M points, the 256^2 network at batches of 1 and 16).
"""
from __future__ import annotations

import math
import random
import sys
from pathlib import Path

import numpy as np
import torch

_PKG = Path.cwd() / "surface-remesher_amd"
if str(_PKG) not in sys.path:
    sys.path.insert(0, str(_PKG))

import cvtamd                                    # noqa: E402
from cvtamd import compat, recover, weighting    # noqa: E402
from cvtamd.delaunay import Delaunay             # noqa: E402
from cvtamd.warmstart import UNet                # noqa: E402

DEV = "cuda"
WEIGHTS = _PKG / "weights" / "warmstart_r256.bin"


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # a small patch: uniform density, 1024 sites, where every launch counts
        {"name": "lloyd-512", "kind": "lloyd", "width": 512, "height": 512, "sites": 1024,
         "density": "uniform", "iterations": 50},
        # the headline patch: a disk with Gaussian bumps, 16384 sites
        {"name": "lloyd-2048", "kind": "lloyd", "width": 2048, "height": 2048, "sites": 16384,
         "density": "disk", "iterations": 40},
        # the largest patch: a star domain, 65536 sites
        {"name": "lloyd-4096", "kind": "lloyd", "width": 4096, "height": 4096, "sites": 65536,
         "density": "star", "iterations": 16},
        # a grid of no round size, its width not a multiple of four
        {"name": "lloyd-767x509", "kind": "lloyd", "width": 767, "height": 509, "sites": 1525,
         "density": "disk", "iterations": 50},
        # many patches of 256^2 .. 2048^2 advanced together (training pairs of
        # the warm start, a model cut into patches)
        {"name": "batch-64", "kind": "batch", "patches": 64, "layout": 4, "iterations": 10},
        # the reference's entry point: integer sites, host buffers
        {"name": "gcvt-1024", "kind": "gcvt", "n": 1024, "sites": 4096, "depth": 1,
         "max_iter": 60},
        # a patch's density: vertex weights of an 11858-face mesh, then its raster
        {"name": "density-12k-2048", "kind": "density", "mesh": 78, "n": 2048},
        # lifting the remeshed patch: 16384 sites and 32768 centroids located
        {"name": "locate-12k-49k", "kind": "locate", "mesh": 78, "queries": 49152},
        # a large point set triangulated inside the corners of its square
        {"name": "delaunay-1m", "kind": "delaunay", "points": 1000000, "ring": 4,
         "constrained": False},
        # a remeshed patch: its sites inside a constrained square boundary
        {"name": "delaunay-16k-ring", "kind": "delaunay", "points": 16384, "ring": 1024,
         "constrained": True},
        # the warm start of one patch: the network's forward pass
        {"name": "unet-forward-1", "kind": "unet", "batch": 1, "train": False},
        # a training step of the network: forward, loss and backward
        {"name": "unet-train-16", "kind": "unet", "batch": 16, "train": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["lloyd"] * 5 + ["batch", "gcvt", "density", "locate", "delaunay", "delaunay",
                                       "unet", "unet"])
    if kind == "lloyd":
        # patches of a parameterized surface: sides 256 .. 4096, aspect up to
        # 2, 128 .. 1024 pixels per site; four in five have a width that is a
        # multiple of four
        w = _log_int(rng, 256, 4096)
        h = min(4096, max(256, int(round(w * 2.0 ** rng.uniform(-1.0, 1.0)))))
        if rng.random() < 0.8:
            w = max(256, 4 * (w // 4))
        px = math.exp(rng.uniform(math.log(128.0), math.log(1024.0)))
        its = max(4, min(50, int(2.6e8 / (w * h))))
        return {"kind": "lloyd", "width": w, "height": h, "sites": max(256, int(w * h / px)),
                "density": rng.choice(["uniform", "disk", "star"]), "iterations": its}
    if kind == "batch":
        return {"kind": "batch", "patches": rng.randint(8, 48), "layout": rng.randint(5, 10 ** 6),
                "iterations": 10}
    if kind == "gcvt":
        n = _log_int(rng, 256, 1024)
        return {"kind": "gcvt", "n": n, "sites": max(64, int(n * n / rng.uniform(128, 512))),
                "depth": 1, "max_iter": 60}
    if kind == "density":
        return {"kind": "density", "mesh": _log_int(rng, 20, 400), "n": _log_int(rng, 256, 2048)}
    if kind == "locate":
        return {"kind": "locate", "mesh": _log_int(rng, 20, 120),
                "queries": _log_int(rng, 1000, 200000)}
    if kind == "delaunay":
        ring = rng.choice([4, 256, 1024])
        return {"kind": "delaunay", "points": _log_int(rng, 1000, 900000 if ring == 4 else 100000),
                "ring": ring, "constrained": ring > 4}
    train = rng.random() < 0.5
    return {"kind": "unet", "batch": rng.randint(2, 15 if train else 16), "train": train}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) & 0x7FFFFFFFFFFFFFFF)


def _unif(g, *shape):
    return torch.rand(*shape, dtype=torch.float64, device=DEV, generator=g)


def _density(kind, w, h, seed):
    """float32 (h, w) density of a patch: uniform, Gaussian bumps on the
    inscribed ellipse (disk), or waves and bumps in a star-shaped domain."""
    r = random.Random(seed)
    x = ((torch.arange(w, dtype=torch.float64, device=DEV) + 0.5) / w)[None, :]
    y = ((torch.arange(h, dtype=torch.float64, device=DEV) + 0.5) / h)[:, None]
    if kind == "uniform":
        return torch.ones((h, w), dtype=torch.float32, device=DEV)
    if kind == "disk":
        rho = torch.full((h, w), 0.2, dtype=torch.float64, device=DEV)
        for _ in range(8):
            rad, t = 0.5 * math.sqrt(r.random()), 2 * math.pi * r.random()
            cx, cy = 0.5 + rad * math.cos(t), 0.5 + rad * math.sin(t)
            amp, sx, sy = r.uniform(0.5, 2.0), r.uniform(0.04, 0.2), r.uniform(0.04, 0.2)
            c, s = math.cos(a := r.uniform(0.0, math.pi)), math.sin(a)
            u, v = c * (x - cx) + s * (y - cy), -s * (x - cx) + c * (y - cy)
            rho += amp * torch.exp(-0.5 * (u * u / (sx * sx) + v * v / (sy * sy)))
        inside = (x - 0.5) ** 2 + (y - 0.5) ** 2 <= 0.25
    else:
        k = 64
        rad = torch.tensor([r.uniform(0.6, 1.0) * 0.5 for _ in range(k)], dtype=torch.float64,
                           device=DEV)
        ang = 2 * math.pi * torch.arange(k, dtype=torch.float64, device=DEV) / k
        vx, vy = 0.5 + rad * torch.cos(ang), 0.5 + rad * torch.sin(ang)
        theta = torch.remainder(torch.atan2(y - 0.5, x - 0.5), 2 * math.pi)
        a = (theta / (2 * math.pi / k)).long().clamp_(max=k - 1)
        b = (a + 1) % k
        inside = ((vx[b] - vx[a]) * (y - vy[a]) - (vy[b] - vy[a]) * (x - vx[a])) >= 0
        rho = 0.3 + (torch.sin(7 * x) * torch.cos(5 * y)) ** 2
        for _ in range(4):
            cx, cy = r.uniform(0.3, 0.7), r.uniform(0.3, 0.7)
            rho = rho + torch.exp(-((x - cx) ** 2 + (y - cy) ** 2) / 0.01)
    return torch.where(inside, rho, torch.zeros_like(rho)).float()


def _sites(rho, num, g):
    """float32 (num, 2) sites in pixel units, drawn with probability
    proportional to the density by rejection."""
    h, w = rho.shape
    top = float(rho.max())
    out = []
    have = 0
    while have < num:
        u = _unif(g, max(6 * num, 4096), 3)
        px = (u[:, 0] * w).long().clamp_(max=w - 1)
        py = (u[:, 1] * h).long().clamp_(max=h - 1)
        ok = rho[py, px].double() > u[:, 2] * top
        p = torch.stack([(px + u[:, 0] * w % 1.0), (py + u[:, 1] * h % 1.0)], 1)[ok]
        out.append(p)
        have += p.shape[0]
    return torch.cat(out)[:num].float().contiguous()


def _batch_layout(case):
    """(side, sites) of every patch: sides log-uniform in 256 .. 2048, rounded
    to 64, about 256 pixels per site."""
    r = random.Random(case["layout"])
    out = []
    for _ in range(case["patches"]):
        side = 64 * round(math.exp(r.uniform(math.log(256.0), math.log(2048.0))) / 64)
        side = min(2048, max(256, side))
        out.append((side, max(256, round(side * side * r.uniform(0.5, 1.0) / 256))))
    return out


def _mesh(m, g):
    """A parameterized patch: an m x m jittered grid of [0, 1]^2 in 2 (m-1)^2
    shuffled triangles, and the surface z = 0.3 sin(3u) cos(2v) over it."""
    h = 1.0 / (m - 1)
    i = torch.arange(m, dtype=torch.float64, device=DEV) * h
    y, x = torch.meshgrid(i, i, indexing="ij")
    uv = torch.stack([x.reshape(-1), y.reshape(-1)], 1)
    inner = ((uv > 0) & (uv < 1 - 0.5 * h)).all(1)
    jit = (_unif(g, m * m, 2) - 0.5) * (0.6 * h)
    uv = torch.where(inner[:, None], uv + jit, uv).contiguous()
    c = torch.arange(m - 1, device=DEV)
    a = (c[:, None] * m + c[None, :]).reshape(-1)
    tri = torch.cat([torch.stack([a, a + 1, a + m + 1], 1), torch.stack([a, a + m + 1, a + m], 1)])
    tri = tri[torch.randperm(tri.shape[0], device=DEV, generator=g)].int().contiguous()
    p3 = torch.stack([uv[:, 0], uv[:, 1],
                      0.3 * torch.sin(3 * uv[:, 0]) * torch.cos(2 * uv[:, 1])], 1).contiguous()
    return uv, p3, tri


def _unet_input(nb, seed):
    """(nb, 256, 256, 32) bfloat16 network inputs (density over its mean, the
    smoothed site density, the domain), site positions and displacements."""
    R, S = 256, 1024
    x = torch.zeros((nb, R, R, 32), dtype=torch.bfloat16, device=DEV)
    uvs, tgs = [], []
    g = _gen(seed * 7919 + 3)
    for b in range(nb):
        rho = _density("disk", R, R, seed * 64 + b)
        xy = _sites(rho, S, g)
        cell = xy.long().clamp_(max=R - 1)
        cnt = torch.zeros((1, 1, R, R), dtype=torch.float64, device=DEV)
        cnt.view(-1).index_add_(0, cell[:, 1] * R + cell[:, 0],
                                torch.full((S,), R * R / S, dtype=torch.float64, device=DEV))
        win = torch.nn.functional.avg_pool2d(cnt, 15, stride=1, padding=7)[0, 0]
        x[b, :, :, 0] = rho / rho.double().mean().float()
        x[b, :, :, 1] = win.float()
        x[b, :, :, 2] = (rho > 0).float()
        uvs.append(xy / R)
        # a converged solution moves the sites by a few per cent of the side
        tgs.append(0.02 * torch.sin(6.0 * (xy / R).flip(1)))
    return x, torch.stack(uvs).contiguous(), torch.stack(tgs).float().contiguous()


def _ring(n, lo, hi):
    """n boundary points of a square, in order."""
    k = n // 4
    t = np.arange(k) * ((hi - lo) / k)
    return np.concatenate([np.stack([lo + t, 0 * t + lo], 1), np.stack([0 * t + hi, lo + t], 1),
                           np.stack([hi - t, 0 * t + hi], 1), np.stack([0 * t + lo, hi - t], 1)])


def _inputs(case, seed):
    """The arrays of a case, from its sizes and the seed alone."""
    kind = case["kind"]
    if kind == "lloyd":
        rho = _density(case["density"], case["width"], case["height"], seed)
        return {"rho": rho, "xy": _sites(rho, case["sites"], _gen(seed))}
    if kind == "batch":
        out = []
        for p, (side, num) in enumerate(_batch_layout(case)):
            rho = _density("disk", side, side, seed * 1000 + p)
            out.append((rho, _sites(rho, num, _gen(seed * 1000 + p))))
        return {"patches": out}
    if kind == "gcvt":
        n = case["n"]
        rho = _density("disk", n, n, seed)
        # constraint pixels on the domain's boundary, as a patch's corners are
        mask = np.zeros((n, n), np.uint8)
        for t in range(16):
            a = 2 * math.pi * t / 16
            mask[int(n * (0.5 + 0.48 * math.sin(a))), int(n * (0.5 + 0.48 * math.cos(a)))] = 1
        density = rho.cpu().numpy()
        first, _ = compat.ref_init_sites(density, case["sites"], mask,
                                         np.array([seed + 1, 362436069, 521288629, 7654321],
                                                  np.uint32))
        return {"density": density, "mask": mask, "first": first}
    if kind in ("density", "locate"):
        g = _gen(seed)
        uv, p3, tri = _mesh(case["mesh"], g)
        if kind == "density":
            return {"uv": uv, "p3": p3, "tri": tri, "scale": 1.0 / (case["n"] - 1)}
        ns = max(3, case["queries"] // 3)
        s = _unif(g, ns, 2)
        t = torch.randint(0, ns, (case["queries"] - ns, 3), device=DEV, generator=g)
        q = torch.cat([s, (s[t[:, 0]] + s[t[:, 1]] + s[t[:, 2]]) / 3.0]).contiguous()
        return {"uv": uv, "p3": p3, "tri": tri, "q": q}
    if kind == "delaunay":
        pts = (_unif(_gen(seed), case["points"], 2) * 4096.0).float().double()
        ring = _ring(case["ring"], -1.0, 4097.0)
        k, n = len(ring), case["points"]
        seg = np.stack([n + np.arange(k), n + (np.arange(k) + 1) % k], 1).astype(np.int32)
        pts = torch.cat([pts, torch.from_numpy(ring).to(DEV)]).contiguous()
        return {"points": pts,
                "segments": torch.from_numpy(seg).to(DEV) if case["constrained"] else None}
    x, uv, target = _unet_input(case["batch"], seed)
    return {"x": x, "uv": uv, "target": target}


def prepare(case, seed):
    s = dict(_inputs(case, seed), case=case)
    kind = case["kind"]
    if kind == "lloyd":
        w, h = case["width"], case["height"]
        s["engine"] = cvtamd.Engine(w, h, case["sites"])
        # densities that gather the sites take a small moment tile (a tile can
        # meet a bounded number of sites; the results do not depend on it)
        if case["density"] != "uniform":
            s["engine"].tile = 64 if w * h >= 250 * case["sites"] else 32
        s["out"] = torch.empty((case["sites"], 2), dtype=torch.float32, device=DEV)
        s["labels"] = torch.empty((h, w), dtype=torch.int32, device=DEV)
    elif kind == "batch":
        lay = _batch_layout(case)
        s["batch"] = cvtamd.Batch([(a, a) for a, _ in lay], [n for _, n in lay])
        for p in range(len(lay)):
            s["batch"].set_tile(p, 64)
    elif kind == "density":
        s["weights"] = torch.empty(s["uv"].shape[0], dtype=torch.float64, device=DEV)
        s["out"] = torch.empty((case["n"], case["n"]), dtype=torch.float32, device=DEV)
    elif kind == "locate":
        nq = case["queries"]
        s["out"] = (torch.empty(nq, dtype=torch.int32, device=DEV),
                    torch.empty((nq, 3), dtype=torch.float64, device=DEV),
                    torch.empty((nq, 3), dtype=torch.float64, device=DEV))
    elif kind == "delaunay":
        s["context"] = Delaunay(s["points"].shape[0])
    elif kind == "unet":
        net = UNet(256, case["batch"], 0)
        net.load(WEIGHTS)
        s["net"] = net
        s["field"] = torch.empty((case["batch"], 256, 256, 2), dtype=torch.float32, device=DEV)
        if case["train"]:
            s["grads"] = torch.empty(net.num_params, dtype=torch.float32, device=DEV)
    torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "lloyd":
        # a new patch in the program's engine: its density and initial sites,
        # the iterations, then the sites, their cells and the energies
        e = s["engine"]
        e.set_density(s["rho"])
        e.set_sites(s["xy"])
        e.clear_history()
        e.lloyd(case["iterations"])
        e.sites(out=s["out"])
        history = e.history()
        e.voronoi()
        e.labels(out=s["labels"])
        return {"sites": s["out"], "history": history, "labels": s["labels"]}
    if kind == "batch":
        b = s["batch"]
        for p, (rho, xy) in enumerate(s["patches"]):
            b.set_density(p, rho)
            b.set_sites(p, xy)
        b.lloyd(case["iterations"])
        b.synchronize()
        return [b.sites(p) for p in range(len(s["patches"]))]
    if kind == "gcvt":
        v = s["first"].copy()
        it, ns = compat.gcvt(v, s["density"], s["mask"], case["depth"], case["max_iter"])
        return {"map": v, "iterations": it, "sites": ns}
    if kind == "density":
        weighting.vertex_weights(s["uv"], s["p3"], s["tri"], out=s["weights"])
        compat.rasterize(s["uv"], s["weights"], s["tri"], s["scale"], case["n"], out=s["out"])
        return {"weights": s["weights"], "density": s["out"]}
    if kind == "locate":
        face, w, xyz = recover.locate_points(s["uv"], s["tri"], s["q"], p3=s["p3"], out=s["out"])
        return {"face": face, "weights": w, "xyz": xyz}
    if kind == "delaunay":
        tri, opp = s["context"].compute(s["points"], segments=s["segments"])
        return {"tri": tri, "opp": opp}
    net, nb = s["net"], case["batch"]
    net.set_input(s["x"], nb)
    net.forward(nb)
    if not case["train"]:
        return {"field": net.field(nb, out=s["field"])}
    loss = net.loss_backward(nb, s["uv"], s["target"], s["uv"].shape[1])
    return {"field": net.field(nb, out=s["field"]), "loss": loss, "grads": net.grads(out=s["grads"])}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
# the network's convolutions (Cin, Cout, level); the first takes 3 channels
_CONVS = [(32, 32, 0), (32, 32, 0), (32, 64, 1), (64, 64, 1), (64, 96, 2), (96, 96, 2),
          (96, 128, 3), (128, 128, 3), (224, 96, 2), (96, 96, 2), (160, 64, 1), (64, 64, 1),
          (96, 32, 0), (32, 32, 0)]


def work(case):
    kind = case["kind"]
    if kind == "lloyd":
        px, S, it = case["width"] * case["height"], case["sites"], case["iterations"]
        # an iteration reads the density and reads and writes the sites; the
        # call writes the labels.  Per pixel: the distance of two candidate
        # sites compared (10) and its four moments added (8)
        return {"bytes": it * (4.0 * px + 16.0 * S) + 8.0 * px, "flops": 18.0 * px * it}
    if kind == "batch":
        px = sum(a * a for a, _ in _batch_layout(case))
        S, it = sum(n for _, n in _batch_layout(case)), case["iterations"]
        return {"bytes": it * (4.0 * px + 16.0 * S) + 4.0 * px, "flops": 18.0 * px * it}
    if kind == "gcvt":
        px, it = case["n"] ** 2, case["max_iter"]
        return {"bytes": it * 4.0 * px + 13.0 * px, "flops": 18.0 * px * it}
    if kind == "density":
        nv, nf, px = case["mesh"] ** 2, 2 * (case["mesh"] - 1) ** 2, case["n"] ** 2
        return {"bytes": 64.0 * nv + 24.0 * nf + 4.0 * px, "flops": 40.0 * nf + 30.0 * px}
    if kind == "locate":
        nv, nf, nq = case["mesh"] ** 2, 2 * (case["mesh"] - 1) ** 2, case["queries"]
        return {"bytes": 40.0 * nv + 12.0 * nf + 68.0 * nq, "flops": 45.0 * nq}
    if kind == "delaunay":
        n = case["points"] + case["ring"]
        # per point: two triangles written (24 B each), and about ten in-circle
        # tests of 40 operations
        return {"bytes": 16.0 * n + 48.0 * n + 8.0 * case["ring"], "flops": 400.0 * n}
    nb = case["batch"]
    fwd = sum(2.0 * 9 * ci * co * (256 >> l) ** 2 for ci, co, l in _CONVS) * nb
    act = sum(2.0 * co * (256 >> l) ** 2 for _, co, l in _CONVS) * nb
    inp = 64.0 * 256 * 256 * nb
    if not case["train"]:
        return {"bytes": inp + 8.0 * 256 * 256 * nb + 2.0 * 900000, "flops": fwd}
    # the backward pass reads every activation that the forward pass wrote
    return {"bytes": inp + 8.0 * 256 * 256 * nb + 2.0 * act + 6.0 * 900000,
            "flops": 3.0 * fwd - 2.0 * 9 * 32 * 32 * 256 * 256 * nb}


# ---------------------------------------------------------------------------
# the same numbers in 64 bits
# ---------------------------------------------------------------------------
def _jfa64(w, h, sx, sy):
    """Label map of jump flooding plus one more pass of step 1, distances in
    float64, ties to the lower index."""
    S = sx.shape[0]
    none = S
    px = sx.floor().long().clamp(0, w - 1)
    py = sy.floor().long().clamp(0, h - 1)
    lab = torch.full((h * w,), none, dtype=torch.int64, device=DEV)
    lab.scatter_reduce_(0, py * w + px, torch.arange(S, device=DEV), "amin", include_self=True)
    lab = lab.view(h, w)
    inf = torch.full((1,), math.inf, dtype=torch.float64, device=DEV)
    tx, ty = torch.cat([sx, inf]), torch.cat([sy, inf])
    cx = (torch.arange(w, dtype=torch.float64, device=DEV) + 0.5)[None, :]
    cy = (torch.arange(h, dtype=torch.float64, device=DEV) + 0.5)[:, None]
    step = 1
    while step * 2 < max(w, h):
        step *= 2
    steps = []
    while step:
        steps.append(step)
        step //= 2
    for st in steps + [1]:
        best, bd = lab, (tx[lab] - cx) ** 2 + (ty[lab] - cy) ** 2
        for dy in (-st, 0, st):
            for dx in (-st, 0, st):
                y0, y1, x0, x1 = max(0, -dy), min(h, h - dy), max(0, -dx), min(w, w - dx)
                if (dx == 0 and dy == 0) or y1 <= y0 or x1 <= x0:
                    continue
                c = lab[y0 + dy:y1 + dy, x0 + dx:x1 + dx]
                d = (tx[c] - cx[:, x0:x1]) ** 2 + (ty[c] - cy[y0:y1]) ** 2
                ob, od = best[y0:y1, x0:x1], bd[y0:y1, x0:x1]
                take = (d < od) | ((d == od) & (c < ob))
                if best is lab:
                    best, bd = lab.clone(), bd.clone()
                    ob, od = best[y0:y1, x0:x1], bd[y0:y1, x0:x1]
                ob.copy_(torch.where(take, c, ob))
                od.copy_(torch.where(take, d, od))
        lab = best
    return lab


def _lloyd64(rho, xy, iterations):
    h, w = rho.shape
    r = rho.double().reshape(-1)
    s = xy.double().clone()
    S = s.shape[0]
    cx = (torch.arange(w, dtype=torch.float64, device=DEV) + 0.5).repeat(h)
    cy = (torch.arange(h, dtype=torch.float64, device=DEV) + 0.5).repeat_interleave(w)
    hist = np.zeros((iterations, 2))
    for k in range(iterations):
        lab = _jfa64(w, h, s[:, 0].contiguous(), s[:, 1].contiguous()).reshape(-1)
        live = lab < S
        l, rr = lab[live], r[live]
        dx, dy = cx[live] - s[l, 0], cy[live] - s[l, 1]
        m = torch.zeros((4, S), dtype=torch.float64, device=DEV)
        for q, v in enumerate((rr, rr * dx, rr * dy, rr * (dx * dx + dy * dy))):
            m[q].index_add_(0, l, v)
        hist[k, 0] = float(m[3].sum()) / (w * h)
        hist[k, 1] = 2.0 / (w * h) * math.sqrt(float((m[1] ** 2 + m[2] ** 2).sum()))
        mv = m[0] > 0
        d = torch.where(mv[:, None], torch.stack([m[1], m[2]], 1) / m[0].clamp_min(1e-300)[:, None],
                        torch.zeros_like(s))
        s = s + d
    return s, hist


def _raster64(uv, wt, tri, scale, n):
    out = np.zeros((n, n))
    for t in tri[::-1]:                       # the first triangle in order is written last
        a, b, c = uv[t[0]], uv[t[1]], uv[t[2]]
        lo, hi = np.minimum(np.minimum(a, b), c), np.maximum(np.maximum(a, b), c)
        x0, y0 = max(0, int(lo[0] / scale) - 1), max(0, int(lo[1] / scale) - 1)
        x1, y1 = min(n - 1, int(hi[0] / scale) + 1), min(n - 1, int(hi[1] / scale) + 1)
        if x1 < x0 or y1 < y0:
            continue
        px = (np.arange(x0, x1 + 1) * scale)[None, :] - a[0]
        py = (np.arange(y0, y1 + 1) * scale)[:, None] - a[1]
        e0, e1 = b - a, c - a
        d00, d01, d11 = e0 @ e0, e0 @ e1, e1 @ e1
        den = d00 * d11 - d01 * d01
        if den == 0:
            continue
        d20, d21 = px * e0[0] + py * e0[1], px * e1[0] + py * e1[1]
        v, u = (d11 * d20 - d01 * d21) / den, (d00 * d21 - d01 * d20) / den
        z = 1.0 - v - u
        hit = (v >= 0) & (u >= 0) & (z >= 0)
        val = z * wt[t[0]] + v * wt[t[1]] + u * wt[t[2]]
        win = out[y0:y1 + 1, x0:x1 + 1]
        win[hit] = val[hit]
    return out


def _weights64(uv, p3, tri):
    a, b, c = (uv[tri[:, k]] for k in range(3))
    area2 = 0.5 * np.abs((b[:, 0] - a[:, 0]) * (c[:, 1] - a[:, 1]) -
                         (b[:, 1] - a[:, 1]) * (c[:, 0] - a[:, 0]))
    a, b, c = (p3[tri[:, k]] for k in range(3))
    area3 = 0.5 * np.sqrt((np.cross(b - a, c - a) ** 2).sum(1))
    s2, s3 = np.zeros(len(uv)), np.zeros(len(uv))
    for k in range(3):
        np.add.at(s2, tri[:, k], area2)
        np.add.at(s3, tri[:, k], area3)
    return s3 / s2


def _locate64(uv, p3, tri, q):
    """Weights and lifted points of each query in the first face holding it."""
    f = tri.long()
    a, b, c = uv[f[:, 0]], uv[f[:, 1]], uv[f[:, 2]]
    e0, e1 = b - a, c - a
    d00, d01, d11 = (e0 * e0).sum(1), (e0 * e1).sum(1), (e1 * e1).sum(1)
    den = d00 * d11 - d01 * d01
    ws, xs = [], []
    for p in q.split(max(1, 40_000_000 // max(1, f.shape[0]))):
        d = p[:, None, :] - a[None]
        d20, d21 = (d * e0).sum(2), (d * e1).sum(2)
        v, u = (d11 * d20 - d01 * d21) / den, (d00 * d21 - d01 * d20) / den
        z = 1.0 - v - u
        hit = (v >= 0) & (u >= 0) & (z >= 0)
        first = hit.int().argmax(1)
        ok = hit.any(1)
        rows = torch.arange(p.shape[0], device=DEV)
        w = torch.stack([z[rows, first], v[rows, first], u[rows, first]], 1)
        w = torch.where(ok[:, None], w, torch.full_like(w, -1.0))
        x = (w[:, :, None] * p3[f[first]]).sum(1)
        ws.append(w)
        xs.append(torch.where(ok[:, None], x, torch.zeros_like(x)))
    return torch.cat(ws), torch.cat(xs)


def _unet64(case, inp):
    """The network in float64 from the weight file: convolutions with
    [tap][Cout][Cin] weights and a bias, ReLU, 2x2 means, nearest upsampling
    joined to the skip, a 1x1 head; gradients by differentiation."""
    raw = WEIGHTS.read_bytes()
    bits = np.frombuffer(raw[24:], np.uint16).astype(np.uint32) << 16
    p = torch.from_numpy(bits.view(np.float32).astype(np.float64)).to(DEV)
    p.requires_grad_(case["train"])
    cuts, off = [], 0
    for ci, co, _ in _CONVS:
        cuts.append((off, off + 9 * ci * co, off + 9 * ci * co + co))
        off += 9 * ci * co + co

    def conv(l, x):
        ci, co, _ = _CONVS[l]
        o, ob, oe = cuts[l]
        k = p[o:ob].view(9, co, ci)
        n, h, w, _ = x.shape
        xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
        y = p[ob:oe].expand(n * h * w, co)
        for t in range(9):
            v = xp[:, t // 3:t // 3 + h, t % 3:t % 3 + w].reshape(-1, ci)
            y = y + v @ k[t].t().contiguous()
        return torch.relu(y).view(n, h, w, co)

    def pool(x):
        return 0.25 * (x[:, 0::2, 0::2] + x[:, 1::2, 0::2] + x[:, 0::2, 1::2] + x[:, 1::2, 1::2])

    def up(x, skip):
        return torch.cat([x.repeat_interleave(2, 1).repeat_interleave(2, 2), skip], 3)

    x = inp["x"].double()
    s1 = conv(1, conv(0, x))
    s2 = conv(3, conv(2, pool(s1)))
    s3 = conv(5, conv(4, pool(s2)))
    y = conv(7, conv(6, pool(s3)))
    y = conv(9, conv(8, up(y, s3)))
    y = conv(11, conv(10, up(y, s2)))
    y = conv(13, conv(12, up(y, s1)))
    field = y @ p[off:off + 64].view(2, 32).t() + p[off + 64:off + 66]
    if not case["train"]:
        return {"field": field}
    R = 256
    pos = (inp["uv"].double() * R - 0.5).clamp(0, R - 1)
    i0 = pos.floor().long()
    i1 = (i0 + 1).clamp(max=R - 1)
    t = pos - i0
    b = torch.arange(field.shape[0], device=DEV)[:, None]

    def at(ix, iy):
        return field[b, iy, ix]

    tx, ty = t[..., 0:1], t[..., 1:2]
    val = ((1 - tx) * (1 - ty) * at(i0[..., 0], i0[..., 1]) +
           tx * (1 - ty) * at(i1[..., 0], i0[..., 1]) +
           (1 - tx) * ty * at(i0[..., 0], i1[..., 1]) + tx * ty * at(i1[..., 0], i1[..., 1]))
    loss = ((val - inp["target"].double()) ** 2).sum(2).mean()
    loss.backward()
    return {"field": field.detach(), "loss": float(loss.detach()), "grads": p.grad}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("gcvt", "delaunay"):
        return None                               # whole numbers
    inp = _inputs(case, seed)
    if kind == "lloyd":
        s, hist = _lloyd64(inp["rho"], inp["xy"], case["iterations"])
        return {"sites": s, "history": hist, "labels": None}
    if kind == "batch":
        return [_lloyd64(rho, xy, case["iterations"])[0].cpu().numpy()
                for rho, xy in inp["patches"]]
    if kind == "density":
        if case["mesh"] > 150:
            return None
        uv, p3, tri = (inp[k].cpu().numpy() for k in ("uv", "p3", "tri"))
        wt = _weights64(uv, p3, tri)
        return {"weights": wt, "density": _raster64(uv, wt, tri, inp["scale"], case["n"])}
    if kind == "locate":
        w, x = _locate64(inp["uv"], inp["p3"], inp["tri"], inp["q"])
        return {"face": None, "weights": w, "xyz": x}
    return _unet64(case, inp)
