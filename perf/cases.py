"""The calls a user of lvr2_amd makes, as measurable cases.

Every case is one way the package is used in earnest: normals of one scan, a whole job on a
small scan, a replayed multi-scan project, signed distances at a lattice, the reconstruction
from the lattice to the mesh, neighbour searches, and the differentiable signed distance.  The
clouds are the package's own synthetic scenes; the parameters are those of its workload
configurations (``lvr2_amd.scenes``) and of ``bench.py``.

    listed()            the cases with a name
    draw(rng)           one more case of the same ranges
    prepare(case, seed) what the caller's program holds before the call
    run(state)          one pass through the public entry points, and its outputs
    work(case)          bytes and operations one pass cannot do without
    exact(case, seed)   the same outputs in 64 bits (plain torch), for the clouds small enough
"""
from __future__ import annotations

import math

import numpy as np
import torch

from lvr2_amd import HipSurface, scenes
from lvr2_amd.autograd import hoppe_sdf

DEV = "cuda:0"
AREA = {"room": 900.0, "outdoor": 30000.0}  # surface of the scenes within a scan's reach, m^2
VIEW = 1e6  # HipSurface's default flip point is (VIEW, VIEW, VIEW)


# ---- the cases ----------------------------------------------------------------------------------


def listed() -> list[dict]:
    return [
        # A whole job on a small scan (one frame of a hand-held scanner): surface from a device
        # tensor, PCA normals with lvr2's default neighbourhoods, interpolation,
        # normals out.  Handle creation, allocations and launches count.
        {"name": "job_plain_30k", "kind": "job", "scene": "plain", "n": 30_000, "kn": 10, "ki": 10, "method": "PCA"},
        # The same job on a mid-sized terrestrial scan of an odd number of points, with the
        # scan-project neighbourhoods.
        {"name": "job_outdoor_500k", "kind": "job", "scene": "outdoor", "n": 500_003, "kn": 50, "ki": 20,
         "method": "PCA"},
        # The README's workload shape: 300,000 points, kn 10, ki 10, least-squares planes, on a
        # surface that the program keeps.
        {"name": "normals_plain_300k_ls", "kind": "normals", "scene": "plain", "n": 300_000, "kn": 10, "ki": 10,
         "method": "LS"},
        # The benchmark's terrestrial room scan: adaptive PCA normals and their interpolation.
        {"name": "normals_room_4m", "kind": "normals", "scene": "room", "n": 4_000_000, "kn": 50, "ki": 20,
         "method": "PCA"},
        # The large single cloud: the outdoor scan with the large configuration's neighbourhoods.
        {"name": "normals_outdoor_16m", "kind": "normals", "scene": "outdoor", "n": 16_000_000, "kn": 100, "ki": 30,
         "method": "PCA"},
        # A scan project in the batched form, replayed from its graph (tree rebuilt from the point
        # buffer, normals, interpolation): a program that refills one buffer with new scans.
        {"name": "project_graph_12", "kind": "project", "scans": 12, "lo": 50_000, "hi": 800_000, "kn": 50, "ki": 20},
        # Signed distances at the room's lattice vertices (the benchmark's voxel and kd).
        {"name": "sdf_room_lattice", "kind": "sdf", "scene": "room", "n": 4_000_000, "m": 700_000, "kd": 10,
         "voxel": 0.05},
        # The reconstruction of a mid-sized room scan: lattice, distances, PMC mesh, kept in the
        # fixed vertex and face buffers of a viewer.
        {"name": "reconstruct_room_1m", "kind": "mesh", "scene": "room", "n": 1_000_000, "kd": 10, "voxel": 0.05,
         "decomposition": "PMC"},
        # A handful of neighbour queries from host memory (SearchTree::kSearch for one chunk of
        # positions): latency.
        {"name": "ksearch_plain_500", "kind": "search", "scene": "plain", "n": 300_000, "m": 500, "k": 10},
        # Many neighbour queries from host memory, rows returned to the host.
        {"name": "ksearch_torus_200k", "kind": "search", "scene": "torus", "n": 300_000, "m": 200_001, "k": 20},
        # The differentiation form: surface, normals, distances in a two-voxel band and the reverse
        # pass to the points (the denoising step).
        {"name": "adjoint_torus_1m", "kind": "adjoint", "n": 1_000_000, "m": 500_000, "kn": 30, "kd": 10},
    ]


def _log_int(rng, lo: float, hi: float) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["job", "normals", "normals", "project", "sdf", "sdf", "mesh", "search", "search", "adjoint"])
    if kind in ("job", "normals"):
        scene = rng.choice(["plain", "room", "outdoor", "torus"])
        kn, ki = {"plain": (10, 10), "room": (50, 20), "outdoor": (rng.choice([50, 100]), rng.choice([20, 30])),
                  "torus": (30, rng.choice([10, 20]))}[scene]
        n = _log_int(rng, 10_000, 500_000) if kind == "job" else _log_int(rng, 50_000, 6_000_000)
        method = rng.choice(["PCA", "PCA", "LS", "ITERATIVE"]) if scene == "plain" else "PCA"
        return {"kind": kind, "scene": scene, "n": n, "kn": kn, "ki": ki, "method": method}
    if kind == "project":
        lo = _log_int(rng, 10_000, 100_000)
        return {"kind": kind, "scans": rng.randint(2, 16), "lo": lo, "hi": lo * rng.choice([1, 4, 10]),
                "kn": rng.choice([20, 50]), "ki": rng.choice([10, 20])}
    if kind in ("sdf", "mesh"):
        scene = rng.choice(["room", "outdoor"])
        n = _log_int(rng, 100_000, 3_000_000)
        out = {"kind": kind, "scene": scene, "n": n, "kd": rng.choice([5, 10, 10, 20]),
               "voxel": rng.choice([0.05, 0.08, 0.1]) if scene == "room" else rng.choice([0.2, 0.4])}
        if kind == "sdf":
            out["m"] = _log_int(rng, 2_000, 600_000)
        else:
            out["decomposition"] = rng.choice(["PMC", "PMC", "MC"])
        return out
    if kind == "search":
        return {"kind": kind, "scene": rng.choice(["plain", "torus", "room"]), "n": _log_int(rng, 20_000, 1_000_000),
                "m": _log_int(rng, 1, 300_000), "k": rng.choice([1, 5, 10, 20, 32, 50])}
    n = _log_int(rng, 50_000, 800_000)
    return {"kind": "adjoint", "n": n, "m": max(1000, n // rng.choice([2, 5])), "kn": 30, "kd": rng.choice([5, 10])}


# ---- inputs -------------------------------------------------------------------------------------


def _cloud(scene: str, n: int, seed: int):
    """(points (n, 3) float32 on the host, flip point): the package's scenes with exactly n points."""
    if scene == "plain":
        return scenes.plane_boxes_sphere(seed, n, 0.5), (VIEW, VIEW, VIEW)
    if scene == "torus":
        return scenes.sphere_torus(seed, n, 1.0, 0.01), (VIEW, VIEW, VIEW)
    if scene == "room":  # a 2.56 : 1 ray grid, cut to n
        n_el = max(4, int(round(math.sqrt(n / 2.56))))
        n_az = -(-n // n_el)
        return np.ascontiguousarray(scenes.room_scan(seed, n_az, n_el)[:n]), (0.0, 0.0, 0.0)
    pts, sc = scenes.outdoor_scan(seed, n)
    return pts, tuple(float(c) for c in sc)


def _positions(points: np.ndarray, m: int, seed: int) -> np.ndarray:
    """m positions near the cloud: points of it moved by about the spacing of 100 of them."""
    ext = points.max(0) - points.min(0)
    return scenes.band_queries(points, m, float(np.sqrt(np.prod(np.sort(ext)[1:]) / len(points)) * 10), seed + 1)


def _towards(points: np.ndarray, flip) -> np.ndarray:
    """Normals as a scanner file gives them for lack of better: the unit direction to the scanner."""
    d = np.asarray(flip, np.float64)[None] - points.astype(np.float64)
    l = np.linalg.norm(d, axis=1, keepdims=True)
    return (d / np.where(l > 0, l, 1.0)).astype(np.float32)


def _scan_sizes(case: dict) -> list[int]:
    """Points per scan of a project, evenly spread over [lo, hi] on a log scale, out of order."""
    k = case["scans"]
    step = math.log(case["hi"] / case["lo"]) / max(1, k - 1)
    return [int(case["lo"] * math.exp(step * (7 * i % k if k % 7 else i))) for i in range(k)]


def _mesh_cap(case: dict) -> int:
    """Rows of the vertex and face buffers: several times the scene's surface cells (two triangles
    each), objects and noise included."""
    return int(8 * AREA[case["scene"]] / case["voxel"] ** 2)


def _surface(points: torch.Tensor, case: dict, flip) -> HipSurface:
    s = HipSurface(points)
    s.setKn(case["kn"])
    s.setKi(case["ki"])
    s.setMethod(case.get("method", "PCA"))
    s.setFlippoint(*flip)
    return s


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind == "project":
        sizes = _scan_sizes(case)
        flips = [scenes.outdoor_pose(seed, 1000 + i) for i in range(len(sizes))]
        pts = np.concatenate([scenes.outdoor_scan_at(seed, f, n, 7000 + i) for i, (f, n) in enumerate(zip(flips, sizes))])
        pts = torch.from_numpy(pts).to(DEV)
        s = HipSurface(pts, scan_sizes=sizes)
        s.setKn(case["kn"])
        s.setKi(case["ki"])
        s.setScanFlippoints(np.asarray(flips, np.float32))
        out = torch.empty_like(pts)
        s.captureGraph(out, rebuild=True)
        return {"case": case, "surface": s, "points": pts, "out": out}
    if kind == "adjoint":
        pts = scenes.sphere_torus(seed, case["n"], 1.0, 0.01)
        q = scenes.band_queries(pts, case["m"], 0.1, seed + 1)
        return {"case": case, "points": torch.from_numpy(pts).to(DEV).requires_grad_(True),
                "queries": torch.from_numpy(q).to(DEV)}
    pts, flip = _cloud(case["scene"], case["n"], seed)
    dev = torch.from_numpy(pts).to(DEV)
    st = {"case": case, "points": dev, "flip": flip}
    if kind == "job":
        return st
    if kind == "normals":
        st["surface"] = _surface(dev, case, flip)
        st["out"] = torch.empty_like(dev)
        return st
    s = HipSurface(dev)
    st["surface"] = s
    if kind == "search":
        st["queries"] = _positions(pts, case["m"], seed)
        return st
    s.setKd(case["kd"])
    s.setNormals(_towards(pts, flip))
    if kind == "sdf":
        m = case["m"]  # the lattice's first m vertices: one slab of it
        v, _, _ = s.grid(case["voxel"], device=True)
        st["queries"] = v[torch.arange(m, device=DEV) % len(v)].contiguous()
        st["out"] = (torch.empty(m, dtype=torch.float32, device=DEV), torch.empty(m, dtype=torch.float32, device=DEV),
                     torch.empty(m, dtype=torch.uint8, device=DEV))
    else:
        cap = _mesh_cap(case)
        st["vertices"] = torch.zeros((cap, 3), dtype=torch.float32, device=DEV)
        st["faces"] = torch.zeros((cap, 3), dtype=torch.int32, device=DEV)
    return st


# ---- the calls ----------------------------------------------------------------------------------


def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind == "job":
        s = _surface(state["points"], case, state["flip"])
        s.calculateNormals()
        s.interpolateNormals()
        return s.getNormals(torch.empty_like(state["points"]))
    s = state.get("surface")
    if kind == "normals":
        s.calculateNormals()
        s.interpolateNormals()
        return s.getNormals(state["out"])
    if kind == "project":
        s.launchGraph()
        return state["out"]
    if kind == "sdf":
        return s.distances(state["queries"], case["voxel"], out=state["out"])
    if kind == "mesh":
        v, f = s.reconstruct(case["voxel"], decomposition=case["decomposition"], device=True)
        state["vertices"][:len(v)] = v
        state["faces"][:len(f)] = f
        return len(v), len(f), state["vertices"], state["faces"]
    if kind == "search":
        return s.kSearch(state["queries"], case["k"])
    p = state["points"]
    p.grad = None
    proj = hoppe_sdf(p, state["queries"], kn=case["kn"], kd=case["kd"], flip=(VIEW, VIEW, VIEW), voxel=0.05)
    (proj * proj).sum().backward()
    return proj.detach(), p.grad


def work(case: dict) -> dict:
    """Inputs read once, outputs written once; the operations are those of the neighbour sets' own
    arithmetic (8 per distance, about 20 per moment sum) on the neighbours alone."""
    kind = case["kind"]
    if kind in ("job", "normals"):
        return {"bytes": 24.0 * case["n"], "flops": case["n"] * (2 * case["kn"] * 28.0 + case["ki"] * 11.0)}
    if kind == "project":
        n = sum(_scan_sizes(case))
        return {"bytes": 24.0 * n, "flops": n * (2 * case["kn"] * 28.0 + case["ki"] * 11.0)}
    if kind in ("sdf", "mesh"):
        # a mesh's lattice: about two vertices per surface cell, no more than the points touch
        m = case["m"] if kind == "sdf" else min(2.0 * AREA[case["scene"]] / case["voxel"] ** 2, 3.0 * case["n"])
        return {"bytes": 24.0 * case["n"] + (21.0 if kind == "sdf" else 60.0) * m, "flops": m * case["kd"] * 14.0}
    if kind == "search":
        return {"bytes": 12.0 * min(case["n"], case["m"] * case["k"]) + case["m"] * (12.0 + 8.0 * case["k"]), "flops": case["m"] * case["k"] * 8.0}
    return {"bytes": 36.0 * case["n"] + 16.0 * case["m"],
            "flops": 3.0 * case["n"] * 2 * case["kn"] * 28.0 + 3.0 * case["m"] * case["kd"] * 14.0}


# ---- the same in 64 bits --------------------------------------------------------------------------


def _keys(q: torch.Tensor, p: torch.Tensor, idx: torch.Tensor) -> torch.Tensor:
    """(fp32 d^2, index) keys of every (query, point) pair, d^2 = (dx dx + dy dy) + dz dz."""
    d = q[:, None, 0] - p[None, :, 0]
    acc = d * d
    d = q[:, None, 1] - p[None, :, 1]
    acc += d * d
    d = q[:, None, 2] - p[None, :, 2]
    acc += d * d
    return (acc.view(torch.int32).to(torch.int64) << 32) | idx


def _nearest(q: torch.Tensor, p: torch.Tensor, k: int):
    """Per chunk of queries: (first row, indices of the k nearest points, ascending by key)."""
    idx = torch.arange(len(p), device=p.device)
    rows = max(1, min(1024, int(1.5e8 // len(p))))
    for a in range(0, len(q), rows):
        key = torch.topk(_keys(q[a:a + rows], p, idx), min(k, len(p)), dim=1, largest=False, sorted=True).values
        yield a, key & 0xFFFFFFFF


def _plane(method: str, q: torch.Tensor, nb: torch.Tensor) -> torch.Tensor:
    """Plane normals (unoriented) of the neighbourhoods nb (r, k, 3) of the points q (r, 3), fp64."""
    rel = nb - q[:, None]
    k = rel.shape[1]
    if method == "LS":  # y = c0 + c1 x + c2 z on the k-set; two tangents from the point
        a = torch.stack([torch.ones_like(rel[..., 0]), rel[..., 0], rel[..., 2]], -1)
        c = torch.linalg.solve(a.transpose(1, 2) @ a, (a.transpose(1, 2) @ rel[..., 1:2]))[..., 0]
        eps = 100.0
        d1 = torch.stack([torch.full_like(c[:, 0], eps), c[:, 0] + c[:, 1] * eps, torch.zeros_like(c[:, 0])], -1)
        d2 = torch.stack([torch.zeros_like(c[:, 0]), c[:, 0] + c[:, 2] * eps, torch.full_like(c[:, 0], eps)], -1)
        n = torch.linalg.cross(d1, d2)
        return n / n.norm(dim=1, keepdim=True)
    s2 = rel.transpose(1, 2) @ rel
    if method == "ITERATIVE":
        xx, xy, xz, yy, yz, zz = s2[:, 0, 0], s2[:, 0, 1], s2[:, 0, 2], s2[:, 1, 1], s2[:, 1, 2], s2[:, 2, 2]
        det = torch.stack([yy * zz - yz * yz, xx * zz - xz * xz, xx * yy - xy * xy], 1)
        a, b, c = xz * yz - xy * zz, xy * yz - xz * yy, xy * xz - yz * xx
        n = torch.stack([torch.stack([det[:, 0], a, b], 1), torch.stack([a, det[:, 1], c], 1),
                         torch.stack([b, c, det[:, 2]], 1)], 1)
        n = n[torch.arange(len(n), device=n.device), det.argmax(1)]
        return n / n.norm(dim=1, keepdim=True)
    mean = rel.sum(1) / (k + 1)  # the point itself is one sample more
    return torch.linalg.eigh(s2 / (k + 1) - mean[:, :, None] * mean[:, None, :]).eigenvectors[..., 0]


def _exact_normals(p: torch.Tensor, kn: int, ki: int, method: str, flip) -> torch.Tensor:
    n = len(p)
    p64 = p.double()
    f = torch.tensor(flip, dtype=torch.float64, device=p.device)
    raw = torch.empty((n, 3), dtype=torch.float64, device=p.device)
    near = torch.empty((n, min(ki, n)), dtype=torch.int64, device=p.device)
    for a, nb in _nearest(p, p, max(32 * kn, ki)):
        q = p64[a:a + len(nb)]
        near[a:a + len(nb)] = nb[:, :ki]
        todo = torch.arange(len(nb), device=p.device)
        for r in range(1, 6):
            if len(todo) == 0:
                break
            nbp = p64[nb[todo, :kn << r]]
            ext = nbp.amax(1) - nbp.amin(1)
            ok = (ext[:, :, None] >= 0.05 * ext[:, None, :]).all(2).all(1) | (r == 5)
            at = todo[ok]
            if len(at):
                raw[a + at] = _plane(method, q[at], nbp[ok])
            todo = todo[~ok]
    side = (raw * (f - p64)).sum(1)
    raw = torch.where(side[:, None] < 0, -raw, raw)
    out = raw + raw[near].sum(1)
    return out / out.norm(dim=1, keepdim=True)


def exact(case: dict, seed: int):
    kind = case["kind"]
    pairs = case.get("n", 0) * (case["m"] if kind == "search" else case.get("n", 0))
    if kind not in ("job", "normals", "search") or pairs > 9.1e10:
        return None
    if kind != "search" and case["n"] * case["n"] * case["kn"] > 9.1e11:  # the sort of 32 kn neighbours
        return None
    pts, flip = _cloud(case["scene"], case["n"], seed)
    p = torch.from_numpy(pts).to(DEV)
    if kind != "search":
        return _exact_normals(p, case["kn"], case["ki"], case["method"], flip)
    q = torch.from_numpy(_positions(pts, case["m"], seed)).to(DEV)
    d2 = np.empty((case["m"], case["k"]), np.float64)
    for a, nb in _nearest(q, p, case["k"]):
        d = q[a:a + len(nb)].double()[:, None] - p[nb].double()
        d2[a:a + len(nb)] = (d * d).sum(2).cpu().numpy()
    return None, d2
