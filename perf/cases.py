"""The work a user of this framework has it do, as timed cases.

listed() names the cases, draw() gives more of the same ranges, prepare()
makes what a program holds before the call, run() is one pass through the
public entry points, work() the bytes and operations a pass cannot do without,
and exact() the 64-bit values of the outputs that have one.
"""
from __future__ import annotations

import itertools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "opengjk-gpu_amd"))

import ogjk  # noqa: E402
from ogjk import gen  # noqa: E402


def listed() -> list[dict]:
    return [
        # One frame of a small simulation or a planner's single query: a handful of close
        # pairs of small hulls at the library's default launch shape.  Latency and launches.
        dict(name="tiny_frame", kind="pairs", family=gen.ELLIPSOID, pairs=64, nmin=4, nmax=64,
             box=1.0, mode=3, gjk=8, epa=32),
        # Distance queries only, the reference's 1,000-pair batch.
        dict(name="distance_1k", kind="pairs", family=gen.SPHERE, pairs=1000, nmin=32, nmax=32,
             box=2.0, mode=1, gjk=64, epa=32),
        # The drop-in with host arrays, called as the reference's example does: distances,
        # then collision information from the simplices it got (1,000 pairs of 50 vertices).
        dict(name="host_two_calls", kind="host", family=gen.SPHERE, pairs=1000, nmin=50, nmax=50,
             box=1.5),
        # Batches of small hulls with many contacts (robotics and graphics meshes' pieces).
        dict(name="sphere64_100k", kind="pairs", family=gen.SPHERE, pairs=100_000, nmin=64,
             nmax=64, box=1.29, mode=3, gjk=8, epa=32),
        # Bodies of very different sizes over a resident, clustered scene.
        dict(name="uneven_100k", kind="clustered", family=gen.ELLIPSOID, pairs=100_000, nmin=4,
             nmax=4096, box=1.5, rebuild=False),
        # The same on new geometry each time (deforming bodies, one-shot queries): the
        # clusters are built in the pass; 40-byte contact records out.
        dict(name="uneven_new_20k", kind="clustered", family=gen.ELLIPSOID, pairs=20_000, nmin=4,
             nmax=4096, box=1.5, rebuild=True),
        # Scanned meshes: few pairs of very large hulls.
        dict(name="scans_1k", kind="clustered", family=gen.NOISY_SPHERE, pairs=1000, nmin=50_000,
             nmax=50_000, box=1.5, rebuild=False),
        # A serving process: a burst of requests of posed pairs against a resident scene,
        # host arrays in and out.
        dict(name="serving_burst", kind="serving", bodies=20_000, nmin=8, nmax=512, requests=8,
             kmax=10_000),
        # A simulation step over one scene: bounding spheres, broad phase, narrow phase.
        dict(name="scene_step_20k", kind="scene_step", bodies=20_000, nmin=8, nmax=512, tbox=40.0),
        # The broad phase alone on a large particle-like scene.
        dict(name="broad_1m", kind="broad", objects=1_000_000, cap=0),
        # Ingestion of many small convex pieces (the reference's random hull variants).
        dict(name="hulls_100k", kind="hulls", clouds=100_000, nmin=8, nmax=32, ellipsoid=False),
        # Ingestion of a scene's bodies of mixed sizes.
        dict(name="hulls_mixed_2k", kind="hulls", clouds=2000, nmin=8, nmax=512, ellipsoid=True),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["pairs", "pairs", "pairs", "host", "clustered", "clustered", "scans",
                       "serving", "scene_step", "broad", "hulls", "hulls"])
    if kind == "pairs":
        nmax = _log_int(rng, 8, 512)
        gjk, epa = (8, 32) if nmax <= 64 else rng.choice([(32, 32), (64, 64)])
        return dict(kind=kind, family=rng.choice([gen.SPHERE, gen.ELLIPSOID]),
                    pairs=_log_int(rng, 16, 100_000 if nmax <= 64 else 30_000),
                    nmin=_log_int(rng, 4, nmax), nmax=nmax, box=rng.uniform(0.8, 2.5),
                    mode=rng.choice([1, 3, 3]), gjk=gjk, epa=epa)
    if kind == "host":
        nmax = _log_int(rng, 8, 200)
        return dict(kind=kind, family=rng.choice([gen.SPHERE, gen.ELLIPSOID]),
                    pairs=_log_int(rng, 10, 10_000), nmin=_log_int(rng, 4, nmax), nmax=nmax,
                    box=rng.uniform(1.0, 2.5))
    if kind == "clustered":
        return dict(kind=kind, family=gen.ELLIPSOID, pairs=_log_int(rng, 500, 100_000),
                    nmin=_log_int(rng, 4, 64), nmax=_log_int(rng, 600, 4096),
                    box=rng.uniform(1.0, 2.0), rebuild=rng.random() < 0.4)
    if kind == "scans":
        nv = _log_int(rng, 4200, 100_000)
        return dict(kind="clustered", family=gen.NOISY_SPHERE,
                    pairs=_log_int(rng, 20, min(2000, 100_000_000 // (2 * nv))), nmin=nv, nmax=nv,
                    box=rng.uniform(1.0, 2.0), rebuild=rng.random() < 0.3)
    if kind == "serving":
        return dict(kind=kind, bodies=2 * _log_int(rng, 250, 10_000), nmin=8,
                    nmax=_log_int(rng, 32, 512), requests=rng.randint(1, 8),
                    kmax=_log_int(rng, 10, 10_000))
    if kind == "scene_step":
        nb = 2 * _log_int(rng, 250, 10_000)
        return dict(kind=kind, bodies=nb, nmin=8, nmax=_log_int(rng, 32, 512),
                    tbox=40.0 * (nb / 20_000) ** (1 / 3) * rng.uniform(0.9, 1.3))
    if kind == "broad":
        return dict(kind=kind, objects=_log_int(rng, 1000, 1_000_000), cap=rng.choice([0, 0, 512]))
    small = rng.random() < 0.6
    return dict(kind=kind, clouds=_log_int(rng, 50, 100_000 if small else 2000), nmin=8,
                nmax=rng.randint(16, 32) if small else _log_int(rng, 48, 512),
                ellipsoid=not small)


# ------------------------------------------------------------------ inputs

def _threads() -> int:
    return min(len(os.sched_getaffinity(0)), 16)


def _batch(case, seed):
    """The case's pairs; bodies of nmin..nmax vertices (log-uniform)."""
    if case["nmin"] == case["nmax"] or case["family"] != gen.ELLIPSOID:
        return gen.make(case["family"], case["pairs"], seed=seed, nverts=case["nmax"],
                        box=case["box"], nthreads=_threads(), nmin=case["nmin"],
                        nmax=case["nmax"])
    return gen.make(case["family"], case["pairs"], seed=seed, box=case["box"], nmin=case["nmin"],
                    nmax=case["nmax"], nthreads=_threads())


def _scene_bodies(case, seed):
    """Bodies in their local frames, as a resident scene holds them."""
    return gen.make(gen.ELLIPSOID, case["bodies"] // 2, seed=seed, box=0.0, nmin=case["nmin"],
                    nmax=case["nmax"], nthreads=_threads())


def _spheres(case, seed):
    n = case["objects"]
    half = n ** (1.0 / 3.0)  # about one object per cell of edge 2
    return gen.spheres(n, seed=seed, box=half, rmin=0.2, rmax=1.0), half, max(1, int(half))


def _clouds(case, seed):
    """Point clouds on unit spheres or on rotated ellipsoids (axes U[0.3, 2]);
    the sizes are the case's (log-uniform for ellipsoids), the points the seed's."""
    n, lo, hi = case["clouds"], case["nmin"], case["nmax"]
    sizes, rng = np.random.default_rng(n), np.random.default_rng(seed)
    if case["ellipsoid"]:
        cnt = np.minimum(np.exp(sizes.uniform(math.log(lo), math.log(hi + 1), n)), hi)
    else:
        cnt = sizes.integers(lo, hi + 1, n)
    cnt = cnt.astype(np.int32)
    off = np.zeros(n, np.int64)
    off[1:] = np.cumsum(cnt)[:-1]
    u = rng.normal(size=(int(cnt.sum()), 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    if case["ellipsoid"]:
        frame = np.linalg.qr(rng.normal(size=(n, 3, 3)))[0] * rng.uniform(0.3, 2.0, (n, 1, 3))
        u = (frame[np.repeat(np.arange(n), cnt)] @ u[..., None])[..., 0]
    return u.astype(np.float32), off, cnt


def _requests(case, seed):
    """Posed requests of evenly spread sizes up to kmax, in mixed order."""
    r, k = case["requests"], case["kmax"]
    sizes = [max(1, k * (2 * ((5 * i + 2) % r if r % 5 else i) + 1) // (2 * r)) for i in range(r)]
    pairs, poses = gen.posed_requests(case["bodies"], 1, seed=seed, kmin=sum(sizes),
                                      kmax=sum(sizes))[0]
    cut = np.cumsum(sizes)[:-1]
    return list(zip(np.split(pairs, cut), np.split(poses, cut)))


def _shape(case) -> dict:
    """The launch shape a program sets for the case's scene, the ones the
    benchmark uses: a bucket table for bodies of mixed sizes, else one shape."""
    kind = case["kind"]
    if kind == "clustered" and case["family"] == gen.ELLIPSOID:
        return dict(max_verts=(64,), gjk=(8, 64), epa=(32, 64), gjk_waves=(2, 1), epa_waves=(4, 4))
    if kind in ("clustered", "serving", "scene_step"):
        return dict(gjk=64, epa=64)
    if kind == "host":
        return dict(gjk=8, epa=32)
    if kind == "pairs":
        return dict(gjk=case["gjk"], epa=case["epa"])
    return {}


_set_shape: dict = {}


def _use(shape: dict) -> None:
    """The launch shape is the process's: set when the program turns to
    another scene."""
    global _set_shape
    if not shape or shape == _set_shape:
        return
    if "max_verts" in shape:
        ogjk.set_buckets(shape["max_verts"], shape["gjk"], shape["epa"])
        ogjk.set_block_waves(shape["gjk_waves"], shape["epa_waves"])
    else:
        ogjk.set_config(shape["gjk"], shape["epa"])
    _set_shape = shape


def _clear(*buffers) -> None:
    """Result buffers with room for more than a pass finds start out as zeros."""
    for b in buffers:
        b.zero_()


def prepare(case, seed):
    kind = case["kind"]
    st = dict(case=case, shape=_shape(case))
    if kind == "pairs":
        st["scene"] = ogjk.DeviceScene(_batch(case, seed))
        st["out"] = st["scene"].outputs(case["pairs"])
    elif kind == "host":
        st["batch"] = _batch(case, seed)
    elif kind == "clustered":
        big = case["nmax"] > 4096
        st["cluster_min"] = 1024 if big else 512
        st["scene"] = ogjk.DeviceScene(_batch(case, seed))
        if not case["rebuild"]:
            st["scene"].build_clusters(st["cluster_min"])
            st["out"] = st["scene"].outputs(case["pairs"])
        else:
            st["out"] = st["scene"].contacts(case["pairs"])
            st["ws"] = torch.empty(int(ogjk.lib().ogjk_workspace_bytes(case["pairs"])),
                                   dtype=torch.uint8, device="cuda")
    elif kind == "serving":
        st["scene"] = ogjk.DeviceScene(_scene_bodies(case, seed))
        st["requests"] = _requests(case, seed)
        st["server"] = ogjk.Server(st["scene"])
    elif kind == "scene_step":
        b = _scene_bodies(case, seed)
        radii = gen.body_radii(b.coords, b.off, b.cnt)
        grid = ogjk.Grid.for_spheres(float(radii.max()), case["tbox"], 64)
        st["step"] = ogjk.SceneStep(ogjk.DeviceScene(b), radii, grid, max_pairs=20 * len(b.cnt),
                                    contacts=True)
        _clear(st["step"].bp.pairs, st["step"].out["contacts"])
        st["poses"] = torch.from_numpy(gen.body_poses(len(b.cnt), seed=seed,
                                                      tbox=case["tbox"])).cuda()
    elif kind == "broad":
        s, half, g = _spheres(case, seed)
        n = case["objects"]
        st["bp"] = ogjk.BroadPhase(n, ogjk.Grid(2.0 * half / g, half, g, case["cap"]),
                                   max_pairs=8 * n)
        _clear(st["bp"].pairs)
        st["spheres"] = torch.from_numpy(s).cuda()
    else:
        pts, off, cnt = _clouds(case, seed)
        st["points"] = torch.from_numpy(np.ascontiguousarray(pts)).cuda()
        st["off"] = torch.from_numpy(np.ascontiguousarray(off)).cuda()
        st["cnt"] = torch.from_numpy(np.ascontiguousarray(cnt)).cuda()
        st["index"] = torch.full((int(16 * cnt.sum() + 64 * len(cnt)), 3), -1,
                                 dtype=torch.int32, device="cuda")
    return st


# -------------------------------------------------------------------- pass

def _arrays(simp, dist, nrm):
    return dict(simplices=simp.view(np.int32).reshape(len(simp), 27), distances=dist, normals=nrm)


def run(state):
    case = state["case"]
    kind = case["kind"]
    _use(state["shape"])
    if kind == "pairs":
        out = state["scene"].collide(case["mode"], case["pairs"], out=state["out"])
        return {k: out[k] for k in ("simplices", "distances", "normals")}
    if kind == "host":
        b = state["batch"]
        simp, dist, _ = ogjk.collide_host(ogjk.GJK, b)
        simp2, dist2, nrm = ogjk.collide_host(ogjk.EPA, b, simp, dist)
        return [_arrays(simp, dist, None), _arrays(simp2, dist2, nrm)]
    if kind == "clustered":
        sc = state["scene"]
        if case["rebuild"]:
            sc.build_clusters(state["cluster_min"])
            return sc.collide_contacts(ogjk.GJK_EPA, case["pairs"], out=state["out"],
                                       workspace=state["ws"])["contacts"]
        out = sc.collide(ogjk.GJK_EPA, case["pairs"], out=state["out"])
        return {k: out[k] for k in ("simplices", "distances", "normals")}
    if kind == "serving":
        srv = state["server"]
        tickets = [srv.submit(p, q) for p, q in state["requests"]]
        done = [srv.wait(t)[0] for t in tickets]
        return [_arrays(o["simplices"], o["distances"], o["normals"]) for o in done]
    if kind == "scene_step":
        step = state["step"]
        _, found, out = step(state["poses"])
        return step.bp.pairs, found, out["contacts"]
    if kind == "broad":
        _, found = state["bp"](state["spheres"])
        return state["bp"].pairs, found
    r = ogjk.ingest_hulls(state["points"], state["off"], state["cnt"])
    # the face lists as one index buffer, without the unused capacity between clouds
    nf = r["nfaces"].clamp(min=0).long()
    first = torch.cumsum(nf, 0) - nf
    rows = torch.repeat_interleave(r["face_off"][:-1] - first, nf)
    rows += torch.arange(rows.numel(), device=rows.device)
    state["index"][:rows.numel()] = r["faces"][rows]
    return dict(points=r["points"], faces=state["index"], nfaces=r["nfaces"], com=r["com"],
                inertia_k=r["inertia_k"], volume=r["volume"])


# -------------------------------------------------------------------- work

def _mean_verts(case) -> float:
    """Mean body size: log-uniform integers of nmin..nmax (ellipsoids)."""
    lo, hi = case["nmin"], case["nmax"]
    if lo == hi or case.get("family", gen.ELLIPSOID) != gen.ELLIPSOID:
        return float(hi)
    return (hi + 1 - lo) / math.log((hi + 1) / lo) - 0.5


def work(case) -> dict:
    """Every input read once, every output written once.  Operations: each body
    swept at least twice, once towards its pair's closest feature and once to
    confirm it (5 per vertex and sweep)."""
    kind = case["kind"]
    if kind in ("pairs", "host", "clustered"):
        n, verts = case["pairs"], 2 * case["pairs"] * _mean_verts(case)
        per_body = 12 + 4 if kind == "host" else 16
        out = 108 + 4 + 12
        if kind == "pairs" and case["mode"] == 1:
            out = 108 + 4
        if kind == "clustered" and case["rebuild"]:
            out = 40
        if kind == "host":  # two calls: the second reads and writes the first one's results
            return dict(bytes=2 * (12 * verts + 2 * n * per_body) + n * (112 + 112 + 124),
                        flops=20 * verts)
        return dict(bytes=12 * verts + 2 * n * per_body + n * out, flops=10 * verts)
    if kind == "serving":
        n = case["requests"] * case["kmax"] / 2
        verts = 2 * n * _mean_verts(case)
        scene = 12 * case["bodies"] * _mean_verts(case)
        return dict(bytes=min(12 * verts, scene) + n * (64 + 32 + 124), flops=10 * verts)
    if kind == "scene_step":
        nb, m = case["bodies"], _mean_verts(case)
        # pairs found: neighbours within twice the mean radius (1.5) at the scene's density
        n = nb * nb / 2 * (4 / 3 * math.pi * 3.0 ** 3) / (2 * case["tbox"]) ** 3
        return dict(bytes=nb * (12 * m + 28 + 16 + 16) + n * (8 + 40), flops=10 * 2 * n * m)
    if kind == "broad":
        n = case["objects"]
        return dict(bytes=16 * n + 8 * 0.55 * n, flops=14 * 10 * n)
    n, m = case["clouds"], _mean_verts(case) if case["ellipsoid"] else \
        (case["nmin"] + case["nmax"]) / 2
    faces = n * (2 * m - 4)
    return dict(bytes=n * (12 * m + 12 + 12) + 12 * n * m + 12 * faces + n * (4 + 24 + 8),
                flops=2 * 20 * n * m + 2 * 60 * faces)


# ------------------------------------------------------------ 64-bit values

def _min_norm(P: np.ndarray) -> float:
    """Distance from the origin to the convex hull of the rows of P (Wolfe's
    nearest-point algorithm in float64)."""
    S = [int(np.argmin((P * P).sum(1)))]
    w = np.ones(1)
    x = P[S[0]]
    for _ in range(200):
        k = int(np.argmin(P @ x))
        if x @ x - P[k] @ x <= 1e-15 * max(1.0, float((P[k] * P[k]).sum())) or k in S:
            break
        S.append(k)
        w = np.append(w, 0.0)
        while True:
            Q = P[S]
            m = len(S)
            K = np.zeros((m + 1, m + 1))
            K[0, 1:] = K[1:, 0] = 1.0
            K[1:, 1:] = Q @ Q.T
            rhs = np.zeros(m + 1)
            rhs[0] = 1.0
            a = np.linalg.lstsq(K, rhs, rcond=None)[0][1:]
            if (a > 1e-14).all():
                w = a
                break
            neg = a <= 1e-14
            t = min(1.0, float((w[neg] / np.maximum(w[neg] - a[neg], 1e-300)).min()))
            w = (1 - t) * w + t * a
            keep = w > 1e-14
            if keep.all():
                keep[int(np.argmin(w))] = False
            S = [s for s, kk in zip(S, keep) if kk]
            w = w[keep] / w[keep].sum()
        x = w @ P[S]
        if x @ x <= 1e-26:
            return 0.0  # the origin lies in the hull
    return float(math.sqrt(x @ x))


def _hull_triples(P: torch.Tensor, tri: torch.Tensor):
    """Of the index triples tri of the clouds P (c, n, 3) in float64, which are
    hull faces, and on which side the cloud lies (c, t) each."""
    a, b, c = P[:, tri[:, 0]], P[:, tri[:, 1]], P[:, tri[:, 2]]
    nrm = torch.linalg.cross(b - a, c - a)
    d = nrm @ P.transpose(1, 2) - (nrm * a).sum(-1, keepdim=True)
    k = torch.arange(len(tri), device=P.device)
    for j in range(3):
        d[:, k, tri[:, j]] = 0.0
    return (d <= 0).all(-1), (d >= 0).all(-1), nrm


def _depth(A: torch.Tensor, B: torch.Tensor, tri) -> float:
    """Penetration depth of two overlapping hulls: the least overlap over the
    face normals of both and the cross products of their edges."""
    dirs, edges = [], []
    for P in (A, B):
        t = tri(len(P))
        below, above, nrm = _hull_triples(P[None], t)
        f = (below | above)[0]
        dirs.append(nrm[0][f])
        e = torch.cat([t[f][:, [0, 1]], t[f][:, [1, 2]], t[f][:, [0, 2]]])
        e = torch.unique(torch.sort(e, 1)[0], dim=0)
        edges.append(P[e[:, 1]] - P[e[:, 0]])
    dirs.append(torch.linalg.cross(edges[0][:, None].expand(-1, len(edges[1]), -1),
                                   edges[1][None].expand(len(edges[0]), -1, -1)).reshape(-1, 3))
    D = torch.cat(dirs)
    ln = D.norm(dim=1)
    D = D[ln > 1e-12] / ln[ln > 1e-12, None]
    pa, pb = D @ A.T, D @ B.T
    return float(torch.minimum(pa.max(1)[0] - pb.min(1)[0], pb.max(1)[0] - pa.min(1)[0]).min())


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _triples(dev):
    memo = {}

    def tri(n):
        if n not in memo:
            memo[n] = torch.tensor(list(itertools.combinations(range(n), 3)), device=dev)
        return memo[n]
    return tri


def _distances(batch, depth: bool):
    """Distance of each pair and, with depth, minus the depth of each
    overlapping one."""
    n = batch.n_pairs
    dist = np.zeros(n)
    dev = _device()
    tri = _triples(dev)
    pen = np.zeros(n)
    for i in range(n):
        A = batch.body(int(batch.pa[i])).astype(np.float64)
        B = batch.body(int(batch.pb[i])).astype(np.float64)
        dist[i] = _min_norm((A[:, None] - B[None]).reshape(-1, 3))
        pen[i] = dist[i]
        if depth and dist[i] <= 1e-12:
            pen[i] = -_depth(torch.from_numpy(A).to(dev), torch.from_numpy(B).to(dev), tri)
    return dist, pen


def _mass(pts, off, cnt):
    """Volume, centre of mass and second moments over volume of each cloud's
    hull, all index triples of equally large clouds tried at once."""
    dev = _device()
    tri = _triples(dev)
    n = len(cnt)
    vol = torch.zeros(n, dtype=torch.float64, device=dev)
    com = torch.zeros((n, 3), dtype=torch.float64, device=dev)
    ine = torch.zeros((n, 3), dtype=torch.float64, device=dev)
    P = torch.from_numpy(np.ascontiguousarray(pts)).to(dev).double()
    for k in np.unique(cnt):
        ids = np.nonzero(cnt == k)[0]
        t = tri(int(k))
        step = max(1, 40_000_000 // (len(t) * int(k)))
        for s in range(0, len(ids), step):
            m = torch.from_numpy(ids[s:s + step]).to(dev)
            rows = torch.from_numpy(off[ids[s:s + step]]).to(dev)[:, None] + \
                torch.arange(int(k), device=dev)
            Q = P[rows]
            below, above, _ = _hull_triples(Q, t)
            a, b, c = Q[:, t[:, 0]], Q[:, t[:, 1]], Q[:, t[:, 2]]
            sign = below.double() - above.double()
            dv = sign * (a * torch.linalg.cross(b, c)).sum(-1) / 6.0
            v = dv.sum(1)
            cm = (dv[..., None] * (a + b + c)).sum(1) / (4.0 * v[:, None])
            sq = a * a + b * b + c * c + a * b + a * c + b * c
            vol[m], com[m] = v, cm
            ine[m] = (dv[..., None] / 10.0 * sq).sum(1) / v[:, None] - cm * cm
    return vol, com, ine


def exact(case, seed):
    kind = case["kind"]
    if kind == "pairs" and case["nmax"] <= 64 and case["pairs"] <= 1000:
        dist, pen = _distances(_batch(case, seed), case["mode"] == 3)
        return dict(simplices=None, distances=pen if case["mode"] == 3 else dist, normals=None)
    if kind == "host" and case["nmax"] <= 64 and case["pairs"] <= 1000:
        dist, pen = _distances(_batch(case, seed), True)
        return [dict(simplices=None, distances=dist, normals=None),
                dict(simplices=None, distances=pen, normals=None)]
    if kind == "hulls" and case["nmax"] <= 32:
        pts, off, cnt = _clouds(case, seed)
        vol, com, ine = _mass(pts, off, cnt)
        cloud = np.repeat(np.arange(len(cnt)), cnt)
        centred = pts.astype(np.float64) - com.cpu().numpy()[cloud]
        return dict(points=centred, faces=None, nfaces=None, com=com, inertia_k=ine, volume=vol)
    # the others take minutes in plain 64-bit arithmetic, or give whole numbers only
    return None
