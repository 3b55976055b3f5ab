"""Performance cases of the framework: what a program has it do, through its
public entry points (ray queries on device and host buffers, plain and batched
rendering, the render server), from calls of a thousand rays to frames of
millions of rays and batches of a hundred million samples.

A case is a dict of plain values.  ``kind`` picks the entry point:

``query``   Scene.intersect_device on rays resident in HBM; ``pattern`` is
            ``incoherent`` (secondary rays: origins uniform in the scene's box,
            directions uniform) or ``camera`` (a pinhole frame of ``rays``
            pixels); ``counters`` / ``frames`` ask for the per-ray work
            counters and the shading frames beside the hits
``host``    Scene.intersect on numpy arrays (staged over PCIe)
``plain``   render(): one job, one launch per sample
``batch``   render_batch(): several jobs in one call
``serve``   Server: all jobs submitted at once, then waited for

``scene`` names the geometry: ``sphere`` (one displaced icosphere of
``subdiv``), ``spheres`` (``instances`` transformed copies of it, mirror and
Lambert, over a ground quad), ``plain`` (ground quad and three lat-long
spheres, 4,802 faces; ``normals`` gives the spheres vertex normals and the
scene two point lights).
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from polytope_amd import COUNTER_DTYPE, HIT_DTYPE, Device, Scene, Server, render, render_batch
from polytope_amd import scenes as S


def _query(name, subdiv, rays, pattern, counters=False, frames=False, kind="query"):
    return {"name": name, "kind": kind, "scene": "sphere", "subdiv": subdiv, "rays": rays, "pattern": pattern,
            "counters": counters, "frames": frames}


def _render(name, kind, scene, jobs, width, height, spp, depth, subdiv=0, instances=0, materials=False,
            normals=False, nee=False):
    return {"name": name, "kind": kind, "scene": scene, "subdiv": subdiv, "instances": instances,
            "materials": materials, "normals": normals, "nee": nee, "jobs": jobs, "width": width, "height": height,
            "spp": spp, "depth": depth}


def listed():
    return [
        # picking, line-of-sight and probe queries: a thousand rays, where launches and latency are the cost
        _query("query-smallest", 5, 1000, "incoherent"),
        # an ordinary batch of secondary rays from a renderer's own loop, no round number of them
        _query("query-ragged", 6, 50_021, "incoherent"),
        # the headline workload: 2^21 incoherent rays on 1,310,720 faces
        _query("query-incoherent", 8, 1 << 21, "incoherent"),
        # the largest query: the primary rays of a 4K frame on the same faces
        _query("query-camera-4k", 8, 3840 * 2160, "camera"),
        # analysis and debugging views: hits with work counters and shading frames
        _query("query-counters-frames", 6, 200_003, "incoherent", True, True),
        # a program whose rays and hits live in numpy
        _query("query-host", 7, (1 << 20) + 17, "incoherent", kind="host"),
        # one frame of a small scene at 640x480, 16 samples, depth 5
        _render("render-plain", "plain", "plain", 1, 640, 480, 16, 5),
        # a thumbnail: the smallest batched call
        _render("batch-smallest", "batch", "plain", 1, 64, 48, 4, 4),
        # the batched render workload at 2.7 M faces: 16 jobs from 256x256 to 1920x1080, 16 samples, depth 8
        _render("batch-16-jobs", "batch", "spheres", 16, 1920, 1080, 16, 8, subdiv=6, instances=32),
        # textured Lambert and glossy materials, odd film sizes
        _render("batch-materials", "batch", "spheres", 3, 961, 541, 16, 6, subdiv=6, instances=8, materials=True),
        # next-event estimation to two point lights, smooth normals
        _render("batch-nee-normals", "batch", "plain", 2, 800, 600, 16, 5, normals=True, nee=True),
        # the render server under a burst of requests over one scene
        _render("serve-burst", "serve", "spheres", 8, 1280, 720, 12, 8, subdiv=5, instances=16),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["query", "query", "query", "host", "plain", "batch", "batch", "serve"])
    if kind in ("query", "host"):
        extra = kind == "query" and rng.random() < 0.3
        n = log_int(200, 4_000_000 if kind == "query" and not extra else 800_000)
        case = _query("", rng.randint(3, 8), n, rng.choice(["incoherent", "camera"]),
                      extra, extra and rng.random() < 0.5, kind)
    else:
        small = kind == "plain" or rng.random() < 0.4
        w = log_int(40, 1300)
        case = _render("", kind, "plain" if small else "spheres", 1 if kind == "plain" else rng.randint(1, 6), w,
                       max(9, int(w * rng.uniform(0.4, 1.0))), log_int(1, 16), rng.randint(1, 8),
                       0 if small else rng.randint(3, 6), 0 if small else rng.randint(1, 24),
                       not small and rng.random() < 0.3, small and rng.random() < 0.5, small and rng.random() < 0.4)
        case["nee"] = case["nee"] and case["normals"]
    del case["name"]
    return case


# ---------------------------------------------------------------- geometry and rays

@functools.lru_cache(maxsize=None)
def _device():
    return Device(0)


@functools.lru_cache(maxsize=8)
def _sphere(subdiv):
    v, f = S.icosphere(subdiv, noise=0.05, seed=2)
    return [S.MeshData(v, f)]


@functools.lru_cache(maxsize=8)
def _spheres(subdiv, instances, materials):
    meshes, sky, _ = S.batched_render_workload(subdiv, instances, 1, 1, 1)
    return (S.with_materials(meshes) if materials else meshes), sky


@functools.lru_cache(maxsize=2)
def _plain(normals):
    meshes, _, sky = S.plain_render_scene(1, 64, 48)
    if normals:
        for m in meshes[1:]:
            m.normals = m.verts                 # unit spheres at the origin, transformed into place
    return meshes, sky


_LIGHTS = [((-4.0, 6.0, -3.0), (9000.0, 8500.0, 8000.0)), ((5.0, 4.0, 0.0), (3000.0, 3500.0, 4500.0))]


def _turn(seed):
    """The seed's place on the circle that cameras stand on, 0 to 1."""
    return (seed * 0.6180339887498949) % 1.0


def _rays(case, seed):
    meshes = _sphere(case["subdiv"])
    n = case["rays"]
    if case["pattern"] == "incoherent":
        lo, hi = S.scene_bounds(meshes)
        return S.rays_incoherent(lo, hi, n, seed)
    nx = max(1, int(round(math.sqrt(n * 16 / 9))))
    if n == 3840 * 2160:
        nx = 3840
    ny = -(-n // nx)
    a = 2 * math.pi * _turn(seed)
    cam = S.Camera(S.look_at((2.5 * math.sin(a), 0.3, -2.5 * math.cos(a)), (0.0, 0.0, 0.0)), 44.0, nx, ny)
    return S.rays_coherent(cam, nx, ny)[:n]


def _jobs(case, seed):
    """(camera, spp, depth, seed) per job: film sizes step up to the case's, the cameras stand round the scene."""
    out = []
    n = case["jobs"]
    w0, h0 = min(256, case["width"]), min(256, case["height"])
    for j in range(n):
        t = j / (n - 1) if n > 1 else 1.0
        w, h = round(w0 + (case["width"] - w0) * t), round(h0 + (case["height"] - h0) * t)
        a = 2 * math.pi * (j / n + _turn(seed))
        if case["scene"] == "spheres":
            eye, at = (22.0 * math.cos(a), 9.0, 22.0 * math.sin(a)), (0.0, 2.0, 0.0)
            fov = 55.0
        else:
            eye, at, fov = (6.0 * math.sin(0.3 * a), 2.2, -6.0 * math.cos(0.3 * a)), (0.0, 0.8, 1.5), 60.0
        out.append((S.Camera(S.look_at(eye, at), fov, w, h), case["spp"], case["depth"], (seed + j) & 0x7FFFFFFF))
    return out


# ---------------------------------------------------------------- the passes

def prepare(case, seed):
    dev = _device()
    if case["scene"] == "sphere":
        st = {"kind": case["kind"], "scene": Scene(dev, _sphere(case["subdiv"]))}
        rays = _rays(case, seed)
        n = st["n"] = case["rays"]
        if case["kind"] == "host":
            st["rays"] = rays
            st["hits"] = np.zeros(n, HIT_DTYPE)      # reused between calls, as a loop over batches keeps it
            return st
        st["rays"] = torch.from_numpy(rays).cuda()
        hits = torch.empty((n, 6), dtype=torch.int32, device="cuda")
        st["out"] = {"ids": hits[:, :2], "t": hits.view(torch.float32)[:, 2], "uvw": hits.view(torch.float32)[:, 3:]}
        st["hits_ptr"], st["rays_ptr"] = hits.data_ptr(), st["rays"].data_ptr()
        st["counters_ptr"] = st["frames_ptr"] = 0
        if case["counters"]:
            st["out"]["counters"] = torch.empty((n, 3), dtype=torch.int32, device="cuda")
            st["counters_ptr"] = st["out"]["counters"].data_ptr()
        if case["frames"]:
            st["out"]["frames"] = torch.empty((n, 15), dtype=torch.float32, device="cuda")
            st["frames_ptr"] = st["out"]["frames"].data_ptr()
        return st
    lights = None
    if case["scene"] == "spheres":
        meshes, sky = _spheres(case["subdiv"], case["instances"], case["materials"])
    else:
        meshes, sky = _plain(case["normals"])
        lights = _LIGHTS if case["nee"] else None
    scene = Scene(dev, meshes, sky, lights=lights)
    st = {"kind": case["kind"], "scene": scene, "jobs": [(scene, *j, case["nee"]) for j in _jobs(case, seed)]}
    if case["kind"] == "serve":
        st["server"] = Server(dev, hbm_budget_bytes=16 << 30)
    return st


def run(st):
    kind = st["kind"]
    if kind == "query":
        st["scene"].intersect_device(st["rays_ptr"], st["n"], st["hits_ptr"], st["counters_ptr"], st["frames_ptr"],
                                     torch.cuda.current_stream().cuda_stream)
        return st["out"]
    if kind == "host":
        h = st["scene"].intersect(st["rays"], out=(st["hits"], None))
        return {"mesh": h["mesh"], "face": h["face"], "t": h["t"], "u": h["u"], "v": h["v"], "w": h["w"]}
    if kind == "plain":
        return [render(*j) for j in st["jobs"]]
    if kind == "batch":
        return render_batch(st["jobs"])
    ids = [st["server"].submit(*j) for j in st["jobs"]]
    return [st["server"].wait(i)[0] for i in ids]


def _faces(case):
    if case["scene"] == "sphere":
        return 20 * 4 ** case["subdiv"]
    return 4802 if case["scene"] == "plain" else 20 * 4 ** case["subdiv"] * (case["instances"] + 1) + 2


def work(case):
    """Bytes: every face's vertices once (36 B), each ray in (24 B) and each hit
    out (24 B; counters 12 B, frames 60 B), each film out (12 B a pixel).
    Operations: per ray the slab tests of both children (18 operations a box)
    down one root-to-leaf path of a binary tree and two face tests of 60
    operations; a render traces a pixel's primary ray once and at least one
    bounce ray per sample."""
    faces = _faces(case)
    per_ray = 36 * math.log2(max(2, faces)) + 120
    if case["scene"] == "sphere":
        n = case["rays"]
        return {"bytes": 36 * faces + n * (48 + 12 * case["counters"] + 60 * case["frames"]), "flops": n * per_ray}
    pixels = sum(c.width * c.height for c, *_ in _jobs(case, 0))
    return {"bytes": 36 * faces + 12 * pixels, "flops": pixels * (1 + case["spp"]) * per_ray}


def exact(case, seed):
    """Closest hits by a scan of every face in float64 (Moller-Trumbore), where
    that scan is short.  Films are Monte Carlo estimates whose paths branch on
    every hit, so they have no value in another arithmetic."""
    if case["scene"] != "sphere" or case["rays"] * _faces(case) > 2e10:
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    m = _sphere(case["subdiv"])[0]
    tri = torch.from_numpy(m.verts[m.faces.astype(np.int64)]).to(dev, torch.float64)
    rays = torch.from_numpy(_rays(case, seed)).to(dev, torch.float64)
    n, nf = rays.shape[0], tri.shape[0]
    best = torch.full((n,), math.inf, dtype=torch.float64, device=dev)
    uvw = torch.zeros((n, 3), dtype=torch.float64, device=dev)
    step_f = min(nf, 4096)
    step_r = max(1, (1 << 24) // step_f)
    for r0 in range(0, n, step_r):
        o, d = rays[r0:r0 + step_r, None, :3], rays[r0:r0 + step_r, None, 3:]
        for f0 in range(0, nf, step_f):
            a = tri[None, f0:f0 + step_f, 0]
            e1, e2 = tri[None, f0:f0 + step_f, 1] - a, tri[None, f0:f0 + step_f, 2] - a
            p = torch.linalg.cross(d.expand(-1, e2.shape[1], -1), e2.expand(d.shape[0], -1, -1))
            inv = 1.0 / (p * e1).sum(-1)
            s = o - a
            v = (s * p).sum(-1) * inv
            q = torch.linalg.cross(s, e1.expand(s.shape[0], -1, -1))
            w = (q * d).sum(-1) * inv
            t = (q * e2).sum(-1) * inv
            t = torch.where((v >= 0) & (w >= 0) & (v + w <= 1) & (t > 0), t, math.inf)
            tm, k = t.min(1)
            near = tm < best[r0:r0 + step_r]
            v, w = v.gather(1, k[:, None])[:, 0], w.gather(1, k[:, None])[:, 0]
            uvw[r0:r0 + step_r][near] = torch.stack([1 - v - w, v, w], 1)[near]
            best[r0:r0 + step_r] = torch.where(near, tm, best[r0:r0 + step_r])
    if case["kind"] == "host":
        return {"mesh": None, "face": None, "t": best, "u": uvw[:, 0], "v": uvw[:, 1], "w": uvw[:, 2]}
    out = {"ids": None, "t": best, "uvw": uvw}
    if case["counters"]:
        out["counters"] = None
    if case["frames"]:
        out["frames"] = None
    return out
