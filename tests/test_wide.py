"""The four-wide traversal (polytope_amd/csrc/wide.h) against the binary one.

CPU: the headers' tests and the host builder, compiled for the host, visit the
leaves of the reference's traversal in its order (tests/wide_check.cpp).  GPU:
queries for hits and frames take the four-wide form and queries for counters
the binary one, so both answers for the same rays must be equal bit for bit:
scenes of one face, of leaves past two faces and of none that a small LDS stack
holds, sizes around a wave and a block, and rays with zero, negative-zero,
tiny, infinite and NaN components and origins on the vertices' planes."""
from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

from polytope_amd import scenes as S

ROOT = Path(__file__).resolve().parents[1]


def test_wide_traversal_visits_the_reference_leaves(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(hipcc).exists():
        pytest.skip("hipcc not found")
    exe = tmp_path / "wide_check"
    csrc = ROOT / "polytope_amd" / "csrc"
    subprocess.run([hipcc, "-O2", "-std=c++17", "-ffp-contract=off", "-x", "hip", "--offload-arch=gfx950",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                    f"-I{csrc}", f"-I{ROOT / 'include'}", str(ROOT / "tests" / "wide_check.cpp"),
                    *(str(csrc / f) for f in ("wide_build.cpp", "bvh_build.cpp", "scene.cpp")), "-lpthread",
                    "-o", str(exe)], check=True, capture_output=True, timeout=300)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout
    assert " 0 mismatches" in out.stdout


def _edge_rays(rays: np.ndarray, verts: np.ndarray) -> np.ndarray:
    """Every second ray of ``rays`` with components that make slab values infinite or NaN."""
    r = rays.copy()
    rng = np.random.default_rng(3)
    n = len(r)
    for a in range(3):
        k = rng.integers(0, 24, n)
        for i, x in enumerate((0.0, -0.0, 1e-39, -1e-30, 1e25)):
            r[(k == i) & (np.arange(n) % 2 == 1), 3 + a] = x
        on = (k > 18) & (np.arange(n) % 2 == 1)
        r[on, a] = verts[rng.integers(0, len(verts), on.sum()), a]
    k = np.arange(n) % 301
    for i, (j, x) in enumerate(((3, np.nan), (4, np.inf), (0, np.nan), (1, -np.inf), (2, 1e25))):
        r[k == i, j] = x
    r[k == 7, 3:] = 0.0
    return r


def _scene(name: str):
    if name == "face":
        v = np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0.5]], np.float32)
        return v, np.array([[0, 1, 2]], np.uint32)
    if name == "duplicates":                     # leaves of many faces: the same three triangles 20 times
        v, f = S.icosphere(0, noise=0.0, seed=1)
        return v, np.concatenate([f[:3]] * 20)
    if name == "slivers":
        return S.sliver_grid(48, 2.0)
    return S.icosphere(6, noise=0.05, seed=2)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["face", "duplicates", "slivers", "sphere"])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 257, 60_001])
def test_wide_and_binary_queries_agree(name, n):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from polytope_amd import Device, Scene
    verts, faces = _scene(name)
    meshes = [S.MeshData(verts, faces)]
    lo, hi = S.scene_bounds(meshes)
    rays = _edge_rays(S.rays_incoherent(np.asarray(lo) - 0.2, np.asarray(hi) + 0.2, n, 9), verts)
    dev = Device(0)
    scene = Scene(dev, meshes)
    r = torch.from_numpy(rays).cuda()
    stream = torch.cuda.current_stream().cuda_stream

    def query(counters: bool, frames: bool):
        h = torch.full((n, 6), -7, dtype=torch.int32, device="cuda")
        c = torch.zeros((n, 3), dtype=torch.int32, device="cuda")
        f = torch.full((n, 15), -7.0, dtype=torch.float32, device="cuda")
        scene.intersect_device(r.data_ptr(), n, h.data_ptr(), c.data_ptr() if counters else 0,
                               f.data_ptr() if frames else 0, stream)
        torch.cuda.synchronize()
        return h.cpu().numpy(), f.cpu().numpy().view(np.uint32)

    try:
        hits, frames = query(True, True)
        for lds, leaf in ((0, 0), (8, 1), (24, 64)):
            dev.set_tuning(lds_stack=lds, leaf_lanes=leaf)
            assert np.array_equal(query(False, False)[0], hits)
            wide = query(False, True)
            assert np.array_equal(wide[0], hits)
            assert np.array_equal(wide[1], frames)
    finally:
        scene.close()
        dev.close()


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["plain", "textured", "nee"])
@pytest.mark.parametrize("size", [(1, 1, 1, 1), (37, 29, 5, 4), (131, 130, 2, 3)])
def test_render_forms_agree(case, size):
    """ptx_render as a batch of one and as one launch per sample, over one
    pixel, a ragged film and one with the debug pixel: the same bits."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from polytope_amd import Device, Scene, _abi, render
    w, h, spp, depth = size
    lights = [((0.0, 5.0, -2.0), (4000.0, 4000.0, 4000.0))] if case == "nee" else None
    if case == "textured":
        meshes, cam, sky = S.textured_render_scene(1, w, h)
    else:
        meshes, cam, sky = S.plain_render_scene(1, w, h)
    dev = Device(0)
    scene = Scene(dev, meshes, sky, lights=lights)
    try:
        film = render(scene, cam, spp, depth, 3, nee=bool(lights))
        for form in (_abi.PLAIN_CACHED, _abi.PLAIN_RETRACE):
            dev.set_tuning(plain_primary=form)
            assert np.array_equal(render(scene, cam, spp, depth, 3, nee=bool(lights)).view(np.uint32),
                                  film.view(np.uint32))
    finally:
        scene.close()
        dev.close()


@pytest.mark.gpu
@pytest.mark.parametrize("extra", [-1, 0, 1, 64])
def test_launches_with_and_without_the_batch_counter_agree(extra):
    """Ids that one block per CU deals out in batches of 64 without the
    counter, which no kernel clears then, and the first that need it, each
    behind a launch that leaves the counter's scratch dirty."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from polytope_amd import Device, Scene
    verts, faces = _scene("slivers")
    meshes = [S.MeshData(verts, faces)]
    n = 4 * 64 * torch.cuda.get_device_properties(0).multi_processor_count + extra
    lo, hi = S.scene_bounds(meshes)
    rays = S.rays_incoherent(np.asarray(lo) - 0.2, np.asarray(hi) + 0.2, 3 * n, 5)
    dev = Device(0)
    scene = Scene(dev, meshes)
    dev.set_tuning(blocks_per_cu=1)
    r = torch.from_numpy(rays).cuda()
    stream = torch.cuda.current_stream().cuda_stream

    def query(m: int, counters: bool):
        h = torch.full((m, 6), -7, dtype=torch.int32, device="cuda")
        c = torch.zeros((m, 3), dtype=torch.int32, device="cuda")
        scene.intersect_device(r.data_ptr(), m, h.data_ptr(), c.data_ptr() if counters else 0, 0, stream)
        torch.cuda.synchronize()
        return h.cpu().numpy()

    try:
        whole = query(3 * n, True)
        for _ in range(2):
            assert np.array_equal(query(3 * n, False), whole)
            assert np.array_equal(query(n, False), whole[:n])
    finally:
        scene.close()
        dev.close()


@pytest.mark.gpu
def test_batch_tables_grow_and_films_span_rounds():
    """Batches of 2, 70 and 2 jobs over one engine (its tables grow once) whose
    films are summed over several rounds and in one: the films of one launch
    per sample."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from polytope_amd import Device, Scene, _abi, render, render_batch
    dev = Device(0)
    scenes, jobs, want = [], [], []
    try:
        dev.set_tuning(plain_primary=_abi.PLAIN_CACHED)
        for w, h in ((17, 9), (32, 8)):
            meshes, cam, sky = S.plain_render_scene(1, w, h)
            scenes.append(Scene(dev, meshes, sky))
            jobs.append((scenes[-1], cam, 5, 3, 3))
            want.append(render(*jobs[-1]).view(np.uint32))
        for paths in (0, 700):
            dev.set_tuning(paths_per_wave=paths)
            for n in (2, 70, 2):
                for i, film in enumerate(render_batch([jobs[i % 2] for i in range(n)])):
                    assert np.array_equal(film.view(np.uint32), want[i % 2])
    finally:
        for s in scenes:
            s.close()
        dev.close()


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [1e-15, 4e15, 2e16, 3e17])
def test_scenes_at_the_edges_of_the_wide_ranges_agree(scale):
    """Extents far below one, just inside and past the limit of the four-wide
    test's range, with directions whose reciprocals lie on both sides of it."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from polytope_amd import Device, Scene
    verts, faces = _scene("sphere")
    lo, hi = S.scene_bounds([S.MeshData(verts, faces)])
    n = 4001
    rays = S.rays_incoherent(np.asarray(lo) - 0.2, np.asarray(hi) + 0.2, n, 9)
    rays[:, :3] *= np.float32(scale)
    for i, d in enumerate((3e-16, -5e-17, 1e-18, 1e20)):
        rays[i::9, 3 + i % 3] = d
    meshes = [S.MeshData((verts * np.float32(scale)).astype(np.float32), faces)]
    dev = Device(0)
    scene = Scene(dev, meshes)
    r = torch.from_numpy(rays).cuda()
    stream = torch.cuda.current_stream().cuda_stream
    out = []
    try:
        for counters in (True, False):
            h = torch.full((n, 6), -7, dtype=torch.int32, device="cuda")
            c = torch.zeros((n, 3), dtype=torch.int32, device="cuda")
            scene.intersect_device(r.data_ptr(), n, h.data_ptr(), c.data_ptr() if counters else 0, 0, stream)
            torch.cuda.synchronize()
            out.append(h.cpu().numpy())
        assert np.array_equal(*out)
    finally:
        scene.close()
        dev.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 64, 65, 20_011])
def test_counters_do_not_depend_on_the_gathering(n):
    """Hits, counters and frames of the binary form with every lane, one lane
    and the defaults gathered at leaves and at refills, over node and window
    records: the same words, and the hits of the four-wide form."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from polytope_amd import Device, Scene, _abi
    verts, faces = _scene("sphere")
    meshes = [S.MeshData(verts, faces)]
    lo, hi = S.scene_bounds(meshes)
    rays = _edge_rays(S.rays_incoherent(np.asarray(lo) - 0.2, np.asarray(hi) + 0.2, n, 9), verts)
    dev = Device(0)
    scene = Scene(dev, meshes)
    r = torch.from_numpy(rays).cuda()
    stream = torch.cuda.current_stream().cuda_stream

    def query(counters: bool):
        h = torch.full((n, 6), -7, dtype=torch.int32, device="cuda")
        c = torch.full((n, 3), -7, dtype=torch.int32, device="cuda")
        f = torch.full((n, 15), -7, dtype=torch.int32, device="cuda")
        scene.intersect_device(r.data_ptr(), n, h.data_ptr(), c.data_ptr() if counters else 0, f.data_ptr(), stream)
        torch.cuda.synchronize()
        return [x.cpu().numpy() for x in (h, c, f)]

    try:
        first = query(True)
        for windows in (_abi.WINDOWS_OFF, _abi.WINDOWS_ON):
            for lanes in (1, 64):
                dev.set_tuning(leaf_lanes=lanes, refill_lanes=lanes, ray_windows=windows, blocks_per_cu=1)
                for a, b in zip(query(True), first):
                    assert np.array_equal(a, b)
        dev.set_tuning(leaf_lanes=64, refill_lanes=64)
        wide = query(False)
        assert np.array_equal(wide[0], first[0]) and np.array_equal(wide[2], first[2])
    finally:
        scene.close()
        dev.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n", [(1 << 18) - 1, (1 << 19) - 1, (1 << 19) + 33, 5 * (1 << 18) + 1])
def test_host_queries_in_parts_agree(n):
    """Host queries of one part, two and four (sizes around where they split),
    with and without counters: the words of the device query."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from polytope_amd import Device, Scene
    verts, faces = _scene("sphere")
    meshes = [S.MeshData(verts, faces)]
    lo, hi = S.scene_bounds(meshes)
    rays = S.rays_incoherent(np.asarray(lo) - 0.2, np.asarray(hi) + 0.2, n, 9)
    dev = Device(0)
    scene = Scene(dev, meshes)
    r = torch.from_numpy(rays).cuda()
    h = torch.full((n, 6), -7, dtype=torch.int32, device="cuda")
    c = torch.zeros((n, 3), dtype=torch.int32, device="cuda")
    try:
        scene.intersect_device(r.data_ptr(), n, h.data_ptr(), c.data_ptr(), 0, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        for _ in range(2):
            hits, cnt = scene.intersect(rays, counters=True)
            assert np.array_equal(hits.view(np.int32).reshape(n, 6), h.cpu().numpy())
            assert np.array_equal(cnt.view(np.int32).reshape(n, 3), c.cpu().numpy())
            assert np.array_equal(scene.intersect(rays).view(np.int32).reshape(n, 6), h.cpu().numpy())
    finally:
        scene.close()
        dev.close()


def test_rays_without_finite_directions_step_over_the_wide_tree(tmp_path):
    """No ray starts over the binary records: a lane whose direction is zero or
    NaN traced there alone held its wave for the whole of it."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(hipcc).exists():
        pytest.skip("hipcc not found")
    exe = tmp_path / "wide_hard_check"
    csrc = ROOT / "polytope_amd" / "csrc"
    subprocess.run([hipcc, "-O2", "-std=c++17", "-ffp-contract=off", "-x", "hip", "--offload-arch=gfx950",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                    f"-I{csrc}", f"-I{ROOT / 'include'}", str(ROOT / "tests" / "wide_hard_check.cpp"),
                    *(str(csrc / f) for f in ("wide_build.cpp", "bvh_build.cpp", "scene.cpp")), "-lpthread",
                    "-o", str(exe)], check=True, capture_output=True, timeout=300)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout
    assert " 0 mismatches" in out.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("share", [1, 2, 64])
def test_idle_lanes_marked_by_their_directions_agree(share):
    """Every share-th ray without a direction, one in sixteen of those NaN or
    infinite, as a program marks the idle lanes of a batch: the hits of the
    binary form."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from polytope_amd import Device, Scene
    verts, faces = _scene("sphere")
    meshes = [S.MeshData(verts, faces)]
    n = 20_011
    lo, hi = S.scene_bounds(meshes)
    rays = S.rays_incoherent(lo, hi, n, 9)
    rays[::share, 3:] = 0.0
    rays[::2 * share, 3] = -0.0
    rays[::16 * share, 4] = np.nan
    rays[7 * share::16 * share, 5] = -np.inf
    dev = Device(0)
    scene = Scene(dev, meshes)
    r = torch.from_numpy(rays).cuda()
    stream = torch.cuda.current_stream().cuda_stream
    out = []
    try:
        for counters in (True, False):
            h = torch.full((n, 6), -7, dtype=torch.int32, device="cuda")
            c = torch.zeros((n, 3), dtype=torch.int32, device="cuda")
            f = torch.full((n, 15), -7.0, dtype=torch.float32, device="cuda")
            scene.intersect_device(r.data_ptr(), n, h.data_ptr(), c.data_ptr() if counters else 0, f.data_ptr(), stream)
            torch.cuda.synchronize()
            out.append((h.cpu().numpy(), f.cpu().numpy()))
        (h0, f0), (h1, f1) = out
        assert np.array_equal(h0[:, :2], h1[:, :2])
        assert np.array_equal(h0[:, 2:].view(np.float32), h1[:, 2:].view(np.float32), equal_nan=True)
        assert np.array_equal(f0, f1, equal_nan=True)
    finally:
        scene.close()
        dev.close()


def test_rays_in_the_planes_of_flat_leaves_step_over_the_wide_tree(tmp_path):
    """Under a direction component of -0 a flat leaf at the origin's coordinate
    is visited or not by the boxes above it, without a second traversal."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(hipcc).exists():
        pytest.skip("hipcc not found")
    exe = tmp_path / "wide_flat_check"
    csrc = ROOT / "polytope_amd" / "csrc"
    subprocess.run([hipcc, "-O2", "-std=c++17", "-ffp-contract=off", "-x", "hip", "--offload-arch=gfx950",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                    f"-I{csrc}", f"-I{ROOT / 'include'}", str(ROOT / "tests" / "wide_flat_check.cpp"),
                    *(str(csrc / f) for f in ("wide_build.cpp", "bvh_build.cpp", "scene.cpp")), "-lpthread",
                    "-o", str(exe)], check=True, capture_output=True, timeout=300)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout
    assert " 0 mismatches" in out.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("side", [1, 6, 40])
@pytest.mark.parametrize("n", [65, 20_011])
def test_rays_in_the_plane_of_a_floor_agree(side, n):
    """A floor of 2 side^2 triangles (face records made by the host, from 40 on
    by the device) below a sphere, rays that start on it with -0 and 0 as their
    vertical component and rays from its corners: the words of the binary form."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from polytope_amd import Device, Scene
    g = np.linspace(-4, 4, side + 1, dtype=np.float32)
    x, z = np.meshgrid(g, g)
    floor = np.stack([x, 0 * x, z], -1).reshape(-1, 3)
    i = np.arange(side * (side + 1)).reshape(side, side + 1)[:, :side].ravel()
    quads = np.concatenate([np.stack([i, i + 1, i + side + 1], 1), np.stack([i + 1, i + side + 2, i + side + 1], 1)])
    v, f = S.icosphere(2, radius=1.0, center=(0.0, 1.0, 0.0), noise=0.05, seed=3)
    meshes = [S.MeshData(floor, quads.astype(np.uint32)), S.MeshData(v, f)]
    rays = S.rays_incoherent((-5.0, -0.5, -5.0), (5.0, 2.0, 5.0), n, 9)
    rays[::2, 1] = 0.0
    rays[::2, 4] = -0.0
    rays[::6, 4] = 0.0
    rays[::10, 0] = -4.0
    rays[::14, 3] = -0.0
    rays[::22, 3:] = -0.0
    dev = Device(0)
    scene = Scene(dev, meshes)
    r = torch.from_numpy(rays).cuda()
    stream = torch.cuda.current_stream().cuda_stream
    out = []
    try:
        for counters in (True, False):
            h = torch.full((n, 6), -7, dtype=torch.int32, device="cuda")
            c = torch.zeros((n, 3), dtype=torch.int32, device="cuda")
            scene.intersect_device(r.data_ptr(), n, h.data_ptr(), c.data_ptr() if counters else 0, 0, stream)
            torch.cuda.synchronize()
            out.append(h.cpu().numpy())
        assert np.array_equal(out[0][:, :2], out[1][:, :2])
        assert np.array_equal(out[0][:, 2:].view(np.float32), out[1][:, 2:].view(np.float32), equal_nan=True)
    finally:
        scene.close()
        dev.close()


@pytest.mark.gpu
@pytest.mark.parametrize("copies", [1, 2, 3, 4, 7])
@pytest.mark.parametrize("widen", [0.0, 0.01])
def test_leaves_of_any_number_of_faces_agree(copies, widen):
    """Leaves of one face to more than two steps' worth, whose boxes are their
    corners' or (in a tree the caller brings) wider: the words of the binary
    form, in queries and in a render."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from polytope_amd import Device, Scene, _abi, build_bvh, render
    verts, faces = S.icosphere(2, noise=0.05, seed=2)
    meshes = [S.MeshData(verts, np.concatenate([faces] * copies))]
    nodes, pairs = build_bvh(meshes)
    nodes["p0"] -= np.float32(widen)
    nodes["p1"] += np.float32(widen)
    n = 5003
    lo, hi = S.scene_bounds(meshes)
    rays = _edge_rays(S.rays_incoherent(np.asarray(lo) - 0.2, np.asarray(hi) + 0.2, n, 9), verts)
    dev = Device(0)
    scene = Scene(dev, meshes, (10.0, 20.0, 30.0), bvh=(nodes, pairs))
    r = torch.from_numpy(rays).cuda()
    stream = torch.cuda.current_stream().cuda_stream
    out = []
    try:
        for counters in (True, False):
            h = torch.full((n, 6), -7, dtype=torch.int32, device="cuda")
            c = torch.zeros((n, 3), dtype=torch.int32, device="cuda")
            f = torch.full((n, 15), -7.0, dtype=torch.float32, device="cuda")
            scene.intersect_device(r.data_ptr(), n, h.data_ptr(), c.data_ptr() if counters else 0, f.data_ptr(), stream)
            torch.cuda.synchronize()
            out.append((h.cpu().numpy(), f.cpu().numpy()))
        (h0, f0), (h1, f1) = out
        assert np.array_equal(h0[:, :2], h1[:, :2])
        assert np.array_equal(h0[:, 2:].view(np.float32), h1[:, 2:].view(np.float32), equal_nan=True)
        assert np.array_equal(f0, f1, equal_nan=True)
        cam = S.Camera(S.look_at((0.3, 0.5, -2.5), (0.0, 0.0, 0.0)), 50.0, 40, 30)
        films = []
        for form in (dict(), dict(plain_primary=_abi.PLAIN_CACHED), dict(render_mode=_abi.RENDER_WAVEFRONT)):
            dev.set_tuning(**form)
            films.append(render(scene, cam, 3, 3, 5).view(np.uint32))
        assert np.array_equal(films[0], films[1]) and np.array_equal(films[0], films[2])
    finally:
        scene.close()
        dev.close()
