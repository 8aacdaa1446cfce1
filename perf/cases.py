"""The work this library is measured on: what its users have it do, through the Python binding.

Every case is a dict of plain values; its "kind" names the entry point it goes through:

  render   HipEngine.render: path-traced frames, or one of the render passes (AOVs)
  adjoint  HipEngine.adjoint: texel gradients of an inverse-rendering step
  batch    BatchRenderer.render: many small scenes in shared launches
  ibl      bake_batch: irradiance maps and prefiltered mips of environment maps
  gl       bake_batch: the GL viewer's cube capture, Riemann irradiance and BRDF table
  rebuild  HipEngine.build_bvh after an edit of the scene, and the pick rays that follow it
  hits     HipEngine.closest_hit: a batch of rays against a scene that stays
  sobol    sobol_fill: a table of Owen-scrambled Sobol samples

Inputs come from the seed: the geometry is stretched per axis, and the camera, the sky's sun,
the rays, the texels and the sample indices are drawn.
"""
import functools
import math
import os
import re

import numpy as np
import torch

from axomae_amd import nova_hip, scenes

PI = math.pi
PASSES = {"path": 0, "normal": nova_hip.INTEGRATOR_PATH | nova_hip.INTEGRATOR_NORMAL, "depth": nova_hip.INTEGRATOR_PATH | nova_hip.INTEGRATOR_DEPTH}
MOST_PATHS = 1920 * 1080 * 64  # paths of the largest listed case


def listed():
    return [
        # the engine's interactive loop on a small scene: one 1-spp frame per call, launches and latency count
        {"name": "frame_box_256", "kind": "render", "scene": "box", "tris": 36, "width": 256, "height": 256, "frames": 1, "depth": 5, "rr": -1,
         "flip": False, "out": "path"},
        # the same loop at display size on the large scene: the engine's per-frame call
        {"name": "frame_1080p", "kind": "render", "scene": "terrain", "tris": 1048576, "width": 1920, "height": 1080, "frames": 1, "depth": 8, "rr": 3,
         "flip": False, "out": "path"},
        # the benchmark's whole job: 64 frames in one call
        {"name": "job_1080p_64", "kind": "render", "scene": "terrain", "tris": 1048576, "width": 1920, "height": 1080, "frames": 64, "depth": 8, "rr": 3,
         "flip": False, "out": "path"},
        # placed meshes (object-space triangle tests), a window of odd size, a few frames per call, image stored bottom-up
        {"name": "frames_placed_odd", "kind": "render", "scene": "placed", "tris": 12000, "width": 1021, "height": 577, "frames": 6, "depth": 6, "rr": -1,
         "flip": True, "out": "path"},
        # a normal buffer for a denoiser or a picker at display size
        {"name": "normals_1080p", "kind": "render", "scene": "terrain", "tris": 1048576, "width": 1920, "height": 1080, "frames": 1, "depth": 1, "rr": -1,
         "flip": False, "out": "normal"},
        # backward of one inverse-rendering step on the benchmark's differentiation scene
        {"name": "adjoint_720p_32", "kind": "adjoint", "tris": 100480, "texels": 512, "width": 1280, "height": 720, "frames": 32, "depth": 4, "rr": -1},
        # a dataset generator: 16 scenes of the benchmark batch's distribution (up to 100k triangles, 512 pixels square)
        {"name": "batch_16_scenes", "kind": "batch", "scenes": 16, "tris": 100000, "side": 512, "depth": 6, "queue": 1 << 24},
        # image-based lighting of 8 maps: Sobol irradiance and 6 prefiltered mips of each, as the benchmark bakes them
        {"name": "bake_ibl_8", "kind": "ibl", "maps": 8, "widest": 4096, "channels": 4, "irradiance": 64, "mip": 256, "mips": 6, "samples": 1024,
         "sobol": True},
        # the viewer's set for one 3-channel map: cube capture, Riemann irradiance, BRDF table
        {"name": "bake_gl_2048", "kind": "gl", "widest": 2048, "channels": 3, "face": 512, "irradiance": 32, "lut": 256, "samples": 1024},
        # an edited scene: the acceleration structure again, and the first rays against it
        {"name": "rebuild_1m", "kind": "rebuild", "tris": 1048576, "rays": 65536},
        # a light-map baker's or simulator's ray batch: camera rays and rays scattered in all directions
        {"name": "hits_262k", "kind": "hits", "tris": 100480, "rays": 262147},
        # a sampler's table over all dimensions, floats and their integers
        {"name": "sobol_4m", "kind": "sobol", "n": 4194301, "dims": 256},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["render", "render", "render", "adjoint", "batch", "ibl", "gl", "rebuild", "hits", "sobol"])
    if kind == "render":
        scene = rng.choice(["box", "terrain", "terrain", "placed"])
        tris = {"box": 36, "placed": _log(rng, 2000, 200000), "terrain": _log(rng, 2000, 1048576)}[scene]
        w, h = _log(rng, 64, 1920), _log(rng, 64, 1080)
        frames = min(_log(rng, 1, 64), max(1, MOST_PATHS // (w * h)))
        depth = rng.randint(1, 8)
        return {"kind": kind, "scene": scene, "tris": tris, "width": w, "height": h, "frames": frames, "depth": depth,
                "rr": rng.choice([-1, min(3, depth)]), "flip": rng.random() < 0.3, "out": rng.choice(["path", "path", "path", "normal", "depth"])}
    if kind == "adjoint":
        return {"kind": kind, "tris": _log(rng, 2000, 100480), "texels": rng.randint(64, 512), "width": _log(rng, 64, 1280), "height": _log(rng, 64, 720),
                "frames": _log(rng, 1, 32), "depth": rng.randint(1, 4), "rr": rng.choice([-1, 1])}
    if kind == "batch":
        return {"kind": kind, "scenes": rng.randint(2, 16), "tris": _log(rng, 1500, 100000), "side": rng.choice([128, 256, 512]), "depth": rng.randint(2, 6),
                "queue": rng.choice([1 << 22, 1 << 23, 1 << 24])}
    if kind == "ibl":
        return {"kind": kind, "maps": rng.randint(1, 8), "widest": rng.choice([512, 1024, 2048, 4096]), "channels": rng.choice([3, 4]),
                "irradiance": rng.randint(12, 64), "mip": _log(rng, 32, 256), "mips": rng.randint(1, 6), "samples": _log(rng, 64, 1024),
                "sobol": rng.random() < 0.5}
    if kind == "gl":
        return {"kind": kind, "widest": rng.choice([512, 1024, 2048]), "channels": rng.choice([3, 4]), "face": _log(rng, 32, 512),
                "irradiance": rng.randint(4, 32), "lut": rng.randint(16, 256), "samples": _log(rng, 128, 1024)}
    if kind == "rebuild":
        return {"kind": kind, "tris": _log(rng, 1500, 1048576), "rays": _log(rng, 64, 65536)}
    if kind == "hits":
        return {"kind": kind, "tris": _log(rng, 1500, 1048576), "rays": _log(rng, 64, 1000000)}
    return {"kind": kind, "n": _log(rng, 1000, 4194301), "dims": rng.choice([2, 42, 256])}


# ------------------------------------------------------------------- inputs

@functools.lru_cache(maxsize=2)
def _terrain(tris):
    """Half the triangles a terrain, half spheres, as the benchmark's scene has them (its own sizes at 1,048,576)."""
    level = 5 if tris >= 500000 else 4 if tris >= 50000 else 3
    return scenes.million_triangles(terrain_cells=max(8, int(math.sqrt(tris / 4))), spheres=max(1, (tris // 2) // (8 * 4 ** level)), sphere_level=level,
                                    sky=(16, 8))


def _stretched(base, rs):
    """A copy of a scene with its geometry stretched per axis by up to 10% each way."""
    s = rs.uniform(0.9, 1.1, 3).astype(np.float32)
    sc = scenes.Scene(materials=list(base.materials), textures=list(base.textures), envmap=base.envmap, inv_P=base.inv_P, inv_V=base.inv_V, name=base.name)
    for m in base.meshes:
        v = (m.vertices.reshape(-1, 3) * s).reshape(-1)
        sc.meshes.append(scenes.Mesh(v, m.normals, m.tangents, m.bitangents, m.uv, m.indices, m.material, m.transform))
    return sc


def _sky(rs, w, h, inten=50.0, size=0.02, channels=4):
    t = scenes.sky_envmap_device(w, h, rs.standard_normal(3) * 0.3 + np.array([0.3, 0.8, 0.3]), inten, size)
    return t if channels == 4 else t.view(-1, 4)[:, :channels].contiguous().view(-1)


def _scene(case, rs):
    w, h = case.get("width", 1920), case.get("height", 1080)
    kind = case.get("scene", "terrain")
    if kind == "box":
        sc = scenes.box_room(seed=int(rs.randint(1 << 30)), width=w, height=h)
        scenes.set_camera(sc, (rs.uniform(-0.3, 0.3), rs.uniform(-0.3, 0.3), 3.6), (0.0, 0.0, 0.0), 40.0, w / h)
        return sc
    if kind == "placed":
        cells = max(8, int(math.sqrt(case["tris"] / 6)))
        level = 3 if case["tris"] < 50000 else 4
        sc = scenes.transformed_scene(seed=int(rs.randint(1 << 30)), terrain_cells=cells, spheres=max(2, 2 * case["tris"] // 3 // (8 * 4 ** level)),
                                      sphere_level=level)
        eye, look, fov = (rs.uniform(-3, 3), rs.uniform(4, 6), 14.0), (0.0, -0.5, 0.0), 55.0
        sky = (256, 128)
    else:
        sc = _stretched(_terrain(case["tris"]), rs)
        eye, look, fov = (rs.uniform(-6, 6), rs.uniform(9, 12), 34.0), (0.0, -2.0, 0.0), 50.0
        sky = (2048, 1024)
    sc.textures[sc.envmap] = scenes.Texture(sky[0], sky[1], 4, _sky(rs, *sky).cpu().numpy())
    scenes.set_camera(sc, eye, look, fov, w / h)
    return sc


def _rays(rs, n):
    """Rays against a terrain scene: a third through a camera's pixels in rows, the rest leaving
    points above the ground in all directions, 64 from each point."""
    cam = n // 3
    wide = max(1, int(math.sqrt(cam * 16 / 9)))
    k = np.arange(cam)
    x, y = (k % wide) / wide * 2 - 1, (k // wide) / max(1, cam // wide) * 2 - 1
    f = math.tan(math.radians(25.0))
    d0 = np.stack([x * f * 16 / 9, -y * f - 0.35, -np.ones(cam)], -1)
    o0 = np.broadcast_to(np.array([rs.uniform(-6, 6), 10.0, 34.0]), (cam, 3))
    m = n - cam
    o1 = np.repeat(rs.uniform((-18, -5, -18), (18, 8, 18), ((m + 63) // 64, 3)), 64, 0)[:m]
    d1 = rs.standard_normal((m, 3))
    o, d = np.concatenate([o0, o1]), np.concatenate([d0, d1])
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return torch.from_numpy(np.concatenate([o, d], 1).astype(np.float32)).cuda()


def _engine(sc):
    eng = nova_hip.HipEngine(0)
    eng.upload(sc)
    eng.build_bvh()
    return eng


def _maps(case, rs, count):
    maps = []
    for k in range(count):
        w = case["widest"] >> (k % 3 if case["widest"] >= 2048 else 0)
        inten = math.exp(rs.uniform(math.log(1e2), math.log(1e4)))
        maps.append((_sky(rs, w, w // 2, inten, 0.002, case["channels"]), (w, w // 2, case["channels"])))
    return maps


def _jobs(case, maps):
    jobs = []
    if case["kind"] == "ibl":
        for m in maps:
            i = case["irradiance"]
            jobs.append((m, i, max(1, i // 2), nova_hip.BAKE_IRRADIANCE_SOBOL if case["sobol"] else nova_hip.BAKE_IRRADIANCE, 0.0))
            for k in range(case["mips"]):
                jobs.append((m, max(2, case["mip"] >> k), max(1, case["mip"] >> (k + 1)), nova_hip.BAKE_PREFILTER, k / 5.0))
    else:
        jobs.append((maps[0], case["face"], case["face"], nova_hip.BAKE_CUBEMAP, 0.0))
        jobs.append((maps[0], case["irradiance"], max(1, case["irradiance"] // 2), nova_hip.BAKE_IRRADIANCE_RIEMANN, 0.0))
        jobs.append((None, case["lut"], case["lut"], nova_hip.BAKE_BRDF_LUT, 0.0))
    return jobs


def prepare(case, seed):
    rs = np.random.RandomState(seed % (1 << 32))
    kind = case["kind"]
    if kind == "render":
        return {"case": case, "eng": _engine(_scene(case, rs)), "start": int(rs.randint(1, 1000))}
    if kind == "adjoint":
        level = 4 if case["tris"] >= 30000 else 3
        n = max(2, case["tris"] // 5 // (8 * 4 ** level))
        sc, alb, rough = scenes.differentiable_scene(seed=int(rs.randint(1 << 30)), width=case["width"], height=case["height"], tex=case["texels"],
                                                     terrain_cells=max(8, int(math.sqrt(0.4 * case["tris"]))), spheres=n, sphere_level=level,
                                                     sky=(256, 128))
        g = torch.Generator(device="cuda").manual_seed(int(rs.randint(1 << 30)))
        dimg = torch.randn((case["height"], case["width"], 4), device="cuda", generator=g) * 0.1  # 2 (image - target) of an L2 loss
        dimg[..., 3] = 0
        return {"case": case, "eng": _engine(sc), "dimg": dimg, "start": 0}
    if kind == "batch":
        jobs = []
        for k in range(case["scenes"]):
            tris, side = int(math.exp(rs.uniform(math.log(1e3), math.log(case["tris"])))), int(case["side"] >> (k % 3))
            spp = (4, 16, 64)[k // 3 % 3]
            jobs.append((_engine(scenes.batch_scene(int(rs.randint(1 << 30)), tris, side)), side, side, spp, case["depth"], {}))
        jobs.sort(key=lambda j: j[1] * j[2] * j[3])
        return {"case": case, "br": nova_hip.BatchRenderer(0), "jobs": jobs, "config": nova_hip.BatchConfig(case["queue"], 6, 4, 1)}
    if kind in ("ibl", "gl"):
        return {"case": case, "jobs": _jobs(case, _maps(case, rs, case.get("maps", 1)))}
    if kind in ("rebuild", "hits"):
        return {"case": case, "eng": _engine(_scene(case, rs)), "rays": _rays(rs, case["rays"])}
    g = torch.Generator(device="cuda").manual_seed(int(rs.randint(1 << 30)))
    idx = torch.randint(-(1 << 31), 1 << 31, (case["n"],), device="cuda", generator=g, dtype=torch.int64).to(torch.int32)
    return {"case": case, "idx": idx, "dims": torch.randint(0, case["dims"], (case["n"],), device="cuda", generator=g, dtype=torch.int32)}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "render":
        return state["eng"].render(case["width"], case["height"], case["frames"], case["depth"], frame_start=state["start"], rr_start=case["rr"],
                                   vertical_invert=case["flip"], integrator_flags=PASSES[case["out"]])
    if kind == "adjoint":
        return state["eng"].adjoint(case["width"], case["height"], case["frames"], case["depth"], state["dimg"], 1.0 / case["frames"], rr_start=case["rr"])
    if kind == "batch":
        return state["br"].render(state["jobs"], state["config"])[0]
    if kind in ("ibl", "gl"):
        return nova_hip.bake_batch(state["jobs"], case["samples"], keep_on_device=True)
    if kind == "rebuild":
        info = state["eng"].build_bvh()
        return [info.binary_nodes, info.binary_depth, info.wide_nodes, info.wide_depth, info.leaves, state["eng"].closest_hit(state["rays"])]
    if kind == "hits":
        return state["eng"].closest_hit(state["rays"])
    return nova_hip.sobol_fill(state["idx"], state["dims"], return_bits=True)


# --------------------------------------------------------------------- work

def _walk_flops(tris):
    """One ray's closest hit: about log2(n) levels of box pairs (24 operations each) and two triangle tests."""
    return 48.0 * max(1.0, math.log2(max(2, tris))) + 2 * 60.0


def work(case):
    kind = case["kind"]
    if kind == "render":
        paths = case["width"] * case["height"] * (case["frames"] if case["out"] == "path" else 1)
        seg = min(1.7, case["depth"] + 1) if case["out"] == "path" else 1.0
        pixels = case["width"] * case["height"]
        return {"bytes": 240.0 * case["tris"] + 48.0 * pixels, "flops": paths * seg * (_walk_flops(case["tris"]) + 800.0)}
    if kind == "adjoint":
        paths = case["width"] * case["height"] * case["frames"]
        return {"bytes": 240.0 * case["tris"] + 16.0 * case["width"] * case["height"] + 32.0 * case["texels"] ** 2,
                "flops": paths * 1.9 * (_walk_flops(case["tris"]) + 2000.0)}
    if kind == "batch":
        paths = sum((case["side"] >> (k % 3)) ** 2 for k in range(case["scenes"])) * 28.0
        return {"bytes": case["scenes"] * 240.0 * case["tris"] / 4 + paths / 28.0 * 32, "flops": paths * 1.7 * (_walk_flops(case["tris"] / 4) + 800.0)}
    if kind in ("ibl", "gl"):
        jobs = _jobs(case, [None] * case.get("maps", 1))
        c = case["channels"]
        widths = [case["widest"] >> (k % 3 if case["widest"] >= 2048 else 0) for k in range(case.get("maps", 1))]
        byte = sum(4.0 * c * w * w / 2 for w in widths)
        flops = 0.0
        for _, ow, oh, k, rough in jobs:
            byte += 4.0 * c * ow * oh * (6 if k == nova_hip.BAKE_CUBEMAP else 1)
            per = 1 if k == nova_hip.BAKE_CUBEMAP or (k == nova_hip.BAKE_PREFILTER and rough == 0.0) else 838 * 210 if k == nova_hip.BAKE_IRRADIANCE_RIEMANN else case["samples"]
            flops += 80.0 * ow * oh * per * (6 if k == nova_hip.BAKE_CUBEMAP else 1)
        return {"bytes": byte, "flops": flops}
    if kind == "rebuild":
        # boxes and centroids in; primitive order, tree and leaf-ordered triangles out; 12 candidate planes per level
        return {"bytes": case["tris"] * (36.0 + 48.0 + 4.0 + 64.0 + 30.0 + 48.0) + 40.0 * case["rays"],
                "flops": case["tris"] * math.log2(max(2, case["tris"])) * 60.0 + case["rays"] * _walk_flops(case["tris"])}
    if kind == "hits":
        return {"bytes": 80.0 * case["tris"] + 40.0 * case["rays"], "flops": case["rays"] * _walk_flops(case["tris"])}
    return {"bytes": 16.0 * case["n"], "flops": 80.0 * case["n"]}


# -------------------------------------------------------------------- exact
# What the entry points compute, in 64 bits. Paths have no such value: one bounce's rounding
# decides what the next one meets, so a path tracer in 64 bits follows other paths.

def _normalize(v):
    return v / v.norm(dim=-1, keepdim=True)


def _cross(a, b):
    return torch.linalg.cross(a, b)


def _atan2(y, x):
    """The path's polynomial atan2 (its definition, up to rounding)."""
    a = (0.99997726, -0.33262347, 0.19354346, -0.11643287, 0.05265332, -0.01172120)
    swap = x.abs() < y.abs()
    r = torch.where(swap, x / y, y / x)
    s = r * r
    p = r * (a[0] + s * (a[1] + s * (a[2] + s * (a[3] + s * (a[4] + s * a[5])))))
    p = torch.where(swap, torch.where(r >= 0, PI / 2, -PI / 2) - p, p)
    return torch.where((x < 0) & (y >= 0), p + PI, torch.where((x < 0) & (y < 0), p - PI, p))


def _acos(x):
    """The path's acos table: 500,000 steps over [-1, 1]."""
    s = ((x + 1) * 250000.0).clamp(0, 499999).floor()
    return torch.acos(s / 500000.0 * 2 - 1)


def _nearest(env, w, h, d):
    u, v = _atan2(d[..., 1], d[..., 0]) / (2 * PI), _acos(d[..., 2]) / PI
    u = torch.where((u > 1) | (u < 0), u - u.floor(), u)
    px = (u * w).floor().long().clamp(0, w) % w
    py = (v * h).floor().long().clamp(0, h) % h
    return env[py, px]


def _sphere(phi, theta):
    return torch.stack([theta.sin() * phi.cos(), theta.sin() * phi.sin(), theta.cos()], -1)


def _texels(ow, oh):
    j, i = torch.meshgrid(torch.arange(oh, device="cuda"), torch.arange(ow, device="cuda"), indexing="ij")
    return i.reshape(-1), j.reshape(-1)


def _radical_inverse(s):
    r = torch.zeros_like(s, dtype=torch.float64)
    for k in range(32):
        r += ((s >> k) & 1).double() * 2.0 ** -(k + 1)
    return r


def _directions():
    """The direction numbers of the 256 dimensions (data: 8,192 words in the repository's table file)."""
    text = open(os.path.join(os.path.dirname(os.path.abspath(nova_hip.__file__)), "csrc", "sobol_table.inc")).read()
    words = [int(x, 16) for x in re.findall(r"0x([0-9a-fA-F]+)", text)]
    if len(words) != 8192:
        words = [int(x) for x in re.findall(r"\b(\d+)[uU]?\b", text)]
    return torch.tensor(words, dtype=torch.int64).view(256, 32).cuda()


def _reverse(x):
    for m, k in ((0x55555555, 1), (0x33333333, 2), (0x0F0F0F0F, 4), (0x00FF00FF, 8), (0x0000FFFF, 16)):
        x = ((x & m) << k) | ((x >> k) & m)
    return x


def _owen_sobol(table, idx, dim):
    """Owen-scrambled Sobol integers (Laine-Karras hash on the reversed bits), int64 holding 32 bits."""
    m32 = 0xFFFFFFFF
    gray = idx ^ (idx >> 1)
    x = torch.zeros_like(gray)
    for b in range(32):
        x ^= torch.where((gray >> b) & 1 != 0, table[dim, b], 0)
    seed = 0xDEADBEEF
    x = _reverse(x)
    mul = lambda a, k: ((a * (k & 0xFFFF)) + (((a * (k >> 16)) & 0xFFFF) << 16)) & m32
    x = x ^ mul(x, 0x3D20ADEA)
    x = (x + seed) & m32
    x = mul(x, (seed >> 16) | 1)
    x = x ^ mul(x, 0x05526C56)
    x = x ^ mul(x, 0x53A22864)
    return _reverse(x)


def _pgc3d(x, y, z):
    m32 = 0xFFFFFFFF
    mul = lambda a, b: ((a * (b & 0xFFFF)) + (((a * (b >> 16)) & 0xFFFF) << 16)) & m32
    k = torch.tensor(1664525, device="cuda", dtype=torch.int64)
    x, y, z = ((mul(v, k) + 1013904223) & m32 for v in (x, y, z))
    for r in range(2):
        x = (x + mul(y, z)) & m32
        y = (y + mul(z, x)) & m32
        if r == 0:
            z = (z + mul(x, y)) & m32
            x, y, z = x ^ (x >> 16), y ^ (y >> 16), z ^ (z >> 16)
    return x.double() / 2.0 ** 32, y.double() / 2.0 ** 32


def _exact_irradiance(env, w, h, ow, oh, samples, sobol):
    i, j = _texels(ow, oh)
    n = _sphere(2 * PI * i.double() / ow, PI * j.double() / oh)
    px = (_atan2(n[:, 1], n[:, 0]) / (2 * PI) * ow).trunc().long() & 0xFFFFFFFF
    py = (_acos(n[:, 2]) / PI * oh).trunc().long()
    right = torch.tensor([1.0, 0, 0], device="cuda", dtype=torch.float64).expand_as(n)
    up = torch.tensor([0, 1.0, 0], device="cuda", dtype=torch.float64).expand_as(n)
    t = torch.where((1 - (right * n).sum(-1, keepdim=True).abs() > 1e-6), _normalize(_cross(right, n)), up)
    b = _cross(n, t)
    table = _directions()
    out = torch.zeros_like(n)
    step = max(1, (1 << 24) // len(i))
    for s0 in range(0, samples, step):
        s = torch.arange(s0, min(samples, s0 + step), device="cuda")[None, :]
        if sobol:
            idx = (j * ow + i)[:, None] * samples + s
            r = [_owen_sobol(table, idx, d).double() / 2.0 ** 32 for d in (0, 1)]
        else:
            r = _pgc3d(px[:, None].expand(-1, s.shape[1]), py[:, None].expand(-1, s.shape[1]), s.expand(len(i), -1))
        st, ct = r[1].sqrt()[..., None], (1 - r[1]).clamp(min=0).sqrt()[..., None]
        d = st * (2 * PI * r[0]).cos()[..., None] * t[:, None] + st * (2 * PI * r[0]).sin()[..., None] * b[:, None] + ct * n[:, None]
        out += _nearest(env, w, h, d)[..., :3].sum(1)
    return out / samples


def _exact_prefilter(env, w, h, ow, oh, samples, rough):
    i, j = _texels(ow, oh)
    n = _normalize(_sphere(2 * PI * i.double() / ow, PI * j.double() / oh))
    if rough == 0.0:
        return _nearest(env, w, h, n)[..., :3]
    a2 = float(np.float32(rough)) ** 4
    z = torch.tensor([0, 0, 1.0], device="cuda", dtype=torch.float64).expand_as(n)
    x = torch.tensor([1.0, 0, 0], device="cuda", dtype=torch.float64).expand_as(n)
    t = _normalize(_cross(torch.where(n[:, 2:].abs() < 0.999, z, x), n))
    b = _cross(n, t)
    out, total = torch.zeros_like(n), torch.zeros_like(n[:, :1])
    step = max(1, (1 << 24) // len(i))
    for s0 in range(0, samples, step):
        s = torch.arange(s0, min(samples, s0 + step), device="cuda")
        xi, ri = s.double() / samples, _radical_inverse(s)
        ct = ((1 - ri) / (1 + (a2 - 1) * ri)).sqrt()
        st = (1 - ct * ct).clamp(min=0).sqrt()
        c, sn = ((2 * PI * xi).cos() * st)[None, :, None], ((2 * PI * xi).sin() * st)[None, :, None]
        hv = _normalize(t[:, None] * c + b[:, None] * sn + n[:, None] * ct[None, :, None])
        l = 2 * (n[:, None] * hv).sum(-1, keepdim=True) * hv - n[:, None]
        wgt = (n[:, None] * l).sum(-1, keepdim=True).clamp(min=0)
        out += (_nearest(env, w, h, l)[..., :3] * wgt).sum(1)
        total += wgt.sum(1)
    return out / total


def _bilinear(env, w, h, d):
    """GL_LINEAR with REPEAT at sphericalToUv(d)."""
    u, v = torch.atan2(-d[..., 2], d[..., 0]) / (2 * PI), torch.acos(d[..., 1].clamp(-1, 1)) / PI
    x, y = u * w - 0.5, v * h - 0.5
    fx, fy = x.floor(), y.floor()
    a, b = (x - fx)[..., None], (y - fy)[..., None]
    i, j = fx.long(), fy.long()
    g = lambda di, dj: env[(j + dj) % h, (i + di) % w][..., :3]
    return (1 - a) * (1 - b) * g(0, 0) + a * (1 - b) * g(1, 0) + (1 - a) * b * g(0, 1) + a * b * g(1, 1)


def _exact_cube(env, w, h, size):
    f = torch.tensor([[-1, 0, 0], [1, 0, 0], [0, -1, 0], [0, 1, 0], [0, 0, 1], [0, 0, -1]], device="cuda", dtype=torch.float64)
    up = torch.tensor([[0, 1, 0], [0, 1, 0], [0, 0, 1], [0, 0, -1], [0, 1, 0], [0, 1, 0]], device="cuda", dtype=torch.float64)
    s = _normalize(_cross(f, up))
    u = _cross(s, f)
    x, y = _texels(size, size)
    nx, ny = ((2 * x + 1) / size - 1).double()[None, :, None], ((2 * y + 1) / size - 1).double()[None, :, None]
    return _bilinear(env, w, h, _normalize(nx * s[:, None] + ny * u[:, None] + f[:, None]))


def _steps(bound):
    a, out = np.float32(0), []
    while a <= np.float32(bound):  # the shader steps in 32 bits: the steps are its definition
        out.append(float(a))
        a = np.float32(a + np.float32(0.0075))
    return torch.tensor(out, device="cuda", dtype=torch.float64)


def _exact_riemann(env, w, h, ow, oh):
    phi, theta = _steps(2 * np.float32(PI)), _steps(np.float32(PI) / np.float32(2))
    i, j = _texels(ow, oh)
    az, po = 2 * PI * (i.double() + 0.5) / ow, PI * (j.double() + 0.5) / oh
    n = torch.stack([az.cos() * po.sin(), po.cos(), -az.sin() * po.sin()], -1)
    y = torch.tensor([0, 1.0, 0], device="cuda", dtype=torch.float64).expand_as(n)
    right = _normalize(_cross(y, n))
    up = _normalize(_cross(n, right))
    out = torch.zeros_like(n)
    ph, th = phi[:, None, None], theta[None, :, None]
    for k in range(len(i)):
        d = _normalize(ph.cos() * th.sin() * right[k] + th.sin() * ph.sin() * up[k] + th.cos() * n[k])
        out[k] = (_bilinear(env, w, h, d) * th.cos() * th.sin()).sum((0, 1))
    return PI * out / (len(phi) * len(theta))


def _exact_lut(ow, oh, samples):
    i, j = _texels(ow, oh)
    ndv, rough = ((i.double() + 0.5) / ow)[:, None], ((j.double() + 0.5) / oh)[:, None]
    s = torch.arange(samples, device="cuda")
    xi, ri = s.double()[None] / samples, _radical_inverse(s)[None]
    g1 = lambda c: c / (c * (1 - rough ** 2 / 2) + rough ** 2 / 2)
    ct = ((1 - ri) / (1 + (rough ** 4 - 1) * ri)).sqrt()
    st = (1 - ct * ct).clamp(min=0).sqrt()
    # with N = z and up = x the tangent is -y and the bitangent x: the half vector's part along V is all that counts
    hx, hz = (2 * PI * xi).sin() * st, ct
    vdh = (1 - ndv ** 2).sqrt() * hx + ndv * hz
    ndl = (2 * vdh * hz - ndv).clamp(min=0)
    vdh = vdh.clamp(min=0)
    vis = torch.where(ndl > 0, g1(ndl) * g1(ndv) * vdh / (hz * ndv), 0.0)
    fc = (1 - vdh) ** 5
    return torch.stack([((1 - fc) * vis).mean(1), (fc * vis).mean(1)], -1)


def _exact_bakes(state):
    case, out = state["case"], []
    for m, ow, oh, kind, rough in state["jobs"]:
        if kind == nova_hip.BAKE_BRDF_LUT:
            out.append(_exact_lut(ow, oh, case["samples"]).view(oh, ow, 2))
            continue
        w, h, c = m[1]
        env = m[0].double().view(h, w, c)
        if kind == nova_hip.BAKE_CUBEMAP:
            r = _exact_cube(env, w, h, ow).view(6, oh, ow, 3)
        elif kind == nova_hip.BAKE_IRRADIANCE_RIEMANN:
            r = _exact_riemann(env, w, h, ow, oh).view(oh, ow, 3)
        elif kind == nova_hip.BAKE_PREFILTER:
            r = _exact_prefilter(env, w, h, ow, oh, case["samples"], rough).view(oh, ow, 3)
        else:
            r = _exact_irradiance(env, w, h, ow, oh, case["samples"], kind == nova_hip.BAKE_IRRADIANCE_SOBOL).view(oh, ow, 3)
        out.append(torch.cat([r, torch.zeros_like(r[..., :c - 3])], -1))
    return out


def _exact_hits(eng, rays):
    """Every ray against every triangle: side products of the ray and the three edges, then the nearest t."""
    tri = []
    for m in eng.scene.meshes:
        v = torch.from_numpy(m.vertices).cuda().double().view(-1, 3)
        tri.append(v[torch.from_numpy(m.indices.astype(np.int64)).cuda()].view(-1, 3, 3))
    tri = torch.cat(tri)
    best = torch.full((len(rays),), math.inf, device="cuda", dtype=torch.float64)
    uv = torch.zeros((len(rays), 2), device="cuda", dtype=torch.float64)
    o, d = rays[:, :3].double(), rays[:, 3:].double()
    line = torch.cat([d, _cross(o, d)], 1)
    for t0 in range(0, len(tri), 4096):
        a, b, c = tri[t0:t0 + 4096].unbind(1)
        edge = [torch.cat([_cross(p, q), q - p], 1) for p, q in ((b, c), (c, a), (a, b))]
        n = _cross(b - a, c - a)
        for r0 in range(0, len(rays), 8192):
            r = slice(r0, min(len(rays), r0 + 8192))
            wa, wb, wc = (line[r] @ e.T for e in edge)
            det = d[r] @ n.T
            t = ((a * n).sum(1) - o[r] @ n.T) / det
            inside = ((wa >= 0) & (wb >= 0) & (wc >= 0)) | ((wa <= 0) & (wb <= 0) & (wc <= 0))
            t = torch.where(inside & (t >= 1e-6) & (det != 0), t, math.inf)
            tm, k = t.min(1)
            total = wa + wb + wc
            pick = lambda x: (x / total).gather(1, k[:, None])
            near = tm < best[r]
            best[r] = torch.where(near, tm, best[r])
            uv[r] = torch.where(near[:, None], torch.cat([pick(wb), pick(wc)], 1), uv[r])
    hit = torch.isfinite(best)
    return torch.cat([torch.where(hit, best, 0.0)[:, None], torch.where(hit[:, None], uv, 0.0)], 1)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("render", "adjoint", "batch"):
        return None
    if kind in ("rebuild", "hits") and case["rays"] * case["tris"] > 4e10:
        return None
    state = prepare(case, seed)
    if kind in ("ibl", "gl"):
        return _exact_bakes(state)
    if kind in ("rebuild", "hits"):
        hits = (None, _exact_hits(state["eng"], state["rays"]))
        return hits if kind == "hits" else [None] * 5 + [hits]
    idx, dims = state["idx"].long() & 0xFFFFFFFF, state["dims"].long()
    return _owen_sobol(_directions(), idx, dims).double() / 2.0 ** 32, None
