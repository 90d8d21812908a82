"""The work a user of the library has it do, as timed cases: ray picks on one
surface, batches of ray-patch pairs and of patch evaluations, closest and any
hits of ray sets, batched queries over several scenes, shaded ray queries, and
rendered frames (plain and sampled).

listed() names the cases; draw() gives more of the same ranges; prepare()
makes what a program holds before the call (a resident scene, device buffers),
run() is one pass through the public entry points, work() what a pass cannot
do without, tolerance() how far a result may be off, exact() the result in 64
bits where the path's outputs have one.
"""
from __future__ import annotations

import dataclasses
import math
import os

import numpy as np
import torch

import cgspline_amd as cgs
from cgspline_amd import scenes

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_SCENE_DIR = os.path.join(_ROOT, "tests", "golden", "assets", "scenes")

# cgs_patch_eval's kinds (CGS_EVAL_*, include/cgs.h)
_KINDS = ("interpolate", "interpolate_mat", "derivative_u", "derivative_v", "derivative_u_mat", "derivative_v_mat",
          "normal", "normal_mat")

_ctx = None


def _context() -> cgs.Context:
    """The program's one context on the GPU."""
    global _ctx
    if _ctx is None:
        torch.cuda.init()
        _ctx = cgs.Context(0)
    return _ctx


def listed():
    return [
        # a click or a short drag on one surface: 64 rays against its patches,
        # where launches and waits are the time
        dict(name="pick_64", kind="pick", patches=256, rays=64, any=False),
        # a program's own (ray, patch) pairs clipped in one call
        dict(name="clip_200k", kind="clip", n=200_000),
        # the same by subdivision, the other leaf method
        dict(name="subdivide_30k", kind="subdivide", n=30_001),
        # normals of a million patches at one (u, v) each (tessellation, offsets)
        dict(name="eval_normal_1m", kind="eval", what="normal", n=1_000_003),
        # patches cut to parameter ranges (trimming, refinement)
        dict(name="subpatch_300k", kind="subpatch", n=300_001),
        # camera rays of a full HD view against 64 closed surfaces, closest hits
        dict(name="closest_hd", kind="closest", scene="closed", size=64, rays=1920 * 1080),
        # scattered rays in a scene of 512 displaced grids (131,072 patches): occlusion
        dict(name="any_random", kind="any", scene="displaced", size=512, rays=777_777),
        # uneven closest and occlusion queries over 12 resident scenes, one captured launch
        dict(name="batch_12", kind="batch", scenes=12, patches=100_000, rays=1 << 20),
        # a small frame of one 256-patch height field with shadows: the interactive size
        dict(name="frame_heightfield_256", kind="render", scene="heightfield", size=256, width=256, height=256, depth=0,
             samples=0),
        # a scene file of many lights: tea sets, 51 point lights, reflection depth 6, full HD
        dict(name="frame_tea_hd", kind="render", scene="Test152", size=0, width=1920, height=1080, depth=6, samples=0),
        # the million-patch frame: 4096 displaced grids, shadows and one reflection bounce
        dict(name="frame_displaced_2048", kind="render", scene="displaced", size=4096, width=2048, height=2048, depth=1,
             samples=0),
        # the Monte Carlo render, a smaller frame at 4 camera rays per pixel
        dict(name="frame_sampled_768", kind="render", scene="displaced", size=1024, width=768, height=768, depth=1,
             samples=4),
    ]


def _log(rng, lo, hi) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pick", "clip", "subdivide", "eval", "subpatch", "closest", "any", "batch", "shade", "render",
                       "render"])
    if kind == "pick":
        n = rng.randint(4, 40)
        any_hit = rng.random() < 0.3
        return dict(kind=kind, patches=n * n, rays=_log(rng, 64 if any_hit else 1, 300_000), any=any_hit)
    if kind == "clip":
        return dict(kind=kind, n=_log(rng, 1, 1_000_000))
    if kind == "subdivide":
        return dict(kind=kind, n=_log(rng, 1, 100_000))
    if kind == "eval":
        return dict(kind=kind, what=rng.choice(_KINDS), n=_log(rng, 1, 2_000_000))
    if kind == "subpatch":
        return dict(kind=kind, n=_log(rng, 1, 1_000_000))
    scene = rng.choice(["heightfield", "closed", "displaced", "displaced"])
    size = {"heightfield": 256, "closed": rng.randint(1, 64), "displaced": _log(rng, 16, 2048)}[scene]
    if kind in ("closest", "any"):
        # (few scattered rays would all miss)
        return dict(kind=kind, scene=scene, size=size, rays=_log(rng, 300 if kind == "closest" else 5_000, 2_000_000))
    if kind == "shade":
        return dict(kind=kind, scene=scene, size=size, rays=_log(rng, 300, 500_000), depth=rng.randint(0, 2))
    if kind == "batch":
        return dict(kind=kind, scenes=rng.randint(2, 16), patches=_log(rng, 2_000, 100_000),
                    rays=_log(rng, 4_096, 1 << 20))
    if rng.random() < 0.25:
        scene, size = rng.choice(["Teaset01", "Teaset02", "teaset", "Test32", "Test56", "Test104"]), 0
    samples = rng.choice([0, 0, 0, 2, 4])
    return dict(kind="render", scene=scene, size=size, width=_log(rng, 40, 1600), height=_log(rng, 40, 1200),
                depth=rng.randint(0, 3), samples=samples)


# --- inputs --------------------------------------------------------------------------

def _workload(case, seed, width=64, height=64) -> scenes.Workload:
    """The seeded scene of a case with its camera."""
    s = case["scene"]
    if s == "heightfield":
        return scenes.heightfield_c1(seed, width, height)
    if s == "closed":
        return scenes.closed_surfaces(seed, case["size"], width, height)
    if s == "displaced":
        box = 25.0 * (case["size"] / 4096.0) ** (1.0 / 3.0)   # the million-patch scene's density
        return scenes.displaced_grids(seed, case["size"], width, height, box=box)
    # a scene file, seen from its own view moved a little by the seed
    wl = scenes.from_dl(os.path.join(_SCENE_DIR, s + ".dl"), width, height)
    rng = np.random.default_rng(seed)
    cam = dataclasses.replace(wl.camera)
    cam.position = (cam.position + rng.uniform(-0.2, 0.2, 3)).astype(np.float32)
    m = cam.to_world.copy()
    m[12:15] = cam.position
    cam.to_world = m
    wl.camera = cam
    return wl


def _rays(case, wl, seed, n) -> np.ndarray:
    """n rays: camera rays of a closest case, half random ones elsewhere."""
    side = max(1, int(math.ceil(math.sqrt(n))))
    w, h = (1920, 1080) if n == 1920 * 1080 else (side, side)
    cam = dataclasses.replace(wl.camera, width=w, height=h)
    rays = scenes.camera_rays(cam)[:n]
    if case["kind"] == "closest":
        return rays
    rng = np.random.default_rng(seed + 77)
    box = {"heightfield": 1.0, "closed": 10.0}.get(case["scene"], 25.0 * (max(case["size"], 1) / 4096.0) ** (1.0 / 3.0))
    m = n if case["kind"] == "any" else n - n // 2
    o = rng.uniform(0.0, box, (m, 3))
    d = rng.normal(size=(m, 3))
    rnd = np.zeros((m, 8), np.float32)
    rnd[:, 0:3], rnd[:, 4:7] = o, d / np.linalg.norm(d, axis=1, keepdims=True)
    rnd[:, 3] = np.where(rng.random(m) < 0.5, np.inf, rng.uniform(0.1, 1.0, m) * box)
    return np.concatenate([rays[: n - m], rnd]).astype(np.float32)


def _patches(n, seed):
    """n bumpy unit-sized patches (n, 64), made on the GPU."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    p = torch.rand((n, 4, 4, 4), generator=g, device="cuda") * 0.25
    grid = torch.arange(4, device="cuda", dtype=torch.float32) / 3.0
    p[..., 0] += grid[None, None, :]
    p[..., 1] += grid[None, :, None]
    p[..., 2] *= torch.rand((n, 1, 1), generator=g, device="cuda") * 4.0
    p[..., 3] = 1.0
    return p.reshape(n, 64).contiguous(), g


def _pair_rays(n, g):
    """A ray per patch of _patches: from around it towards it, two in three hits."""
    o = torch.randn((n, 3), generator=g, device="cuda")
    o = 0.5 + 2.0 * o / o.norm(dim=1, keepdim=True)
    t = torch.rand((n, 3), generator=g, device="cuda") * 1.2 + torch.tensor([0.0, 0.0, -0.2], device="cuda")
    d = t - o
    r = torch.zeros((n, 8), device="cuda")
    r[:, 0:3], r[:, 4:7] = o, d / d.norm(dim=1, keepdim=True)
    r[:, 3] = math.inf
    return r.contiguous()


def _batch_sizes(case):
    """(grids, rays, occlusion) of each scene of a batch: both counts spread
    over the logarithm of their range, in two different orders."""
    m = case["scenes"]
    r0 = min(4_096, case["rays"])
    out = []
    for k in range(m):
        a, b = ((5 * k + 2) % m) / (m - 1), ((7 * k + 3) % m) / (m - 1)
        patches = 1_000 * (case["patches"] / 1_000) ** a
        out.append((max(1, round(patches / 256)), round(r0 * (case["rays"] / r0) ** b), k % 3 == 1))
    return out


def _uv(n, g, m):
    return torch.rand((n, m), generator=g, device="cuda").contiguous()


def _f32(*shape):
    return torch.zeros(shape, dtype=torch.float32, device="cuda")


def _i32(*shape):
    return torch.zeros(shape, dtype=torch.int32, device="cuda")


def prepare(case, seed):
    ctx, kind = _context(), case["kind"]
    s = dict(case=case)
    if kind in ("clip", "subdivide", "eval", "subpatch"):
        n = case["n"]
        s["patches"], g = _patches(n, seed)
        if kind == "eval":
            s["uv"], s["out"] = _uv(n, g, 2), _f32(n, 4)
        elif kind == "subpatch":
            a = _uv(n, g, 4)
            lo, w = 0.6 * a[:, :2], 0.05 + 0.35 * a[:, 2:]
            s["ranges"] = torch.stack([lo[:, 0], lo[:, 0] + w[:, 0], lo[:, 1], lo[:, 1] + w[:, 1]], 1).contiguous()
            s["out"] = _f32(n, 64)
        else:
            s["rays"], s["hits"] = _pair_rays(n, g), _f32(n, 4)
    elif kind == "pick":
        rng = np.random.default_rng(seed)
        side = int(round(math.sqrt(case["patches"])))
        v, i = scenes.heightfield_grid(rng, n=side)
        s["pick"] = ctx.patch_bvh(v, i)
        n = case["rays"]
        o = rng.uniform([0, 0, 0.8], [1, 1, 1.5], (n, 3))
        d = rng.uniform([-0.3, -0.3, -0.2], [1.3, 1.3, 0.2], (n, 3)) - o   # some past the edge
        rays = np.zeros((n, 8), np.float32)
        rays[:, 0:3], rays[:, 3], rays[:, 4:7] = o, np.inf, d / np.linalg.norm(d, axis=1, keepdims=True)
        s["rays"], s["hits"], s["occluded"] = torch.from_numpy(rays).cuda(), _f32(n, 4), _i32(n)
    elif kind == "batch":
        s["scenes"], s["jobs"] = [], []
        for k, (grids, n, occlusion) in enumerate(_batch_sizes(case)):
            one = dict(kind="any", scene="displaced", size=grids)   # half of its rays from the camera, half scattered
            wl = _workload(one, seed + 1000 * k)
            ds = ctx.scene(wl.scene, hash_retries=3)
            rays = np.concatenate([_rays(dict(one, kind="closest"), wl, seed + k, n // 2),
                                   _rays(one, wl, seed + k, n - n // 2)])
            job = dict(scene=ds, rays=torch.from_numpy(rays).cuda(), n=n, any=occlusion)
            if occlusion:
                job["occluded"] = _i32(n)
            else:
                job["hits"], job["objects"] = _f32(n, 4), _i32(n)
            s["scenes"].append(ds)
            s["jobs"].append(job)
        s["batch"] = ctx.batch(s["jobs"])
    else:
        w, h = case.get("width", 64), case.get("height", 64)
        wl = _workload(case, seed, w, h)
        s["scene"] = ctx.scene(wl.scene, hash_retries=3)
        if kind == "render":
            s["camera"], s["frame"], s["color"] = wl.camera, _i32(h, w), _f32(h, w, 3)
        else:
            n = case["rays"]
            s["rays"] = torch.from_numpy(_rays(case, wl, seed, n)).cuda()
            s["hits"], s["objects"], s["occluded"] = _f32(n, 4), _i32(n), _i32(n)
            if kind == "shade":
                s["color"], s["pixels"] = _f32(n, 3), _i32(n)
    torch.cuda.synchronize()
    return s


# --- one pass ------------------------------------------------------------------------

def _hits(h):
    """Hit records as what they hold: t, u, v and the patch word."""
    return {"tuv": h[:, :3], "patch": h.view(torch.int32)[:, 3]}


def run(s):
    case, ctx, lib = s["case"], _context(), cgs.lib()
    kind = case["kind"]
    if kind == "clip":
        n = case["n"]
        st = lib.cgs_bezier_clip(ctx.h, s["rays"].data_ptr(), s["patches"].data_ptr(), n, 2.0 ** -12,
                                 s["hits"].data_ptr(), None)
        out = _hits(s["hits"])
    elif kind == "subdivide":
        n = case["n"]
        st = lib.cgs_subdivision(ctx.h, s["rays"].data_ptr(), s["patches"].data_ptr(), n, 2.0 ** -4,
                                 s["hits"].data_ptr(), None)
        out = _hits(s["hits"])
    elif kind == "eval":
        st = lib.cgs_patch_eval(ctx.h, _KINDS.index(case["what"]), s["patches"].data_ptr(), s["uv"].data_ptr(),
                                case["n"], s["out"].data_ptr(), None)
        out = {"out": s["out"]}
    elif kind == "subpatch":
        st = lib.cgs_patch_subpatch(ctx.h, s["patches"].data_ptr(), s["ranges"].data_ptr(), case["n"],
                                    s["out"].data_ptr(), None)
        out = {"out": s["out"]}
    elif kind == "pick":
        if case["any"]:
            st = lib.cgs_patchbvh_intersect_any(ctx.h, s["pick"].h, s["rays"].data_ptr(), case["rays"],
                                                s["occluded"].data_ptr(), None)
            out = {"occluded": s["occluded"]}
        else:
            st = lib.cgs_patchbvh_intersect(ctx.h, s["pick"].h, s["rays"].data_ptr(), case["rays"],
                                            s["hits"].data_ptr(), None)
            out = _hits(s["hits"])
    elif kind == "closest":
        s["scene"].trace_closest_dev(s["rays"], case["rays"], s["hits"], s["objects"])
        st, out = 0, {**_hits(s["hits"]), "objects": s["objects"]}
    elif kind == "any":
        s["scene"].trace_any_dev(s["rays"], case["rays"], s["occluded"])
        st, out = 0, {"occluded": s["occluded"]}
    elif kind == "shade":
        s["scene"].shade_dev(s["rays"], case["rays"], s["color"], s["pixels"], s["hits"], s["objects"],
                             depth=case["depth"])
        st, out = 0, {**_hits(s["hits"]), "objects": s["objects"], "color": s["color"], "pixels": s["pixels"]}
    elif kind == "batch":
        s["batch"].launch()
        st, out = 0, []
        for j in s["jobs"]:
            out.append({"occluded": j["occluded"]} if j["any"] else {**_hits(j["hits"]), "objects": j["objects"]})
    else:
        if case["samples"]:
            st = s["scene"].render_sampled_dev(s["camera"], s["frame"], s["color"], samples=case["samples"],
                                               depth=case["depth"])
        else:
            st = s["scene"].render_dev(s["camera"], s["frame"], s["color"], depth=case["depth"])
        # a context renders one frame at a time: the program waits for it
        # before it shows the frame or asks for the next
        ctx.sync()
        out = {"color": s["color"], "frame": s["frame"]}
    if st:
        raise RuntimeError(f"{kind}: status {st}")
    return out


# --- what a pass needs, and how exact it is ------------------------------------------

def _scene_patches(case):
    if case["kind"] == "pick":
        return case["patches"]
    return {"heightfield": 256, "closed": 256 * case["size"], "displaced": 256 * case["size"]}.get(case["scene"], 78)


# Operations of one ray: a box test for each level of a tree over the patches
# (27 each), one projection (248), three clipping passes (551 each) and the
# evaluation at the hit (222).
def _ray_flops(patches):
    return 27 * 2 * max(1.0, math.log2(max(2, patches))) + 248 + 3 * 551 + 222


def work(case):
    kind = case["kind"]
    if kind in ("clip", "subdivide"):
        return {"bytes": case["n"] * (32 + 256 + 16), "flops": case["n"] * (248 + 3 * 551 + 222)}
    if kind == "eval":
        return {"bytes": case["n"] * (256 + 8 + 16), "flops": case["n"] * (400 if "normal" in case["what"] else 200)}
    if kind == "subpatch":
        return {"bytes": case["n"] * (256 + 16 + 256), "flops": case["n"] * 1100}
    if kind == "batch":
        sizes = _batch_sizes(case)
        return {"bytes": sum(n * (36 if any else 52) + 256 * 384 * g for g, n, any in sizes),
                "flops": sum(n * _ray_flops(256 * g) for g, n, _ in sizes)}
    rays = case["rays"] if kind != "render" else case["width"] * case["height"] * max(1, case["samples"])
    patches = _scene_patches(case)
    # control points and two BVH nodes of each patch, or a few patches a ray
    scene = min(patches * (256 + 2 * 64), rays * 2048)
    if kind == "render":
        return {"bytes": case["width"] * case["height"] * 16 + scene, "flops": rays * _ray_flops(patches)}
    out = {"pick": 16, "closest": 20, "any": 4, "shade": 36}[kind]
    return {"bytes": rays * (32 + out) + scene, "flops": rays * _ray_flops(patches)}


def tolerance(case):
    """Every result is the reference algorithm's in FP32, rounding by rounding:
    the library promises the same bits whatever the order of its work."""
    return "exact"


def _bernstein(t):
    s = 1.0 - t
    return torch.stack([s * s * s, 3 * s * s * t, 3 * s * t * t, t * t * t], -1)


def _dbernstein(t):
    """The derivative without its factor 3 (the de Casteljau hodograph)."""
    s = 1.0 - t
    return torch.stack([-s * s, s * s - 2 * s * t, 2 * s * t - t * t, t * t], -1)


def exact(case, seed):
    """Evaluations and sub-patches in 64 bits.  Hits and frames have no such
    value: a clip stops at a projected size of 2^-12, and the point it stops
    at, and with it the hit and the pixel, is the FP32 algorithm's own."""
    kind = case["kind"]
    if kind not in ("eval", "subpatch"):
        return None
    s = prepare(case, seed)
    P = s["patches"].double().reshape(-1, 4, 4, 4)     # (n, v, u, xyzw)
    if kind == "eval":
        u, v = s["uv"].double().unbind(1)
        # the matrix forms keep the factor 3 of the derivative
        f = 3.0 if case["what"].endswith("_mat") else 1.0
        ev = lambda bu, bv: torch.einsum("nj,ni,njik->nk", bv, bu, P)   # noqa: E731
        du = f * ev(_dbernstein(u), _bernstein(v))
        dv = f * ev(_bernstein(u), _dbernstein(v))
        w = case["what"]
        if w.startswith("interpolate"):
            o = ev(_bernstein(u), _bernstein(v))
        elif w.startswith("derivative_u"):
            o = du
        elif w.startswith("derivative_v"):
            o = dv
        else:
            o = torch.cat([torch.linalg.cross(du[:, :3], dv[:, :3]), torch.zeros_like(du[:, :1])], 1)
        return {"out": o}
    r = s["ranges"].double()

    def cut(lo, hi):
        """(n, 4, 4): the Bezier net of [lo, hi] from the whole one (blossoms)."""
        rows = []
        for k in range(4):
            t = [hi] * k + [lo] * (3 - k)
            e1, e2, e3 = t[0] + t[1] + t[2], t[0] * t[1] + t[0] * t[2] + t[1] * t[2], t[0] * t[1] * t[2]
            # the blossom of each Bernstein polynomial in the three arguments
            rows.append(torch.stack([1 - e1 + e2 - e3, e1 - 2 * e2 + 3 * e3, e2 - 3 * e3, e3], -1))
        return torch.stack(rows, 1)

    U, V = cut(r[:, 0], r[:, 1]), cut(r[:, 2], r[:, 3])
    Q = (U[:, None, :, :, None] * P[:, :, None, :, :]).sum(3)          # rows cut in u
    return {"out": (V[:, :, :, None, None] * Q[:, None, :, :, :]).sum(2).reshape(-1, 64)}
