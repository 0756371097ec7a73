"""Workloads the renderer is timed on: what programs built on it call, over the sizes they
call it with.

listed() holds one case per use; draw() gives further cases of the same ranges.  A case is a
dict of plain values; `use` picks the entry point:

  render    an integrator's passes into the frame: the naive MIS path tracer, the light
            tracer, the triple tracer or the global-queue tracer.  `read` False leaves the
            frame on the GPU, as an interactive viewer that shows every pass does; True
            copies it to the host, as an offline render does at its end.
  edit      upload of a scene whose MTBVH is built on the device, then one pass: a scene
            edit followed by its first preview frame.
  step      one step of differentiable rendering through the autograd function: image, L2
            loss against a target, gradients of materials and environment texels.  Every
            step takes passes of its own.
  batch     several scenes with uneven sizes and pass counts in one batched launch.
  closest   closest hits of a ray batch in device memory.
  any       occlusion of a ray batch in host memory.

Scenes: the Cornell box (36 triangles, or its faces tessellated), the caustics box (10,040
triangles), the box with every material branch, the textured box and displaced spheres under
a sky environment map with importance sampling.  A seed moves the camera, the geometry's
scale, the colours, the environment's rotation, the per-pixel seeds and the rays.
"""
import copy
import functools
import math

import numpy as np
import torch

from zillumgl_amd import diff, render, scene


def listed():
    return [
        # one progressive pass of the smallest scene: a viewer's frame, latency-bound
        dict(name="preview_cornell_256", use="render", integrator="naive", scene="cornell", detail=1, width=256,
             height=256, passes=1, depth=5, roulette=False, read=False),
        # one interactive pass of a 205,000-triangle scene at 720p and the default depth
        dict(name="interactive_spheres_720p", use="render", integrator="naive", scene="spheres", detail=4, width=1280,
             height=720, passes=1, depth=4, roulette=False, read=False),
        # the headline workload: 819,400 triangles, 1080p, 64 passes, depth 8, read back
        dict(name="final_spheres_1080p_64", use="render", integrator="naive", scene="spheres", detail=5, width=1920,
             height=1080, passes=64, depth=8, roulette=False, read=True),
        # every BSDF branch, thin lens, Russian roulette, an odd film size
        dict(name="materials_lens_roulette", use="render", integrator="naive", scene="materials", detail=1, width=617,
             height=411, passes=8, depth=8, roulette=True, read=True),
        # caustics by light tracing (64 x 1536 paths per pass)
        dict(name="light_caustics_1024", use="render", integrator="light", scene="caustics", detail=1, width=1024,
             height=1024, passes=16, depth=8, roulette=False, read=True),
        # caustics by the triple tracer: camera and light paths combined
        dict(name="triple_caustics_1024", use="render", integrator="triple", scene="caustics", detail=1, width=1024,
             height=1024, passes=8, depth=8, roulette=False, read=True),
        # the global-queue tracer
        dict(name="queue_caustics_512", use="render", integrator="queue", scene="caustics", detail=1, width=512,
             height=512, passes=8, depth=6, roulette=False, read=True),
        # a scene edit: upload with the MTBVH built on the device, then a preview pass
        dict(name="edit_spheres_preview", use="edit", integrator="naive", scene="spheres", detail=4, width=640,
             height=360, passes=1, depth=4, roulette=False, read=False),
        # one optimisation step on the tessellated box (201,588 triangles, 32 materials)
        dict(name="step_tessellated_512", use="step", integrator="naive", scene="tessellated", detail=77, width=512,
             height=512, passes=32, depth=6, roulette=False, read=True),
        # ten small and middling scenes in one launch
        dict(name="batch_10_scenes", use="batch", integrator="naive", scene="boxes", detail=10, width=512, height=512,
             passes=16, depth=8, roulette=False, read=False),
        # a million incoherent rays through the Cornell box
        dict(name="closest_cornell_1m", use="closest", integrator="", scene="cornell", detail=1, width=64, height=64,
             passes=1000000, depth=0, roulette=False, read=False),
        # occlusion of rays handed over in host arrays
        dict(name="any_spheres_200k", use="any", integrator="", scene="spheres", detail=4, width=64, height=64,
             passes=200000, depth=0, roulette=False, read=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    use = rng.choice(["render", "render", "render", "render", "edit", "step", "batch", "closest", "any"])
    c = dict(use=use, integrator="naive", scene="cornell", detail=1, width=_log_int(rng, 64, 1280),
             height=_log_int(rng, 64, 1024), passes=1, depth=rng.randint(3, 10), roulette=rng.random() < 0.3,
             read=rng.random() < 0.5)
    if use == "render":
        c["integrator"] = rng.choice(["naive", "naive", "naive", "light", "triple", "queue"])
        lit = c["integrator"] != "naive"
        c["scene"] = rng.choice(["cornell", "caustics", "materials"] +
                                ([] if lit else ["spheres", "textured", "tessellated"]))
        c["passes"] = _log_int(rng, 1, 24)
    elif use == "edit":
        c.update(scene=rng.choice(["spheres", "tessellated", "caustics"]), depth=4, read=False)
    elif use == "step":
        c.update(scene="tessellated", width=_log_int(rng, 64, 512), height=_log_int(rng, 64, 512),
                 passes=_log_int(rng, 2, 24), depth=rng.randint(3, 7), roulette=False, read=True)
    elif use == "batch":
        c.update(scene="boxes", width=_log_int(rng, 128, 512), height=_log_int(rng, 128, 512),
                 passes=_log_int(rng, 4, 16), read=False)
    else:
        c.update(integrator="", scene=rng.choice(["cornell", "caustics", "spheres", "tessellated"]), width=64,
                 height=64, passes=_log_int(rng, 1000, 1000000), depth=0, roulette=False, read=use == "any")
    if c["scene"] == "spheres":
        c["detail"] = rng.randint(2, 4)
    elif c["scene"] == "tessellated":
        c["detail"] = _log_int(rng, 5, 100)
    elif c["scene"] == "boxes":
        c["detail"] = rng.randint(2, 12)
    return c


# ---------------------------------------------------------------------------
# Scenes
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=3)
def _spheres(detail):
    env = {5: (2048, 1024), 4: (1024, 512)}.get(detail, (501, 250))
    return scene.config2(64, 64, 40, detail, env)


def _desc(name, detail, width, height, seed):
    """The scene with the seed's camera position, scale, colours, sky and pixel seeds."""
    if name == "spheres":
        d = copy.copy(_spheres(detail))
    elif name == "caustics":
        d = scene.config3(width, height, seed=3 + seed % 1000)
    elif name == "materials":
        d = scene.config_materials(width, height, lens_radius=0.02, focal_dist=1.9)
    elif name == "textured":
        d = scene.config_textured(width, height)
    elif name == "tessellated":
        d = scene.config5(width, height, n=detail, seed=5 + seed % 1000)
    else:
        d = scene.config1(width, height)
    d.width, d.height = width, height
    g = np.random.default_rng(seed)
    scale = np.float32(g.uniform(0.9, 1.1))

    def scaled(mesh):
        m = copy.copy(mesh)
        m.positions = np.ascontiguousarray(mesh.positions, np.float32) * scale
        return m

    def coloured(mat):
        m = copy.copy(mat)
        m.base_color = tuple(float(x) for x in np.clip(np.asarray(mat.base_color) * g.uniform(0.8, 1.0, 3), 0, 1))
        return m
    d.objects = [(scaled(mesh), coloured(mat)) for mesh, mat in d.objects]
    d.lights = [(scaled(mesh), power) for mesh, power in d.lights]
    cam = copy.copy(d.camera)
    cam.pos = tuple(float(p * scale + q) for p, q in zip(cam.pos, g.uniform(-0.02, 0.02, 3)))
    d.camera = cam
    d.env_rotation = float(g.uniform(0, 2 * math.pi)) if d.env is not None else 0.0
    d.noise_seed = seed % 100000
    return d


def _packed(case, seed):
    return scene.pack(_desc(case["scene"], case["detail"], case["width"], case["height"], seed), bvh="device")


def _box_scene(case, k, seed):
    """Scene k of a batch: a tessellated box with a triangle count, film and pass count of
    its own (the same for every seed, which moves the boxes); the first is the case's
    largest film."""
    g = np.random.default_rng([case["width"], case["height"], case["detail"], k])
    n = int(round(math.exp(g.uniform(math.log(5), math.log(80)))))
    f = 1.0 if k == 0 else float(g.uniform(0.25, 1.0))
    d = scene.SceneDesc()
    d.objects = scene.cornell_tessellated(n, seed * 100 + k)
    d.lights = [(scene.cornell_light(), (17.0, 12.0, 4.0))]
    d.camera = scene.CameraDesc(pos=(0.5, -1.5, 0.5), angle=(0.0, 0.0, 0.0), fov=40.0)
    d.width, d.height = max(16, int(case["width"] * f)), max(16, int(case["height"] * f))
    d.noise_seed = (seed + k) % 100000
    return scene.pack(d, bvh="device"), max(1, int(case["passes"] * g.uniform(0.25, 1.0))), int(
        g.integers(3, case["depth"] + 1))


class _DeviceFrame:
    """A context's frame as an array torch can wrap.  It holds the context, which owns the
    memory: the frame is freed with the context, not before the last tensor on it."""

    def __init__(self, ctx):
        self.ctx = ctx
        self.__cuda_array_interface__ = dict(shape=(ctx.height, ctx.width, 4), typestr="<f4",
                                             data=(ctx.frame_device_ptr(), False), version=3)


def _frame(ctx):
    t = torch.as_tensor(_DeviceFrame(ctx), device="cuda")
    t.ctx = ctx
    return t


def _integrator(case):
    d, rr = case["depth"], case["roulette"]
    if case["integrator"] == "light":
        return render.LightPathIntegrator(d, rr, 64)
    if case["integrator"] == "triple":
        return render.TriplePathIntegrator(d, rr, 64)
    if case["integrator"] == "queue":
        return render.GlobalQueuePathIntegrator(d, rr)
    return render.NaivePathIntegrator(d, rr)


def _rays(packed, n, seed):
    """Rays from points in the scene's box in uniform directions (SoA, 6 x n)."""
    lo, hi = packed.vertices.min(0).astype(np.float64), packed.vertices.max(0).astype(np.float64)
    r = scene.ray_batch(n, seed).astype(np.float64)
    r[:3] = lo[:, None] + (hi - lo)[:, None] * r[:3]
    return np.ascontiguousarray(r.astype(np.float32))


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def prepare(case, seed):
    use = case["use"]
    st = dict(case=case)
    if use == "batch":
        st["ctxs"], passes = [], []
        for k in range(case["detail"]):
            packed, n, depth = _box_scene(case, k, seed)
            ctx = render.Context(0)
            ctx.upload(packed)
            st["ctxs"].append(ctx)
            passes.append((0, n, 1, depth))
        st["batch"] = render.Batch(0)
        st["batch"].set(st["ctxs"], passes)
        st["frames"] = [_frame(c) for c in st["ctxs"]]
        return st
    packed = _packed(case, seed)
    ctx = st["ctx"] = render.Context(0)
    ctx.upload(packed)
    if use in ("render", "edit"):
        st["packed"] = packed if use == "edit" else None
        st["integrator"] = _integrator(case)
        st["integrator"].init(ctx)
        if not case["read"]:
            st["frame"] = _frame(ctx)
    elif use == "step":
        g = torch.Generator().manual_seed(seed)
        mats, env = (torch.from_numpy(a) for a in diff.scene_parameters(packed))
        st["renderer"] = diff.Renderer(ctx, packed, case["passes"], case["depth"])
        st["mats"], st["env"] = mats, env
        st["target"] = torch.rand((case["height"], case["width"], 3), generator=g)
    else:
        n = case["passes"]
        rays = _rays(packed, n, seed)
        if use == "closest":
            st["rays"] = torch.from_numpy(rays).cuda()
            st["prim"] = torch.empty(n, dtype=torch.int32, device="cuda")
            st["t"] = torch.empty(n, dtype=torch.float32, device="cuda")
            st["bin"] = torch.empty(n, dtype=torch.int32, device="cuda")
        else:
            size = float(np.linalg.norm(packed.vertices.max(0) - packed.vertices.min(0)))
            st["rays"] = rays
            st["tmax"] = np.random.default_rng(seed).uniform(0.01, 0.5, n).astype(np.float32) * np.float32(size)
    return st


def run(st):
    case = st["case"]
    use = case["use"]
    if use in ("render", "edit"):
        it = st["integrator"]
        if use == "edit":
            st["ctx"].upload(st["packed"])
        it.reset()
        it.free_counter = 0
        it.render_one_pass(case["passes"])
        return it.get_frame() if case["read"] else st["frame"]
    if use == "step":
        r = st["renderer"]
        mats = st["mats"].clone().requires_grad_()
        env = st["env"].clone().requires_grad_()
        image = diff.render_image(mats, env, r)
        loss = (image - st["target"]).square().sum()
        loss.backward()
        r.first_pass += r.n_passes
        r.free_counter += r.n_passes
        return dict(image=image.detach(), mats=mats.grad, env=env.grad)
    if use == "batch":
        st["batch"].launch()
        st["batch"].synchronize()
        return st["frames"]
    if use == "closest":
        st["ctx"].trace_closest_device(st["rays"].data_ptr(), case["passes"], st["prim"].data_ptr(),
                                       st["t"].data_ptr(), st["bin"].data_ptr())
        return dict(prim=st["prim"], t=st["t"], bin=st["bin"])
    return st["ctx"].trace_any(st["rays"], st["tmax"])


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _triangles(case):
    k = case["detail"]
    return {"cornell": 36, "caustics": 10040, "materials": 614, "textured": 36, "boxes": 34 * 1000,
            "spheres": 40 * 20 * 4 ** k + 200, "tessellated": 34 * k * k + 2}[case["scene"]]


def work(case):
    """Bytes: the scene's triangles (positions, normals, indices) and environment read once,
    rays read and hits or frames written once.  Operations: a ray meets about 2 log2 n boxes
    (15 operations each) and two triangles (50); a path vertex shades (400) and casts two
    rays; a path of depth d has on average about 0.6 d vertices."""
    n = _triangles(case)
    walk = 2 * math.log2(n) * 15 + 100
    pixels = case["width"] * case["height"]
    env = {5: 2048 * 1024, 4: 1024 * 512}.get(case["detail"], 501 * 250) * 8 if case["scene"] == "spheres" else 0
    geometry = n * 48 + env
    if case["use"] in ("closest", "any"):
        return {"bytes": geometry + case["passes"] * (36 if case["use"] == "closest" else 29),
                "flops": case["passes"] * walk}
    path = walk + 0.6 * case["depth"] * (2 * walk + 400)
    if case["use"] == "batch":
        return {"bytes": case["detail"] * (geometry + 0.4 * pixels * 32),
                "flops": case["detail"] * 0.4 * pixels * 0.6 * case["passes"] * path * 0.7}
    paths = pixels * case["passes"]
    if case["integrator"] == "light":
        paths = 64 * 1536 * case["passes"]
    elif case["integrator"] == "triple":
        paths += 64 * 1536 * case["passes"]
    if case["use"] == "step":
        return {"bytes": geometry + pixels * 28 + 2 * 256 * 128 * 12, "flops": 1.5 * paths * path}
    return {"bytes": geometry * (3 if case["use"] == "edit" else 1) + pixels * 16, "flops": paths * path}


def exact(case, seed):
    """Closest hits against every triangle in 64 bits (distances; the primitives and bins are
    whole numbers).  The image of a path tracer has no such value in reach."""
    if case["use"] != "closest" or case["scene"] != "cornell":
        return None
    packed = _packed(case, seed)
    r = torch.from_numpy(_rays(packed, case["passes"], seed)).cuda().double()
    o, d = r[:3].T, r[3:].T
    v = torch.from_numpy(packed.vertices).cuda().double()
    best = torch.full((o.shape[0],), 1e8, dtype=torch.float64, device="cuda")
    for ia, ib, ic in packed.indices.tolist():
        a, ab, ac = v[ia], v[ib] - v[ia], v[ic] - v[ia]
        p = torch.linalg.cross(d, ac.expand_as(d))
        det = p @ ab
        ao = o - a
        q = torch.linalg.cross(ao, ab.expand_as(ao))
        sign = torch.sign(det)
        u, w = (ao * p).sum(1) * sign, (d * q).sum(1) * sign
        t = (q @ ac) * sign / det.abs()
        hit = (det.abs() >= 1e-6) & (u >= 0) & (w >= 0) & (u + w <= det.abs()) & (t > 0)
        best = torch.where(hit & (t < best), t, best)
    return dict(prim=None, t=best, bin=None)
