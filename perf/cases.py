"""The work that programs built on this framework have it do, as measurable cases.

A case is a dict of plain values; its ``kind`` says which public path it takes:

    frame    a shot of a few frames: history reset, then per frame camera constants, instance
             motion where the scene moves, the path tracer, reprojection and a denoiser
    diff     forward render, L2 loss and backward through ``diff.render``
    infer    the learned denoiser over one image's FP32 features
    train    the learned denoiser's training loss on a batch and its gradients
    cast     a batch of rays against a resident scene
    probes   the ambient-cube grid over a scene: clear, voxelise, bake passes, read back
    load     a new scene into a running context, then a batch of rays against it

Scenes are the package's generators (Cornell box, city, instanced bricks). The seed decides
geometry, materials, camera positions, random streams, rays and images.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import gknextengine_amd as gk
from gknextengine_amd import diff, scenes

FRAME = dict(kind="frame", scene="city", grid=64, width=1920, height=1080, frames=4, estimator="pt_mis",
             samples=1, bounces=8, denoiser="bilateral", sun=False, sky="black", probes=False, hdr=False,
             textured=False, super_resolution=2)


def listed():
    return [
        # the smallest interactive view: a preview box, sixteen progressive frames, one lamp
        dict(FRAME, name="preview_cornell", scene="cornell", width=256, height=256, frames=16, estimator="ref_v2",
             bounces=4, denoiser="none"),
        # the renderer's main view: a large static scene at full HD with many small emitters
        dict(FRAME, name="city_pt_mis"),
        # the engine's own estimator outdoors: sun, sky image and the baked probe grid that ends paths
        dict(FRAME, name="city_ref_v2_sun", estimator="ref_v2", sun=True, sky="image", probes=True),
        # a physics scene: every instance moves every frame, top-level tree rebuilt each time
        dict(FRAME, name="bricks_moving", scene="bricks", grid=16, bounces=4, sky="constant"),
        # a window of odd size, textured, two paths a pixel, learned denoiser, HDR display, upscaled
        dict(FRAME, name="window_textured_unet", grid=24, width=853, height=479, frames=2, samples=2, bounces=5,
             denoiser="unet", sky="image", hdr=True, textured=True, super_resolution=1),
        # material fitting: gradients of an image loss for 256 materials x 5 parameters
        dict(name="fit_materials", kind="diff", width=512, height=512, samples=4, bounces=4),
        # the learned denoiser alone over a full HD image
        dict(name="denoise_full_hd", kind="infer", width=1920, height=1080),
        # the learned denoiser's training step at its usual batch
        dict(name="denoise_train", kind="train", batch=8, width=256, height=256),
        # gameplay queries: a few hundred picking and line-of-sight rays, answered at once
        dict(name="pick_rays", kind="cast", scene="city", grid=64, rays=300, any_hit=False, rays_from="random"),
        # an offline ray batch, incoherent, into the instanced scene
        dict(name="bulk_rays_bricks", kind="cast", scene="bricks", grid=16, rays=2000000, any_hit=False,
             rays_from="random"),
        # relighting: a probe grid over the city voxelised and baked twice
        dict(name="probe_bake", kind="probes", scene="city", grid=64, size_xy=64, size_z=32, passes=2, sun=True,
             sky="image"),
        # loading a level into a running renderer
        dict(name="load_city", kind="load", scene="city", grid=64, rays=4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "diff", "infer", "train", "cast", "cast", "probes", "load"])
    if kind == "frame":
        c = dict(FRAME)
        c["scene"] = rng.choice(["cornell", "city", "city", "bricks"])
        c["grid"] = rng.randint(6, 16) if c["scene"] == "bricks" else rng.randint(12, 64)
        c["width"] = _log_int(rng, 160, 1920)
        c["height"] = max(90, int(c["width"] * rng.choice([9 / 16, 3 / 4, 0.5625, 1.0]))) + rng.choice([0, 0, 1, -3])
        if rng.random() < 0.5:  # window sizes that are whole tiles
            c["width"], c["height"] = (c["width"] + 7) // 8 * 8, (c["height"] + 7) // 8 * 8
        c["height"] = min(c["height"], 1080)
        c["frames"] = rng.randint(1, 4)
        c["estimator"] = rng.choice(["pt_mis", "pt_mis", "ref_v2"])
        c["samples"] = rng.choice([1, 1, 2, 4]) if c["width"] * c["height"] <= 500000 else 1
        c["bounces"] = rng.randint(2, 8)
        c["denoiser"] = rng.choice(["none", "bilateral", "bilateral", "unet"])
        c["sun"] = rng.random() < 0.4
        c["sky"] = rng.choice(["black", "constant", "image"])
        c["probes"] = c["estimator"] == "ref_v2" and c["scene"] != "bricks" and rng.random() < 0.5
        c["hdr"] = rng.random() < 0.3
        c["textured"] = c["scene"] != "bricks" and rng.random() < 0.3
        c["super_resolution"] = rng.choice([2, 2, 1, 0])
        return c
    if kind == "diff":
        w, h = _log_int(rng, 64, 512), _log_int(rng, 64, 512)
        spp = rng.choice([1, 2, 4, 8])
        while w * h * spp > 1048576:
            spp //= 2
        return dict(kind="diff", width=w, height=h, samples=spp, bounces=rng.randint(2, 6))
    if kind == "infer":
        return dict(kind="infer", width=_log_int(rng, 120, 1920), height=_log_int(rng, 90, 1080))
    if kind == "train":
        w, h = 16 * rng.randint(4, 16), 16 * rng.randint(4, 16)
        return dict(kind="train", batch=rng.randint(1, 8), width=w, height=h)
    scene = rng.choice(["city", "bricks", "cornell"])
    grid = rng.randint(6, 16) if scene == "bricks" else rng.randint(12, 64)
    if kind == "cast":
        return dict(kind="cast", scene=scene, grid=grid, rays=_log_int(rng, 1, 2000000), any_hit=rng.random() < 0.4,
                    rays_from=rng.choice(["random", "camera"]))
    if kind == "probes":
        return dict(kind="probes", scene=rng.choice(["city", "cornell"]), grid=rng.randint(12, 64),
                    size_xy=rng.randint(16, 64), size_z=rng.randint(8, 32), passes=rng.randint(1, 2),
                    sun=rng.random() < 0.5, sky=rng.choice(["constant", "image"]))
    return dict(kind="load", scene=scene, grid=grid, rays=_log_int(rng, 64, 4096))


# ---------------------------------------------------------------- scenes, cameras, images
def _textures(scene, seed):
    """Base-colour, roughness and normal maps on half of the materials; texture coordinates are
    the triangles' own corners."""
    rng = np.random.default_rng([seed, 77])
    ids = []
    for k, size in enumerate((256, 128, 256, 64)):
        t = rng.integers(64, 255, (size, size + 16 * k, 4), dtype=np.uint8)
        if k == 2:  # normal map: around +z
            t[..., :2] = rng.integers(108, 148, t.shape[:2] + (2,), dtype=np.uint8)
            t[..., 2] = 255
        t[..., 3] = 255
        ids.append(scene.add_texture(t, srgb=k in (0, 3)))
    for m in scene.meshes:
        p = m["positions"]
        m["texcoords"] = np.ascontiguousarray(np.stack([p[:, 0] + 0.37 * p[:, 1], p[:, 2] - 0.21 * p[:, 1]], 1),
                                              np.float32)
        m["tangents"] = np.ascontiguousarray(np.tile(np.float32([1, 0, 0, 1]), (p.shape[0], 1)))
    for i, mat in enumerate(scene.materials):
        if mat.material_model != gk.MAT_DIFFUSE_LIGHT and i % 2 == 0:
            mat.diffuse_texture_id = ids[0] if i % 4 else ids[3]
            mat.mra_texture_id = ids[1]
            mat.normal_texture_id = ids[2]


def _scene(case, seed):
    """(SceneData, Bricks or None, camera, half extent of the scene)."""
    grid = case.get("grid", 0)
    rng = np.random.default_rng([seed, 5])
    if case["scene"] == "city":
        s = gk.procgen_city(grid, 4, 4 * grid, grid, 1 + seed % 1000003)
        k = grid / 64.0
        cam = dict(eye=(-20.0 * k, 28.0 * k + 2.0, -44.0 * k), target=(2.0 * k, 0.0, 4.0 * k), fov=50.0)
        return s, None, cam, 40.0 * k
    if case["scene"] == "bricks":
        b = scenes.Bricks(n_side=grid, seed=seed % 1000003)
        k = grid / 16.0
        return b.scene, b, dict(eye=(0.0, 10.0 * k, -30.0 * k), target=(0.0, 0.0, 0.0), fov=50.0), 14.0 * k
    s = gk.procgen_cornell()
    for m in s.materials:
        if m.material_model != gk.MAT_DIFFUSE_LIGHT:
            m.diffuse[0:3] = [float(v) for v in np.clip(np.array(m.diffuse[0:3]) * rng.uniform(0.8, 1.1, 3), 0, 0.95)]
    return s, None, dict(scenes.CORNELL_CAM), 0.6


def _sky_image(seed):
    rng = np.random.default_rng([seed, 9])
    h, w = 256, 512
    y = np.linspace(0, 1, h, dtype=np.float32)[:, None]
    img = np.zeros((h, w, 4), np.float32)
    base = rng.uniform(0.3, 0.9, 3).astype(np.float32)
    for c in range(3):
        img[..., c] = base[c] * (1.3 - y) + 0.05 * rng.random((h, w), dtype=np.float32)
    img[40:44, 100:104, :3] += 20.0
    img[..., 3] = 1.0
    return img


def _params(case, seed, cam, w, h, frame, prev, moved):
    rng = np.random.default_rng([seed, 21])
    drift = rng.normal(0.0, 0.01, 3) * moved * frame
    eye = tuple(float(a + d) for a, d in zip(cam["eye"], drift))
    p = gk.make_frame_params(eye, cam["target"], w, h, fov=cam["fov"], frame=frame, taa=True, prev=prev)
    p.estimator = gk.ESTIMATOR_PT_MIS if case["estimator"] == "pt_mis" else gk.ESTIMATOR_REF_V2
    p.samples = case["samples"]
    p.bounces = p.max_bounces = case["bounces"]
    p.global_seed = 1 + seed % 100003
    p.denoiser = {"none": gk.DENOISER_NONE, "bilateral": gk.DENOISER_BILATERAL, "unet": gk.DENOISER_UNET}[
        case["denoiser"]]
    p.hdr = int(case["hdr"])
    _light(p, case)
    return p


def _light(p, case):
    if case["sky"] != "black":
        p.has_sky = 1
        p.sky_color[:] = [1.0, 1.0, 1.0, 1.0] if case["sky"] == "image" else [0.6, 0.7, 0.9, 1.0]
    if case["sun"]:
        d = np.array([0.4, 0.8, -0.3])
        p.has_sun = 1
        p.sun_direction[:] = [*(float(v) for v in d / np.linalg.norm(d)), 0.0]
        p.sun_color[:] = [6.0, 5.5, 5.0, 1.0]


class _Device:
    """A device buffer of the library described for torch.as_tensor."""

    def __init__(self, ptr, shape, typestr):
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (ptr, False), "version": 2}


def _view(owner, ptr, shape, typestr):
    """A tensor over the library's memory (no copy); it keeps the context that owns it alive."""
    d = _Device(ptr, shape, typestr)
    d.owner = owner
    t = torch.as_tensor(d, device="cuda")
    t.owner = owner
    return t


def _target(ctx, name):
    dtype, ch = gk.TARGET_FORMAT[name]
    t = {np.float16: "<f2", np.float32: "<f4", np.uint32: "<i4"}[dtype]
    shape = (ctx.height, ctx.width, ch) if ch > 1 else (ctx.height, ctx.width)
    return _view(ctx, ctx.target_ptr(name), shape, t)


def _rays(case, seed, cam, half):
    n = case["rays"]
    rng = np.random.default_rng([seed, 31])
    r = np.zeros((n, 8), np.float32)
    eye = np.array(cam["eye"], np.float64)
    mid = np.array([0.5, 0.5, 0.5]) if case["scene"] == "cornell" else np.zeros(3)
    if case.get("rays_from") == "camera":  # scanline order over the camera's view
        side = max(1, int(math.ceil(math.sqrt(n))))
        i = np.arange(n)
        f = np.array(cam["target"]) - eye
        f = f / np.linalg.norm(f)
        s = np.cross(f, [0.0, 1.0, 0.0])
        s = s / np.linalg.norm(s)
        u = np.cross(s, f)
        k = math.tan(math.radians(cam["fov"] / 2))
        x, y = ((i % side) + rng.random(n)) / side * 2 - 1, ((i // side) + rng.random(n)) / side * 2 - 1
        d = f + (x * k)[:, None] * s - (y * k)[:, None] * u
        o = np.broadcast_to(eye, (n, 3))
    else:  # segments between two points of the scene's volume
        o = mid + rng.uniform(-half, half, (n, 3)) * [1, 0.4, 1] + [0, 0.3 * half, 0]
        d = mid + rng.uniform(-half, half, (n, 3)) * [1, 0.4, 1] - o
    r[:, 0:3] = o
    r[:, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
    r[:, 3] = 1e-4
    # line of sight: up to the other point, or to a distance around the camera's target
    reach = np.linalg.norm(d, axis=1) if case.get("rays_from") != "camera" else rng.uniform(0.3, 2.0, n) * (
        np.linalg.norm(np.array(cam["target"]) - eye) + half)
    r[:, 7] = reach if case.get("any_hit") else 1e30
    return torch.from_numpy(r).cuda()


def _features(n, h, w, seed):
    """Noisy one-path images as the renderer hands them to the denoiser: smooth radiance under
    heavy-tailed noise, piecewise albedo and normals, depth."""
    g = torch.Generator(device="cuda").manual_seed(seed)

    def smooth(c, cells):
        lo = torch.rand((n, c, cells, cells), device="cuda", generator=g)
        return torch.nn.functional.interpolate(lo, size=(h, w), mode="bilinear").permute(0, 2, 3, 1)

    albedo = (smooth(3, 9) * 6).floor() / 6 * 0.8 + 0.1
    nrm = torch.nn.functional.normalize(smooth(3, 7) * 2 - 1, dim=-1)
    light = smooth(3, 5) * 2.0
    target = (albedo * light).contiguous()
    noise = -torch.log(torch.rand((n, h, w, 1), device="cuda", generator=g).clamp_min(1e-6))
    hit = (torch.rand((n, h, w, 1), device="cuda", generator=g) < 0.4).float() / 0.4
    depth = torch.log1p(smooth(1, 6) * 60.0) / 10
    x = torch.cat([target * noise * hit, albedo, nrm, depth], dim=-1).contiguous()
    return x, target


# ---------------------------------------------------------------- prepare
def prepare(case, seed):
    kind = case["kind"]
    if kind in ("infer", "train"):
        ctx = gk.Context(64, 64)
        net = gk.UNet.pretrained(ctx)
        n = case.get("batch", 1)
        x, target = _features(n, case["height"], case["width"], seed)
        st = {"case": case, "ctx": ctx, "net": net, "x": x, "target": target}
        if kind == "infer":
            st["out"] = torch.empty_like(target)
        else:
            st["grad"] = torch.empty(net.num_params(), device="cuda")
        return st
    if kind == "diff":
        ctx = gk.Context(case["width"], case["height"])
        scene, nmat = scenes.cornell_tiles(seed=seed % 1000003)
        ctx.upload(scene)
        base = list(scene.materials)
        g = torch.Generator().manual_seed(seed)
        theta = diff.params_of(base)
        theta[:nmat] = (theta[:nmat] + 0.05 * torch.randn(nmat, 5, generator=g)).clamp(0.02, 0.98)
        cam = scenes.CORNELL_CAM
        p = gk.make_frame_params(cam["eye"], cam["target"], case["width"], case["height"], fov=cam["fov"])
        p.estimator = gk.ESTIMATOR_PT_MIS
        p.samples, p.bounces, p.max_bounces = case["samples"], case["bounces"], case["bounces"]
        p.total_frames, p.global_seed = 1, 1 + seed % 100003
        target = torch.full((case["height"], case["width"], 3), 0.35)
        target += 0.1 * torch.rand(target.shape, generator=g)
        return {"case": case, "ctx": ctx, "base": base, "theta": theta.cuda(), "params": p, "target": target.cuda()}
    scene, bricks, cam, half = _scene(case, seed)
    if case.get("textured"):
        _textures(scene, seed)
    st = {"case": case, "scene": scene}
    if kind == "frame":
        w, h = gk.render_extent(case["width"], case["height"], case["super_resolution"])
        ctx = gk.Context(w, h)
        ctx.upload(scene)
        if case["sky"] == "image":
            ctx.sky_upload(_sky_image(seed))
        if case["denoiser"] == "unet":
            st["net"] = gk.UNet.pretrained(ctx)
        moved = 10.0 if case["scene"] == "city" else 1.0
        frames, prev = [], None
        for f in range(case["frames"]):
            p = _params(case, seed, cam, w, h, f + 1, prev, moved)
            if f == 0:
                p.temporal_frames = 1  # a cut: the first frame takes nothing from history
            if bricks is not None:
                p.flags |= gk.FRAME_TLAS_REBUILD
            frames.append(p)
            prev = p
        st["frames"] = frames
        if bricks is not None:
            worlds = np.stack([bricks.worlds((seed % 64 + f) / 60.0) for f in range(case["frames"])])
            st["worlds"] = torch.from_numpy(np.ascontiguousarray(np.transpose(worlds, (0, 1, 3, 2)))).cuda()
        if case["probes"]:
            ctx.frame(frames[0])
            span = 2.2 * half if case["scene"] == "city" else 1.2
            ctx.probes_init(48, 16, span / 48, (-span / 2, -0.1, -span / 2) if case["scene"] == "city" else
                            (-0.1, -0.1, -0.1))
            ctx.probes_voxelize()
            ctx.probes_bake()
        if case["super_resolution"] != 2:
            st["shown"] = torch.empty((case["height"], case["width"], 4), dtype=torch.float16, device="cuda")
        st["out"] = {k: _target(ctx, k) for k in ("DENOISED", "ACCUM_DIFFUSE", "ACCUM_SPECULAR", "ACCUM_ALBEDO",
                                                  "NORMAL", "OBJECTID_0", "MOTIONVECTOR")}
        ctx.sync()
        st["ctx"] = ctx
        return st
    ctx = gk.Context(64, 64)
    st["ctx"] = ctx
    if kind == "probes":
        ctx.upload(scene)
        if case["sky"] == "image":
            ctx.sky_upload(_sky_image(seed))
        p = gk.make_frame_params(cam["eye"], cam["target"], 64, 64, fov=cam["fov"])
        _light(p, case)
        ctx.frame(p)
        n = case["size_xy"]
        span = 1.2 * half if case["scene"] == "city" else 1.3
        at = [-span / 2, -0.3, -span / 2] if case["scene"] == "city" else [-0.15, -0.15, -0.15]
        at = [float(a + b) for a, b in zip(at, np.random.default_rng([seed, 41]).uniform(-0.5, 0.5, 3) * span / n)]
        st["grid"] = (n, case["size_z"], span / n, tuple(at))
        return st
    st["rays"] = _rays(case, seed, cam, half)
    st["hits"] = torch.empty((case["rays"], 4), device="cuda")
    st["inst"] = torch.empty(case["rays"], dtype=torch.int32, device="cuda")
    if kind == "cast":
        ctx.upload(scene)
    return st


# ---------------------------------------------------------------- run
def _cast(st):
    ctx, case = st["ctx"], st["case"]
    any_hit = bool(case.get("any_hit"))
    ctx.trace(st["rays"].data_ptr(), case["rays"], st["hits"].data_ptr(), None if any_hit else st["inst"].data_ptr(),
              any_hit=any_hit)
    ctx.sync()  # the caller reads the answers
    words = st["hits"].view(torch.int32)
    if any_hit:
        return {"occluded": words[:, 3]}
    return {"t": st["hits"][:, 0], "uv": st["hits"][:, 1:3], "prim": words[:, 3], "inst": st["inst"]}


def run(st):
    case, kind, ctx = st["case"], st["case"]["kind"], st["ctx"]
    if kind == "frame":
        ctx.reset()
        for f, p in enumerate(st["frames"]):
            if "worlds" in st:
                w = st["worlds"][f]
                for _ in range(2 if f == 0 else 1):  # placed twice at the cut: no motion in the first frame
                    gk.check(gk.lib().gk_instances_update_device(ctx.h, w.data_ptr(), 0, w.shape[0]),
                             "gk_instances_update_device")
            ctx.frame(p)
            ctx.render()
        if "shown" in st:
            ctx.upscale(case["width"], case["height"],
                        gk.UPSCALE_FSR_EASU if case["super_resolution"] == 1 else gk.UPSCALE_LINEAR,
                        st["shown"].data_ptr())
            return {**st["out"], "shown": st["shown"]}
        return st["out"]
    if kind == "diff":
        theta = st["theta"].detach().requires_grad_(True)
        img = diff.render(theta, ctx, st["base"], st["params"])
        loss = ((img - st["target"]) ** 2).mean()
        loss.backward()
        return {"image": img.detach(), "grad": theta.grad, "loss": loss.detach()}
    if kind == "infer":
        st["net"].infer(st["x"].data_ptr(), st["out"].data_ptr(), case["height"], case["width"])
        return st["out"]
    if kind == "train":
        loss = st["net"].grad(st["x"].data_ptr(), st["target"].data_ptr(), case["batch"], case["height"],
                              case["width"], st["grad"].data_ptr())
        return {"grad": st["grad"], "loss": loss}
    if kind == "probes":
        n, nz, unit, off = st["grid"]
        ctx.probes_init(n, nz, unit, off)
        ctx.probes_voxelize()
        for _ in range(case["passes"]):
            ctx.probes_bake()
        cubes, vox = ctx.probes_read()
        return {"cubes": cubes.view(np.int32).reshape(-1, 14), "voxels": vox.view(np.int32).reshape(-1, 4)}
    if kind == "load":
        ctx.upload(st["scene"])
    return _cast(st)


# ---------------------------------------------------------------- work, tolerance, exact values
RAY, VERTEX, PIXEL = 52, 244, 70  # bytes: a ray and its hit, a shaded vertex, a pixel's images


def _net_flops(w, h):
    px = lambda lv: ((w + (1 << lv) - 1) >> lv) * ((h + (1 << lv) - 1) >> lv)  # noqa: E731
    layers = [(10, 32, 0), (32, 32, 0), (32, 48, 1), (48, 64, 2), (64, 96, 3), (96, 128, 4), (224, 96, 3),
              (160, 64, 2), (112, 48, 1), (80, 32, 0), (32, 32, 0), (32, 3, 0)]
    return sum(18.0 * ci * co * px(lv) for ci, co, lv in layers)


def _scene_bytes(case):
    if case["scene"] == "city":
        return 75.0 * (224.0 * case["grid"] ** 2)  # nodes and triangles of about 224 triangles per lot
    if case["scene"] == "bricks":
        return 288.0 * case["grid"] ** 3
    return 8e3


def work(case):
    kind = case["kind"]
    if kind == "frame":
        w, h = gk.render_extent(case["width"], case["height"], case["super_resolution"])
        paths = w * h * case["samples"]
        per = min(case["bounces"], 2.5)  # vertices of a path after the first, on these scenes
        rays = paths * (1 + per * (1.6 if case["estimator"] == "pt_mis" else 1.1))
        b = RAY * rays + VERTEX * paths * (1 + per) + PIXEL * w * h + _scene_bytes(case)
        fl = 1500.0 * rays
        if case["denoiser"] == "unet":
            fl += _net_flops(w, h)
            b += 50.0 * w * h
        return {"bytes": b * case["frames"], "flops": fl * case["frames"]}
    if kind == "diff":
        paths = case["width"] * case["height"] * case["samples"]
        rays = paths * (1 + 1.8 * min(case["bounces"], 3)) * 2
        return {"bytes": 44.0 * case["width"] * case["height"], "flops": 600.0 * rays}
    if kind == "infer":
        return {"bytes": 52.0 * case["width"] * case["height"], "flops": _net_flops(case["width"], case["height"])}
    if kind == "train":
        px = case["batch"] * case["width"] * case["height"]
        return {"bytes": 52.0 * px + 8.0 * 611328, "flops": 3.0 * case["batch"] * _net_flops(case["width"], case["height"])}
    if kind == "cast":
        return {"bytes": 52.0 * case["rays"], "flops": 1500.0 * case["rays"]}
    if kind == "probes":
        n = case["size_xy"] ** 2 * case["size_z"]
        rays = n * (14 + 102.0 * 0.8 * case["passes"])
        return {"bytes": 72.0 * n * (2 + case["passes"]) + _scene_bytes(case), "flops": 1000.0 * rays}
    tris = {"city": 224.0 * case["grid"] ** 2, "bricks": 24.0, "cornell": 36.0}[case["scene"]]
    return {"bytes": 250.0 * tris + _scene_bytes(case) + 52.0 * case["rays"], "flops": 200.0 * tris}


def tolerance(case):
    kind = case["kind"]
    if kind == "frame":
        # images in 16-bit floats: one rounding is 5e-4 of a value; the network's layers are bf16
        return {"rel": 1e-2, "max": 0.2} if case["denoiser"] == "unet" else {"rel": 1e-3, "max": 2e-2}
    if kind == "diff":
        return {"rel": 1e-4, "max": 1e-2}  # 32-bit sums over a million paths of both signs
    if kind == "infer":
        return {"rel": 1e-2, "max": 0.2}
    if kind == "train":
        return {"rel": 2e-2, "max": 0.5}
    if kind in ("cast", "load"):
        return {"rel": 1e-6, "max": 1e-4}
    return "exact"


def _net_layers(net):
    out = []
    w = _view(net.ctx, net.params_ptr(), (net.num_params(),), "<f4").double()
    for i in range(net.LAYERS):
        L = net.layer(i)
        cin = L.cin_a + L.cin_b
        rows = w[L.offset:L.offset + L.cout * L.kpad].reshape(L.cout, L.kpad)
        out.append((rows[:, :9 * cin].reshape(L.cout, 9, cin), rows[:, 9 * cin], L, rows))
    return out


def _net_forward(layers, x):
    """The network in 64 bits: x (n, h, w, 10), h and w multiples of 16 -> (n, h, w, 3) log radiance."""

    def conv(t, i):
        wt, bias, L, _ = layers[i]
        n, h, w, c = t.shape
        p = torch.nn.functional.pad(t, (0, 0, 1, 1, 1, 1))
        acc = bias.expand(n * h * w, L.cout)
        for tap in range(9):
            acc = acc + p[:, tap // 3:tap // 3 + h, tap % 3:tap % 3 + w].reshape(-1, c) @ wt[:, tap].t()
        acc = acc.reshape(n, h, w, L.cout)
        return acc.relu() if L.relu else acc

    def pool(t):
        n, h, w, c = t.shape
        return t.reshape(n, h // 2, 2, w // 2, 2, c).mean(dim=(2, 4))

    def up(t, skip):
        return torch.cat([t.repeat_interleave(2, 1).repeat_interleave(2, 2), skip], dim=-1)

    f = torch.cat([torch.log1p(x[..., :3].clamp_min(0)), x[..., 3:], x.new_zeros(x.shape[:-1] + (6,))], dim=-1)
    s0 = conv(conv(f, 0), 1)
    s1 = conv(pool(s0), 2)
    s2 = conv(pool(s1), 3)
    s3 = conv(pool(s2), 4)
    t = conv(pool(s3), 5)
    for i, s in ((6, s3), (7, s2), (8, s1), (9, s0)):
        t = conv(up(t, s), i)
    return conv(conv(t, 10), 11)[..., :3]


def _closest(case, st):
    """Closest hits by testing every triangle, in 64 bits (single-level scenes)."""
    s = st["scene"]
    m = s.meshes[0]
    p = torch.from_numpy(m["positions"]).cuda().double()
    idx = torch.from_numpy(m["indices"].astype(np.int64)).cuda()
    v0, e1, e2 = p[idx[:, 0]], p[idx[:, 1]] - p[idx[:, 0]], p[idx[:, 2]] - p[idx[:, 0]]
    r = st["rays"].double()
    best = torch.full((r.shape[0],), math.inf, dtype=torch.float64, device="cuda")
    step = max(1, 20000000 // max(1, v0.shape[0]))
    for a in range(0, r.shape[0], step):
        o, d = r[a:a + step, None, 0:3], r[a:a + step, None, 4:7]
        hh = torch.linalg.cross(d.expand(-1, e2.shape[0], -1), e2[None].expand(d.shape[0], -1, -1))
        det = (e1 * hh).sum(-1)
        sv = o - v0
        f = 1 / det
        u = f * (sv * hh).sum(-1)
        q = torch.linalg.cross(sv, e1[None].expand_as(sv))
        v = f * (d * q).sum(-1)
        t = f * (e2 * q).sum(-1)
        ok = (det.abs() >= 1e-7) & (u >= 0) & (u <= 1) & (v >= 0) & (u + v <= 1) & (t > r[a:a + step, 3:4]) & (
            t < r[a:a + step, 7:8])
        best[a:a + step] = torch.where(ok, t, math.inf).min(1).values
    # which of two coincident triangles is named, and so its barycentrics, is a rule on 32-bit ties
    return {"t": best, "uv": None, "prim": None, "inst": None}


def exact(case, seed):
    """64-bit values where they exist: the network and its gradients, and ray hits found by
    testing every triangle. A rendered image is one draw of a random process whose branches
    depend on 32-bit comparisons, and has no such value."""
    kind = case["kind"]
    if kind in ("cast", "load"):
        tris = {"city": 224 * case["grid"] ** 2, "cornell": 36, "bricks": 0}[case["scene"]]
        if case.get("any_hit") or tris == 0 or tris * case["rays"] > 4e9:
            return None
        return _closest(case, prepare(case, seed))
    if kind not in ("infer", "train"):
        return None
    st = prepare(case, seed)
    layers = _net_layers(st["net"])
    x = st["x"].double()
    if kind == "infer":
        h, w = case["height"], case["width"]
        x = torch.nn.functional.pad(x, (0, 0, 0, -w % 16, 0, -h % 16))
        with torch.no_grad():
            z = _net_forward(layers, x)[0, :h, :w]
        return torch.expm1(z).clamp_min(0)[None]
    leaf = [rows.clone().requires_grad_(True) for _, _, _, rows in layers]
    live = []
    for r, (_, _, L, _) in zip(leaf, layers):
        cin = L.cin_a + L.cin_b
        live.append((r[:, :9 * cin].reshape(L.cout, 9, cin), r[:, 9 * cin], L, r))
    z = _net_forward(live, x)
    loss = ((z - torch.log1p(st["target"].double().clamp_min(0))) ** 2).mean()
    loss.backward()
    return {"grad": torch.cat([r.grad.reshape(-1) for r in leaf]), "loss": float(loss.detach())}
