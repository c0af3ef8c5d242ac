"""Adjoint of the differentiable PT_MIS (512x512 Cornell tiles, 256 materials).

Checks:
  * the GPU primal equals the oracle's double-precision detached render;
  * every adjoint gradient component tested equals the central finite difference of the
    oracle's detached render (BSDF values perturbed, sampling held), which pins the
    derivative formulas without restating them;
  * albedo gradients equal finite differences of the GPU primal itself (sampling does not
    depend on albedo, so the fixed-seed primal is differentiable in it);
  * the gradient drives an optimisation towards a perturbed target (loss decreases).
"""
from __future__ import annotations

import copy

import numpy as np
import pytest

import gknextengine_amd as gk
from gknextengine_amd import scenes
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def setup(W=48, H=48, spp=2, bounces=4):
    scene, nmat = scenes.cornell_tiles()
    cam = scenes.CORNELL_CAM
    p = gk.make_frame_params(cam["eye"], cam["target"], W, H, fov=cam["fov"])
    p.estimator = gk.ESTIMATOR_PT_MIS
    p.samples = spp
    p.bounces = p.max_bounces = bounces
    p.total_frames = 11
    p.global_seed = 5
    return scene, nmat, p


@pytest.mark.parametrize("instances", [1, 2])
def test_primal_matches_oracle_and_adjoint_matches_detached_fd(instances):
    import torch
    from gknextengine_amd import diff
    W = H = 48
    scene, nmat, p = setup(W, H)
    if instances == 2:  # the two-level traversal; the second box stands in view, beside the first
        w = np.diag(np.float32([0.5, 0.5, 0.5, 1.0]))
        w[:3, 3] = 0.25, 0.1, -0.6
        scene.add_instance(0, world=w)
    base = list(scene.materials)
    osc = po.OracleScene(scene)
    rng = np.random.default_rng(0)
    dL = rng.normal(size=(H, W, 3)).astype(np.float32)
    cpu_img = osc.diff_render(p, W, H, spp=p.samples, frame0=p.total_frames)
    with gk.Context(W, H) as ctx:
        ctx.upload(scene)
        params = diff.params_of(base).cuda().requires_grad_(True)
        img = diff.render(params, ctx, base, p, decorrelate=False)
        gpu_img = img.detach().cpu().numpy()
        close = np.all(np.abs(gpu_img - cpu_img) <= 1e-3 * (1 + np.abs(cpu_img)), axis=2)
        assert close.mean() > 0.98, close.mean()
        # A float path and a double path can part ways at a grazing hit or a shadow-ray
        # end point; the derivative check weighs only pixels whose paths agree.
        dL *= close[..., None]
        loss = (img * torch.from_numpy(dL).cuda()).sum()
        loss.backward()
        g = params.grad.cpu().numpy()
    # detached central differences on the oracle for a sample of parameters
    lit = np.nonzero(np.abs(g).sum(axis=1) > 0)[0]
    assert len(lit) > 20
    picks = [(int(m), k) for m in rng.choice(lit, 12, replace=False) for k in range(5)]
    h = 1e-4
    errs = []
    for m, k in picks:
        plus, minus = copy.deepcopy(base), copy.deepcopy(base)
        for mm, sign in ((plus, 1.0), (minus, -1.0)):
            x = mm[m]
            if k < 3:
                x.diffuse[k] += sign * h
            elif k == 3:
                x.fuzziness += sign * h
            else:
                x.metalness += sign * h
        ip = osc.diff_render(p, W, H, eval_materials=plus, spp=p.samples, frame0=p.total_frames)
        im = osc.diff_render(p, W, H, eval_materials=minus, spp=p.samples, frame0=p.total_frames)
        fd = float(((ip - im) / (2 * h) * dL).sum())
        errs.append((m, k, g[m, k], fd))
    gg = np.array([e[2] for e in errs])
    ff = np.array([e[3] for e in errs])
    scale = np.abs(ff).max()
    worst = int(np.argmax(np.abs(gg - ff)))
    assert np.abs(gg - ff).max() <= 2e-2 * scale + 1e-6, (errs[worst], list(zip(gg, ff)))
    assert np.corrcoef(gg, ff)[0, 1] > 0.999


def test_albedo_gradient_matches_gpu_finite_differences():
    import torch
    from gknextengine_amd import diff
    W = H = 48
    scene, nmat, p = setup(W, H, spp=2)
    base = list(scene.materials)
    rng = np.random.default_rng(1)
    dL = torch.from_numpy(rng.normal(size=(H, W, 3)).astype(np.float32)).cuda()
    with gk.Context(W, H) as ctx:
        ctx.upload(scene)
        params = diff.params_of(base).cuda().requires_grad_(True)
        (diff.render(params, ctx, base, p, decorrelate=False) * dL).sum().backward()
        g = params.grad.cpu().numpy()
        lit = np.nonzero(np.abs(g[:, :3]).sum(axis=1) > 0)[0]
        h = 1e-2
        for m in rng.choice(lit, 8, replace=False):
            for k in range(3):
                q = params.detach().clone()
                q[m, k] += h
                ip = diff.render(q, ctx, base, p)
                q[m, k] -= 2 * h
                im = diff.render(q, ctx, base, p)
                fd = float(((ip - im) / (2 * h) * dL).sum())
                assert fd == pytest.approx(float(g[m, k]), rel=2e-2, abs=2e-3 * abs(g[:, :3]).max())


def test_gradient_descent_reduces_image_loss():
    import torch
    from gknextengine_amd import diff
    W = H = 48
    scene, nmat, p = setup(W, H, spp=4)
    base = list(scene.materials)
    with gk.Context(W, H) as ctx:
        ctx.upload(scene)
        truth = diff.params_of(base).cuda()
        target = diff.render(truth, ctx, base, p).detach()
        gen = torch.Generator().manual_seed(3)
        start = truth.clone()
        start[:nmat, :3] = (start[:nmat, :3] + 0.15 * torch.randn(nmat, 3, generator=gen).cuda()).clamp(0.05, 0.95)
        params = start.clone().requires_grad_(True)
        opt = torch.optim.Adam([params], lr=0.02)
        losses = []
        for it in range(30):
            opt.zero_grad()
            loss = ((diff.render(params, ctx, base, p) - target) ** 2).mean()
            loss.backward()
            params.grad[nmat:] = 0  # the light is not a parameter
            params.grad[:, 3:] = 0  # fit albedo only
            opt.step()
            with torch.no_grad():
                params[:nmat, :3].clamp_(0.01, 0.99)
            losses.append(loss.item())
    assert losses[-1] < 0.3 * losses[0], losses


def test_backward_replays_its_own_forward_after_interleaved_renders():
    """Two renders (other materials, other seeds) before one backward: each backward
    replays the parameters and frame of its own forward, so the gradients equal those of
    the renders run one at a time."""
    import torch
    from gknextengine_amd import diff
    W = H = 32
    scene, nmat, p = setup(W, H, spp=2)
    q = gk.FrameParams.from_buffer_copy(p)
    q.total_frames, q.global_seed = 77, 9
    base = list(scene.materials)
    rng = np.random.default_rng(4)
    dL = torch.from_numpy(rng.normal(size=(H, W, 3)).astype(np.float32)).cuda()
    with gk.Context(W, H) as ctx:
        ctx.upload(scene)
        pa = diff.params_of(base).cuda()
        pb = pa.clone()
        pb[:nmat, :3] = (pb[:nmat, :3] * 0.7).clamp(0.01, 0.99)
        ga_ref, gb_ref = [], []
        for t, fr, out in ((pa, p, ga_ref), (pb, q, gb_ref)):
            x = t.clone().requires_grad_(True)
            (diff.render(x, ctx, base, fr) * dL).sum().backward()
            out.append(x.grad.clone())
        xa, xb = pa.clone().requires_grad_(True), pb.clone().requires_grad_(True)
        la = (diff.render(xa, ctx, base, p) * dL).sum()
        lb = (diff.render(xb, ctx, base, q) * dL).sum()
        lb.backward()
        la.backward()
        # (a work-group sums its gradient rows with LDS float atomics: last-bit differences)
        for g, r in ((xa.grad, ga_ref[0]), (xb.grad, gb_ref[0])):
            assert torch.allclose(g, r, rtol=1e-4, atol=1e-6 * float(r.abs().max())), (g - r).abs().max()
        assert not torch.allclose(ga_ref[0], gb_ref[0], rtol=1e-2)


def test_descent_recovers_perturbed_parameters_from_an_independent_target():
    """The differentiable render's set-up at reduced size: the target is a 2048-spp render with parameters
    perturbed by N(0, 0.05), drawn from seeds the optimisation never uses; plain
    loss.backward() (adjoint replayed with independent seeds) drives Adam back towards the
    target's albedos.

    Sizing: a material's albedo is recovered to within the noise of the pixels it covers.
    At 128x128 the well-lit tiles cover about 60 pixels each; the target's own noise at
    2048 spp moves their optimum by well under the 0.04 mean perturbation, and 16 spp per
    step keeps Adam's steps dominated by the signal until the error is a fraction of it."""
    import torch
    from gknextengine_amd import diff
    W = H = 128
    scene, nmat, p = setup(W, H, spp=16)
    base = list(scene.materials)
    with gk.Context(W, H) as ctx:
        ctx.upload(scene)
        theta = diff.params_of(base).cuda()
        gen = torch.Generator().manual_seed(12)
        truth = theta.clone()
        truth[:nmat, :3] = (truth[:nmat, :3] + 0.05 * torch.randn(nmat, 3, generator=gen).cuda()).clamp(0.02, 0.98)
        acc = torch.zeros((H, W, 3), device="cuda")
        for k in range(8):
            t = gk.FrameParams.from_buffer_copy(p)
            t.samples, t.total_frames, t.global_seed = 256, 1_000_000 + 256 * k, 99
            with torch.no_grad():
                acc += diff.render(truth, ctx, base, t)
        target = acc / 8
        # coverage: how strongly each material's albedo moves the image (64 spp)
        x = theta.clone().requires_grad_(True)
        c = gk.FrameParams.from_buffer_copy(p)
        c.samples, c.total_frames = 64, 500_000
        diff.render(x, ctx, base, c).sum().backward()
        cover = x.grad[:nmat, :3].abs().sum(dim=1)
        seen = cover > cover.max() * 0.2
        params = theta.clone().requires_grad_(True)
        opt = torch.optim.Adam([params], lr=0.005)
        err0 = (params[:nmat, :3] - truth[:nmat, :3]).abs()[seen].mean().item()
        losses = []
        for it in range(100):
            opt.zero_grad()
            f = gk.FrameParams.from_buffer_copy(p)
            f.total_frames = 100 + 16 * it
            loss = ((diff.render(params, ctx, base, f) - target) ** 2).mean()
            loss.backward()
            params.grad[nmat:] = 0
            params.grad[:, 3:] = 0
            opt.step()
            with torch.no_grad():
                params[:nmat, :3].clamp_(0.01, 0.99)
            losses.append(loss.item())
        err1 = (params[:nmat, :3] - truth[:nmat, :3]).abs()[seen].mean().item()
    print(f"albedo error over {int(seen.sum())} materials: {err0:.4f} -> {err1:.4f}; "
          f"loss {np.mean(losses[:5]):.3e} -> {np.mean(losses[-5:]):.3e}")
    assert err1 < 0.5 * err0, (err0, err1)


# tiles cut by the image's edge, one to five samples (one, two or four waves on a tile), a
# single bounce, many, and a scene of two instances (the two-level traversal)
@pytest.mark.parametrize("W,H,spp,bounces,instances", [(8, 8, 1, 1, 1), (13, 29, 2, 4, 1), (50, 41, 3, 4, 2),
                                                       (33, 16, 5, 12, 1), (64, 64, 4, 64, 2)])
def test_shapes_match_oracle_and_single_samples(W, H, spp, bounces, instances):
    """The image equals the oracle's render; the image and the gradient of spp samples are the
    means of those of the samples rendered one at a time (32-bit sums in another order)."""
    import torch
    from gknextengine_amd import diff
    scene, nmat, p = setup(W, H, spp, bounces)
    if instances == 2:
        w = np.eye(4, dtype=np.float32)
        w[0, 3] = 1.5
        scene.add_instance(0, world=w)
    base = list(scene.materials)
    dL = torch.from_numpy(np.random.default_rng(W).normal(size=(H, W, 3)).astype(np.float32)).cuda()
    ref = po.OracleScene(scene).diff_render(p, W, H, spp=spp, frame0=p.total_frames)

    def both(q):
        x = diff.params_of(base).cuda().requires_grad_(True)
        img = diff.render(x, ctx, base, q, decorrelate=False)
        (img * dL).sum().backward()
        return img.detach(), x.grad

    with gk.Context(W, H) as ctx:
        ctx.upload(scene)
        img, g = both(p)
        parts = []
        for k in range(spp):
            q = gk.FrameParams.from_buffer_copy(p)
            q.samples, q.total_frames = 1, p.total_frames + k
            parts.append(both(q))
    close = np.all(np.abs(img.cpu().numpy() - ref) <= 1e-3 * (1 + np.abs(ref)), axis=2)
    assert close.mean() > 0.95, close.mean()
    mean_img = sum(a for a, _ in parts) / spp
    mean_g = sum(b for _, b in parts) / spp
    assert torch.allclose(img, mean_img, rtol=1e-5, atol=1e-6)
    assert torch.allclose(g, mean_g, rtol=1e-4, atol=2e-6 * float(mean_g.abs().max())), (g - mean_g).abs().max()


@pytest.mark.parametrize("count", [600, 2458, 3276])
def test_material_count_up_to_the_limit(count):
    """Materials no triangle uses get a zero gradient and leave the others' unchanged, up to the
    3276 whose sums fit the work-groups (2458 and more pass 64 KB of LDS with the stacks)."""
    import torch
    from gknextengine_amd import diff
    W = H = 24
    scene, nmat, p = setup(W, H, spp=2)
    base = list(scene.materials)
    dL = torch.from_numpy(np.random.default_rng(8).normal(size=(H, W, 3)).astype(np.float32)).cuda()
    grads = []
    for mats in (base, base + [copy.deepcopy(base[0]) for _ in range(count - len(base))]):
        scene.materials = mats
        with gk.Context(W, H) as ctx:
            ctx.upload(scene)
            x = diff.params_of(mats).cuda().requires_grad_(True)
            (diff.render(x, ctx, mats, p, decorrelate=False) * dL).sum().backward()
            grads.append(x.grad.clone())
    n = len(base)
    assert torch.all(grads[1][n:] == 0)
    assert torch.allclose(grads[1][:n], grads[0], rtol=1e-4, atol=2e-6 * float(grads[0].abs().max()))


def _plain_gradient(ctx, scene, p, dL):
    """The gradient of sum(image * dL) by gk_adjoint itself, on paths of p's own seed."""
    import torch
    g = torch.empty((len(scene.materials), 5), dtype=torch.float32, device="cuda")
    ctx.frame(p)
    torch.cuda.synchronize()
    gk.check(gk.lib().gk_adjoint(ctx.h, dL.data_ptr(), g.data_ptr()), "gk_adjoint")
    ctx.sync()
    return g


def test_time_does_not_depend_on_a_bounce_limit_no_path_reaches():
    """Paths that end at their second vertex cost the same whatever the limit: the launch keeps
    its work-groups. (Records kept to 96 MB gave 170 work-groups at 64 bounces, 2.3 times as long.)"""
    import time

    import torch
    W = H = 512
    scene = gk.SceneData()
    scene.add_mesh([[-50, 0, -50], [50, 0, -50], [50, 0, 50], [-50, 0, 50]], [[0, 2, 1], [0, 3, 2]])
    scene.materials = [scenes.material((0.4, 0.6, 0.8))]
    scene.add_instance(0)
    p = gk.make_frame_params((0, 3, -4), (0, 0, 0), W, H, fov=50.0)
    p.estimator, p.samples, p.has_sky, p.total_frames = gk.ESTIMATOR_PT_MIS, 4, 1, 1
    p.sky_color[:] = [0.5, 0.5, 0.5, 1.0]
    dL = torch.ones((H, W, 4), dtype=torch.float32, device="cuda")
    best, grads = {}, {}
    with gk.Context(W, H) as ctx:
        ctx.upload(scene)
        for turn in range(6):
            for b in (4, 64):
                p.bounces = p.max_bounces = b
                grads[b] = _plain_gradient(ctx, scene, p, dL)
                g = torch.empty_like(grads[b])
                t = time.perf_counter()
                for _ in range(10):
                    gk.check(gk.lib().gk_adjoint(ctx.h, dL.data_ptr(), g.data_ptr()), "gk_adjoint")
                ctx.sync()
                best[b] = min(best.get(b, 1e9), time.perf_counter() - t)
    assert best[64] < 1.5 * best[4], best
    assert float(grads[4].abs().max()) > 0
    # (LDS float atomics: the order of a work-group's additions differs from run to run)
    assert torch.allclose(grads[4], grads[64], rtol=1e-5)


def test_records_that_do_not_fit_take_fewer_work_groups(tmp_path):
    """With 250 MB of device memory the 604 MB of records of a 64-bounce gradient over 512 x 512
    pixels do not fit: fewer work-groups take the image in turns, each using its records and its
    sums for several tiles, and the gradient is the same. (A child process: the limit is read
    once per process.)"""
    import os
    import subprocess
    import sys
    import textwrap
    from pathlib import Path
    code = textwrap.dedent("""
        import sys
        sys.path.insert(0, %r)
        import numpy as np
        import torch
        import gknextengine_amd as gk
        from tests.test_gpu_adjoint import _plain_gradient, setup
        W = H = 512
        scene, nmat, p = setup(W, H, spp=4, bounces=64)
        dL = torch.from_numpy(np.random.default_rng(3).normal(size=(H, W, 4)).astype(np.float32)).cuda()
        with gk.Context(W, H) as ctx:
            ctx.upload(scene)
            np.save(sys.argv[1], _plain_gradient(ctx, scene, p, dL).cpu().numpy())
    """) % (str(Path(__file__).resolve().parents[1]),)
    out = []
    for name, limit in (("all", None), ("few", 250 * 1000 * 1000)):
        env = dict(os.environ)
        if limit:
            env["GKNX_DEVICE_MEMORY_LIMIT"] = str(limit)
        f = tmp_path / f"{name}.npy"
        r = subprocess.run([sys.executable, "-c", code, str(f)], env=env, capture_output=True, text=True, timeout=100)
        assert r.returncode == 0, r.stderr[-2000:]
        out.append(np.load(f))
    assert np.abs(out[0]).max() > 0
    np.testing.assert_allclose(out[1], out[0], rtol=1e-4, atol=2e-6 * np.abs(out[0]).max())


def test_sums_of_32_bits_hold_256_pixels():
    """512 x 576 pixels at one sample are 1152 tile groups of 256 pixels on 1024 work-groups. A
    pixel of group 0 weighs 2^20, one of group 1 cancels it, and the 64 of a tile of group 1024,
    which the work-group of group 0 takes next and by the same wave, weigh 2^-6: added to the
    first pixel's share in 32 bits each is below half of its last bit and is lost. (The order
    within a wave's tile aside, nothing here depends on timing.)"""
    import torch
    W, H = 512, 576
    scene = gk.SceneData()
    scene.add_mesh([[-50, 0, -50], [50, 0, -50], [50, 0, 50], [-50, 0, 50]], [[0, 2, 1], [0, 3, 2]])
    scene.materials = [scenes.material((0.5, 0.5, 0.5))]
    scene.add_instance(0)
    p = gk.make_frame_params((0, 3, -4), (0, 0, 0), W, H, fov=40.0)
    p.estimator, p.samples, p.has_sky, p.total_frames = gk.ESTIMATOR_PT_MIS, 1, 1, 1
    p.bounces = p.max_bounces = 2
    p.sky_color[:] = [0.5, 0.5, 0.5, 1.0]
    zero = torch.zeros((H, W, 4), dtype=torch.float32, device="cuda")
    with gk.Context(W, H) as ctx:
        ctx.upload(scene)

        def grad(*parts):  # (y, x, tile edge, weight)
            dL = zero.clone()
            for y, x, n, w in parts:
                dL[y:y + n, x:x + n, :3] = w
            return _plain_gradient(ctx, scene, p, dL)[0, :3].double()

        def lit(x0, w):  # a pixel of the tile whose one path takes the diffuse lobe and meets the sky
            return next(q for q in ((y, x, 1, w) for y in range(8) for x in range(x0, x0 + 8)) if grad(q)[0] != 0)

        big = lit(0, 2.0 ** 20), lit(32, -2.0 ** 20)
        small = (512, 0, 8, 2.0 ** -6)
        ga, gb, gs, g = grad(big[0]), grad(big[1]), grad(small), grad(*big, small)
    assert torch.all(ga > 2.0 ** 17) and torch.all(gs > 0.1) and torch.all((ga + gb).abs() < 2.0 ** -3 * ga)
    # g is one rounding to 32 bits of the sum of the three
    want = ga + gb + gs
    assert torch.all((g - want).abs() <= 2.0 ** -23 * want.abs() + 0.05 * gs), (g, want, gs)


# 64-pixel tile groups at four samples, 256-pixel ones at one; 1024 work-groups in one level, 768
# in two: groups beyond them by a few, and several turns of 256 pixels
@pytest.mark.parametrize("W,H,spp,bounces,instances", [(264, 264, 4, 4, 1), (520, 520, 1, 3, 1), (768, 701, 1, 3, 2),
                                                       (224, 232, 4, 4, 2), (800, 600, 4, 2, 1)])
def test_work_groups_that_take_several_tile_groups(W, H, spp, bounces, instances):
    """More tile groups than work-groups, so that one uses its records and sums again: the gradient
    is the sum of gradients whose image derivative is masked to as many groups as work-groups."""
    import torch
    scene, nmat, p = setup(W, H, spp, bounces)
    if instances == 2:
        w = np.eye(4, dtype=np.float32)
        w[0, 3] = 1.5
        scene.add_instance(0, world=w)
    per = {1: 4, 2: 2, 4: 1}[spp]  # tiles of a group
    blocks = 1024 if instances == 1 else 768
    tx, ty = -(-W // 8), -(-H // 8)
    group = (np.arange(ty)[:, None] * tx + np.arange(tx)[None, :]) // per
    part = torch.from_numpy(np.kron(group // blocks, np.ones((8, 8), np.int64))[:H, :W]).cuda()
    assert int(part.max()) >= 1
    dL = torch.from_numpy(np.random.default_rng(W).normal(size=(H, W, 4)).astype(np.float32)).cuda()
    with gk.Context(W, H) as ctx:
        ctx.upload(scene)
        whole = _plain_gradient(ctx, scene, p, dL)
        parts = [_plain_gradient(ctx, scene, p, dL * (part == k)[..., None]) for k in range(int(part.max()) + 1)]
    want = sum(g.double() for g in parts)
    assert all(float(g.abs().max()) > 0 for g in parts)
    assert torch.allclose(whole.double(), want, rtol=1e-4, atol=2e-6 * float(want.abs().max())), (whole - want).abs().max()
