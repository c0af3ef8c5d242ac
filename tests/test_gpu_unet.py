"""Learned denoiser on the GPU against the CPU oracle (oracle/unet_oracle.py).

The oracle runs in its bf16 mode (rounding where the GPU stores bfloat16), so the GPU and
the oracle differ by the summation order of FP32 accumulations and by the rare bf16
rounding that order flips; the tolerances below are set for that.
"""
from __future__ import annotations

import numpy as np
import pytest

import gknextengine_amd as gk
from oracle import unet_oracle as U
from tests import scenes

pytestmark = pytest.mark.gpu


def features(rng, n, h, w):
    nrm = rng.normal(size=(n, h, w, 3))
    nrm /= np.linalg.norm(nrm, axis=3, keepdims=True)
    return np.concatenate([rng.gamma(0.4, 2.5, (n, h, w, 3)), rng.uniform(0, 1, (n, h, w, 3)), nrm,
                           rng.uniform(0, 1, (n, h, w, 1))], axis=3).astype(np.float32)


def rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


def test_layer_table_matches_oracle():
    with gk.Context(16, 16) as ctx:
        net = gk.UNet(ctx, 32, seed=1)
        assert net.num_params() == U.num_params(32)
        for i, L in enumerate(U.layers(32)):
            g = net.layer(i)
            assert {k: getattr(g, k) for k in L} == L, i
        p = net.get_params()
        # He-normal over the real inputs, zero bias and padding
        L0 = U.layers(32)[0]
        M = p[:L0["cout"] * L0["kpad"]].reshape(L0["cout"], L0["kpad"])
        assert np.all(M[:, 9 * 16:] == 0) and np.all(M[:, :144].reshape(32, 9, 16)[:, :, 10:] == 0)
        assert abs(M[:, :144].reshape(32, 9, 16)[:, :, :10].std() - np.sqrt(2 / 90)) < 0.02


def test_forward_matches_oracle_with_padding():
    import torch
    rng = np.random.default_rng(0)
    # padded to 48 x 64 inside: every level even, so every convolution stages its input tile
    # in LDS, the level-3 decoder's 86 KB tile (above the default 64 KB) included
    h, w = 40, 56
    f = features(rng, 1, h, w)
    with gk.Context(16, 16) as ctx:
        net = gk.UNet(ctx, 32, seed=2)
        p = net.get_params()
        p += (rng.normal(0, 0.02, p.shape) * (p != 0)).astype(np.float32)  # move off the init
        for L in U.layers(32):  # biases
            cin = L["cin_a"] + L["cin_b"]
            idx = L["offset"] + np.arange(L["cout_real"]) * L["kpad"] + 9 * cin
            p[idx] = rng.normal(0, 0.05, L["cout_real"])
        net.set_params(p)
        d_in = torch.from_numpy(f).cuda()
        d_out = torch.empty(h * w * 3, device="cuda")
        net.infer(d_in.data_ptr(), d_out.data_ptr(), h, w)
        torch.cuda.synchronize()
        gpu = d_out.cpu().numpy().reshape(h, w, 3)
    fp = np.zeros((1, 48, 64, 10), np.float32)
    fp[:, :h, :w] = f
    ref = U.infer(p, fp, 32, bf16_mode=True)[0, :h, :w]
    assert rel(gpu, ref) < 5e-3, rel(gpu, ref)
    assert np.abs(gpu - ref).max() < 2e-2 * np.abs(ref).max()


def test_gradient_matches_oracle():
    import torch
    rng = np.random.default_rng(1)
    n, h, w = 2, 32, 32
    f = features(rng, n, h, w)
    t = rng.gamma(1.0, 1.0, (n, h, w, 3)).astype(np.float32)
    with gk.Context(16, 16) as ctx:
        net = gk.UNet(ctx, 32, seed=3)
        p = net.get_params()
        d_in, d_t = torch.from_numpy(f).cuda(), torch.from_numpy(t).cuda()
        d_g = torch.empty(net.num_params(), device="cuda")
        loss = net.grad(d_in.data_ptr(), d_t.data_ptr(), n, h, w, d_g.data_ptr())
        g = d_g.cpu().numpy()
    lo, go = U.loss_grad(p, f, t, 32, bf16_mode=True)
    assert loss == pytest.approx(lo, rel=2e-3)
    for i, L in enumerate(U.layers(32)):
        sl = slice(L["offset"], L["offset"] + L["cout"] * L["kpad"])
        a, b = g[sl], go[sl]
        cos = float(a @ b / (np.linalg.norm(a) * np.linalg.norm(b)))
        assert rel(a, b) < 3e-2 and cos > 0.999, (i, rel(a, b), cos)
    pad = np.ones(go.size, bool)  # padding parameters get exactly zero gradient
    for i, L in enumerate(U.layers(32)):
        cin = L["cin_a"] + L["cin_b"]
        cin_real = U.IN_CH if i == 0 else cin
        M = pad[L["offset"]:L["offset"] + L["cout"] * L["kpad"]].reshape(L["cout"], L["kpad"])
        for tap in range(9):
            M[:L["cout_real"], tap * cin:tap * cin + cin_real] = False
        M[:L["cout_real"], 9 * cin] = False
    assert np.all(g[pad] == 0)


# widths that are no multiple of a 32-pixel tile row at any level, heights that end inside a
# tile, a single pixel at the coarsest level, and channel counts that take every split of the
# weight gradient's waves (1 to 8 input groups, 1 to 3 output tiles, odd and even segments)
@pytest.mark.parametrize("base,n,h,w", [(32, 1, 16, 16), (32, 2, 48, 80), (8, 3, 64, 32), (16, 1, 16, 112),
                                        (40, 1, 32, 48), (64, 1, 32, 48)])
def test_gradient_shapes_match_oracle(base, n, h, w):
    """As test_gradient_matches_oracle (same bounds: bf16 roundings that the summation order
    flips), and the same bits on a second call: every sum has a fixed order."""
    import torch
    rng = np.random.default_rng(base + h)
    f = features(rng, n, h, w)
    t = rng.gamma(1.0, 1.0, (n, h, w, 3)).astype(np.float32)
    with gk.Context(16, 16) as ctx:
        net = gk.UNet(ctx, base, seed=3)
        p = net.get_params()
        d_in, d_t = torch.from_numpy(f).cuda(), torch.from_numpy(t).cuda()
        d_g = torch.full((2, net.num_params()), float("nan"), device="cuda")
        loss = [net.grad(d_in.data_ptr(), d_t.data_ptr(), n, h, w, d_g[k].data_ptr()) for k in (0, 1)]
        g = d_g.cpu().numpy()
    assert np.array_equal(g[0], g[1])
    lo, go = U.loss_grad(p, f, t, base, bf16_mode=True)
    assert loss[0] == pytest.approx(lo, rel=2e-3)
    for i, L in enumerate(U.layers(base)):
        sl = slice(L["offset"], L["offset"] + L["cout"] * L["kpad"])
        a, b = g[0][sl], go[sl]
        cos = float(a @ b / (np.linalg.norm(a) * np.linalg.norm(b)))
        assert rel(a, b) < 3e-2 and cos > 0.999, (i, rel(a, b), cos)
        M, cin = a.reshape(L["cout"], L["kpad"]), L["cin_a"] + L["cin_b"]
        assert np.all(M[:, 9 * cin + 1:] == 0)  # padding columns


def test_adam_step_and_save_load():
    import torch
    rng = np.random.default_rng(2)
    n, h, w = 1, 32, 32
    f = features(rng, n, h, w)
    t = rng.gamma(1.0, 1.0, (n, h, w, 3)).astype(np.float32)
    with gk.Context(16, 16) as ctx:
        net = gk.UNet(ctx, 32, seed=4)
        p0 = net.get_params()
        d_in, d_t = torch.from_numpy(f).cuda(), torch.from_numpy(t).cuda()
        d_g = torch.empty(net.num_params(), device="cuda")
        net.grad(d_in.data_ptr(), d_t.data_ptr(), n, h, w, d_g.data_ptr())
        g = d_g.cpu().numpy()
        net.train_step(d_in.data_ptr(), d_t.data_ptr(), n, h, w, 1e-3)
        p1 = net.get_params()
        ref, _, _ = U.adam(p0, g, np.zeros_like(p0), np.zeros_like(p0), 1, 1e-3)
        assert np.abs(p1 - ref).max() < 1e-6
        assert np.all(p1[g == 0] == p0[g == 0])
        net.set_params(p0)
        assert np.array_equal(net.get_params(), p0)


def test_training_reduces_loss():
    import torch
    rng = np.random.default_rng(3)
    n, h, w = 4, 64, 64
    # smooth radiance + noise: the network has to learn to smooth
    yy, xx = np.mgrid[0:h, 0:w] / 64.0
    clean = np.stack([1 + np.sin(6 * xx + 3 * k) * np.cos(4 * yy) for k in range(3)], axis=2)
    clean = np.broadcast_to(clean, (n, h, w, 3)).astype(np.float32)
    f = features(rng, n, h, w)
    f[..., :3] = clean * rng.gamma(1.0, 1.0, clean.shape)
    with gk.Context(16, 16) as ctx:
        net = gk.UNet(ctx, 32, seed=5)
        d_in, d_t = torch.from_numpy(f).cuda(), torch.from_numpy(np.ascontiguousarray(clean)).cuda()
        losses = [net.train_step(d_in.data_ptr(), d_t.data_ptr(), n, h, w, 1e-3) for _ in range(60)]
    assert np.all(np.isfinite(losses))
    assert np.mean(losses[-5:]) < 0.3 * losses[0], losses[::10]


def test_frame_denoiser_path_equals_infer():
    import torch

    from bench import gt_tonemap
    from gknextengine_amd import scenes
    W = H = 64
    s = gk.procgen_cornell()
    cam = scenes.CORNELL_CAM
    p = gk.make_frame_params(cam["eye"], cam["target"], W, H, fov=cam["fov"])
    p.estimator = gk.ESTIMATOR_PT_MIS
    p.temporal_frames = 1
    p.denoiser = gk.DENOISER_UNET
    with gk.Context(W, H) as ctx:
        ctx.upload(s)
        net = gk.UNet(ctx, 32, seed=6)
        ctx.frame(p)
        ctx.render()
        ctx.sync()
        den = ctx.read("DENOISED")[..., :3].astype(np.float32)
        d_f = torch.empty(W * H * 10, device="cuda")
        ctx.denoise_input(d_f.data_ptr())
        d_o = torch.empty(W * H * 3, device="cuda")
        net.infer(d_f.data_ptr(), d_o.data_ptr(), H, W)
        torch.cuda.synchronize()
        out = d_o.cpu().numpy().reshape(H, W, 3)
        feats = d_f.cpu().numpy().reshape(H, W, 10)
    expect = gt_tonemap(out * (p.paper_white_nit / 40000.0))
    assert np.abs(den - expect).max() < 2e-3
    # features: radiance = accumulated diffuse * albedo + specular; albedo; normal; depth
    assert np.all(feats[..., :3] >= 0) and np.all(np.abs(np.linalg.norm(feats[..., 6:9], axis=2) - 1) < 1e-2)
    assert np.all((feats[..., 9] >= 0) & (feats[..., 9] <= 1))


def test_trained_network_beats_bilateral_on_new_views():
    """The shipped weights (gknextengine_amd/weights, trained by denoise_train on its own
    rendered pairs) against the bilateral filter on the same 1-spp frames of views drawn from
    a seed the training did not use; relMSE of linear radiance against a 1024-spp render."""
    import torch

    from bench import relmse_stats
    from gknextengine_amd import denoise_train as dt
    pr = dt.PairRenderer()
    try:
        net = gk.UNet.pretrained(pr.ctx["city"])
        rng = np.random.default_rng(777)
        d_feat = torch.empty((dt.TILE, dt.TILE, gk.UNet.IN_CHANNELS), device="cuda")
        out = torch.empty(dt.TILE * dt.TILE * 3, device="cuda")
        for which in ("cornell", "city", "city"):
            view = dt.cornell_view(rng) if which == "cornell" else dt.city_view(rng)
            tgt, bil = pr.pair(which, view, int(rng.integers(1 << 30)), int(rng.integers(1 << 20)), 1024,
                               d_feat.data_ptr())
            net.infer(d_feat.data_ptr(), out.data_ptr(), dt.TILE, dt.TILE)
            net.ctx.sync()
            u = out.cpu().numpy().reshape(dt.TILE, dt.TILE, 3)
            rb, rb_finite, _ = relmse_stats(bil, tgt)
            ru, _, nu = relmse_stats(u, tgt)
            noisy = relmse_stats(d_feat.cpu().numpy()[..., :3], tgt)[0]
            print(which, "noisy", noisy, "bilateral", rb, rb_finite, "unet", ru)
            assert nu == 0
            assert ru < rb and ru < rb_finite and ru < 0.2 * noisy
    finally:
        pr.close()


def test_trained_network_beats_bilateral_on_held_out_scenes():
    """Scenes the network never saw in training: the 4096 instanced bricks (its own
    geometry, materials and small emissive studs) and a procedural city generated from
    another seed (other heights, materials and light positions). The shipped weights
    against the bilateral filter on 1-spp frames, relMSE of linear radiance against a
    1024-spp render."""
    import torch

    from bench import relmse_stats
    from gknextengine_amd import denoise_train as dt
    pr = dt.PairRenderer()
    try:
        for name, scene in (("bricks", scenes.Bricks().scene), ("city_seed99", gk.procgen_city(64, 4, 256, 64, 99))):
            c = gk.Context(dt.TILE, dt.TILE)
            c.upload(scene)
            pr.ctx[name] = c
        net = gk.UNet.pretrained(pr.ctx["city"])
        rng = np.random.default_rng(4242)
        d_feat = torch.empty((dt.TILE, dt.TILE, gk.UNet.IN_CHANNELS), device="cuda")
        out = torch.empty(dt.TILE * dt.TILE * 3, device="cuda")
        cam = scenes.BRICKS_CAM
        results = []
        for which in ("bricks", "bricks", "city_seed99", "city_seed99"):
            for _ in range(8):  # a random view may see no light at all: draw another
                if which == "bricks":
                    eye = np.asarray(cam["eye"]) + rng.normal(0, 3.0, 3)
                    view = (tuple(eye), tuple(np.asarray(cam["target"]) + rng.normal(0, 2.0, 3)), cam["fov"])
                else:
                    view = dt.city_view(rng)
                tgt, bil = pr.pair(which, view, int(rng.integers(1 << 30)), int(rng.integers(1 << 20)), 1024,
                                   d_feat.data_ptr())
                if tgt.mean() > 1e-3:
                    break
            net.infer(d_feat.data_ptr(), out.data_ptr(), dt.TILE, dt.TILE)
            net.ctx.sync()
            u = out.cpu().numpy().reshape(dt.TILE, dt.TILE, 3)
            rb, rb_finite, _ = relmse_stats(bil, tgt)
            ru, _, nu = relmse_stats(u, tgt)
            noisy = relmse_stats(d_feat.cpu().numpy()[..., :3], tgt)[0]
            print(which, "noisy", noisy, "bilateral", rb, rb_finite, "unet", ru, "target mean", float(tgt.mean()))
            results.append((which, noisy, rb, rb_finite, ru, nu, float(tgt.mean())))
        for which, noisy, rb, rb_finite, ru, nu, mean in results:
            assert mean > 1e-3, which   # the view holds light
            assert nu == 0
            assert ru < rb and ru < rb_finite and ru < 0.5 * noisy, (which, noisy, rb, ru)
    finally:
        pr.close()


def test_fixed_shape_forward_equals_runtime_shape_kernels():
    """The forward pass of the 32-channel network through the kernels built for its layer
    shapes (unrolled K loop, fused 2x2 pooling) equals the runtime-shape convolutions and
    separate pooling bit for bit, on an image whose coarsest level is not a multiple of 16."""
    import os

    import torch
    rng = np.random.default_rng(7)
    h, w = 208, 176
    x = features(rng, 1, h, w)
    outs = []
    for generic in ("0", "1"):
        os.environ["GKNX_UNET_GENERIC"] = generic
        try:
            with gk.Context(16, 16) as ctx:
                net = gk.UNet(ctx, 32, seed=3)
                d_in = torch.from_numpy(x).cuda()
                d_out = torch.empty(h * w * 3, device="cuda")
                net.infer(d_in.data_ptr(), d_out.data_ptr(), h, w)
                ctx.sync()
                outs.append(d_out.cpu().numpy().copy())
        finally:
            os.environ.pop("GKNX_UNET_GENERIC", None)
    assert np.isfinite(outs[0]).all() and np.abs(outs[0]).max() > 0
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
