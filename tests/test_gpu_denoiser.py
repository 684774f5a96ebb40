"""The denoiser's HIP kernels (BF16 MFMA convolutions, FP32 accumulation)
against plain PyTorch CPU references of the same operations."""
import numpy as np
import pytest
import torch

from aurora_amd import denoiser as dn

pytestmark = pytest.mark.gpu


def bf16_bits(x):
    return (torch.from_numpy(np.ascontiguousarray(x, np.float32)).to(torch.bfloat16).view(torch.int16).numpy()
            .view(np.uint16))


def test_mfma_lane_layout(ctx):
    print("mfma selftest", flush=True)
    rng = np.random.default_rng(0)
    A = rng.integers(-8, 9, (16, 32)).astype(np.float32)
    B = rng.integers(-8, 9, (32, 16)).astype(np.float32)
    D = dn.mfma_selftest(ctx, bf16_bits(A), bf16_bits(B))
    assert np.array_equal(D, A @ B)


def inputs(B, H, W, seed=0, spp=4):
    g = torch.Generator().manual_seed(seed)
    rgb = torch.rand((B, H, W, 3), generator=g) * 3 * spp
    alb = torch.rand((B, H, W, 3), generator=g) * spp
    nrm = (torch.rand((B, H, W, 3), generator=g) * 2 - 1) * spp
    tgt = torch.rand((B, H, W, 3), generator=g) * 2
    return rgb, alb, nrm, tgt


def random_params(n, seed):
    # larger than the zero-initialised output layer so every layer matters
    rng = np.random.default_rng(seed)
    return (rng.normal(size=n) * 0.05).astype(np.float32)


# Launch shapes (unet_conv.hip's dispatch picks them from the pixel-block count
# of each layer).  32x48: every layer has fewer than 128 blocks, so every conv
# takes the channel-split form (one 16-channel tile per wave, NT = 1).
# 1024x1024, the inference workload: levels 0 and 1 take two rows per wave where
# their tiles fit 80 KB (32 and 48 output channels, NT = 2 and 3, pooling in the
# epilogue; 2048 and 512 blocks), level 2 one row per wave (64 channels, NT = 4,
# 256 blocks), rows of 16 to 4 segments of 64 pixels with their halos, encoder and
# concatenating decoder forms; level 3 (128^2, 64 blocks) the channel split.
@pytest.mark.parametrize("H,W", [(32, 48), (1024, 1024)])
def test_forward_matches_torch(ctx, H, W):
    print("denoiser forward", H, W, flush=True)
    net = dn.Denoiser(ctx, seed=1)
    p = random_params(net.n, 1)
    net.set_params(p)
    spp = 4
    rgb, alb, nrm, _ = inputs(1, H, W, spp=spp)
    out = net.denoise(rgb[0].cuda(), alb[0].cuda(), nrm[0].cuda(), spp).cpu().numpy()
    out16, noisy_log = dn.torch_reference(torch.from_numpy(p), rgb, alb, nrm, spp)
    ref = torch.clamp(torch.expm1(noisy_log + out16[:, :3]), min=0).permute(0, 2, 3, 1)[0].numpy()
    err = np.abs(out - ref)
    print("max abs err", err.max(), "mean", err.mean(), flush=True)
    assert np.allclose(out, ref, rtol=2e-2, atol=2e-2)
    assert err.mean() < 2e-3


# 8 x 128^2 is the training step's batch: the forward and the data-gradient
# convolutions take one row per wave, NT = 2 (level 0, 512 blocks) and NT = 3
# (level 1, 128 blocks), and two row segments per 128-pixel row; levels 2-3 the
# channel split; the weight gradient sums up to 128 partial blocks per input part.
@pytest.mark.parametrize("B,H,W", [(2, 16, 32), (8, 128, 128)])
@pytest.mark.parametrize("kind", ["log", "rel"])
def test_gradients_match_torch_autograd(ctx, kind, B, H, W):
    print("denoiser gradients", kind, B, H, W, flush=True)
    net = dn.Denoiser(ctx, seed=2)
    net.set_loss(kind)
    p = random_params(net.n, 2)
    net.set_params(p)
    spp = 4
    rgb, alb, nrm, tgt = inputs(B, H, W, seed=3, spp=spp)
    loss, g = net.loss_grad(rgb.cuda(), alb.cuda(), nrm.cuda(), tgt.cuda(), spp)
    pt = torch.from_numpy(p).to(torch.float64).requires_grad_(True)
    out16, noisy_log = dn.torch_reference(pt, rgb, alb, nrm, spp, emulate_bf16=False)
    pred = noisy_log + out16[:, :3]
    t64 = tgt.to(torch.float64).permute(0, 3, 1, 2)
    if kind == "log":
        ref_loss = ((pred - torch.log1p(t64)) ** 2).mean()
    else:
        # relative L2 with the denominator held constant (detached)
        D = torch.expm1(pred)
        ref_loss = ((D - t64) ** 2 / (D.detach() ** 2 + 0.01)).mean()
    ref_loss.backward()
    gr = pt.grad.numpy()
    cos = float(g @ gr / (np.linalg.norm(g) * np.linalg.norm(gr)))
    rel = float(np.linalg.norm(g - gr) / np.linalg.norm(gr))
    print("loss", loss, float(ref_loss.detach()), "cos", cos, "rel", rel, flush=True)
    assert abs(loss - float(ref_loss)) < 2e-2 * abs(float(ref_loss))
    assert cos > 0.995 and rel < 0.1
    # per layer: every layer's gradient agrees (catches a wrong layer mapping)
    off = 0
    for cout, cin in dn.layer_shapes():
        nw = cout * 9 * cin
        a, b = g[off:off + nw], gr[off:off + nw]
        if np.linalg.norm(b) > 1e-8:
            assert a @ b / (np.linalg.norm(a) * np.linalg.norm(b)) > 0.98, (cout, cin)
        off += nw + cout


def test_gradient_finite_difference(ctx):
    print("denoiser finite differences", flush=True)
    net = dn.Denoiser(ctx, seed=4)
    p = random_params(net.n, 4)
    net.set_params(p)
    B, H, W, spp = 1, 16, 16, 4
    rgb, alb, nrm, tgt = [t.cuda() for t in inputs(B, H, W, seed=5, spp=spp)]
    loss0, g = net.loss_grad(rgb, alb, nrm, tgt, spp)
    # along the gradient, with a step that moves the loss by ~4%: the BF16
    # forward's rounding noise is far below that change
    v = g / np.linalg.norm(g)
    eps = 0.02 * loss0 / np.linalg.norm(g)
    net.set_params(p + eps * v)
    lp, _ = net.loss_grad(rgb, alb, nrm, tgt, spp, grads=False)
    net.set_params(p - eps * v)
    lm, _ = net.loss_grad(rgb, alb, nrm, tgt, spp, grads=False)
    fd = (lp - lm) / (2 * eps)
    an = float(g @ v)
    print("fd", fd, "analytic", an, flush=True)
    assert abs(fd - an) < 0.1 * abs(an)


def test_training_reduces_loss(ctx):
    print("denoiser training smoke", flush=True)
    net = dn.Denoiser(ctx, seed=7)
    B, H, W, spp = 2, 32, 32, 4
    rgb, alb, nrm, tgt = [t.cuda() for t in inputs(B, H, W, seed=8, spp=spp)]
    first = net.train_step(rgb, alb, nrm, tgt, spp, 1e-3)
    for _ in range(30):
        last = net.train_step(rgb, alb, nrm, tgt, spp, 1e-3)
    print("loss", first, "->", last, flush=True)
    # random targets leave an irreducible loss; the fit must still improve
    assert last < 0.9 * first


def test_trained_network_gains_over_plain_render(ctx):
    """What the shipped network gains over the method without it: on
    held-out Cornell variants (seeds the training never saw) at 256^2, the
    denoised image of an N-spp render is closer to a 2048-spp target than
    the plain N-spp mean, by a wide margin (relMSE at least 10x lower at
    4 and 16 spp, and lower at 256 spp)."""
    import os

    from aurora_amd import train
    weights = os.path.join(os.path.dirname(dn.__file__), os.pardir, "weights", "unet_cornell.f32")
    net = dn.Denoiser(ctx)
    net.load(weights)
    print("held-out gain", flush=True)
    data = train.make_dataset(ctx, [100000 + k for k in range(4)], 256, [4, 16, 256], 2048, progress=False)
    res = train.evaluate(net, data)
    print(res, flush=True)
    for k in (4, 16):
        assert res[k]["denoised_relmse"] * 10 < res[k]["plain_relmse"], (k, res[k])
    assert res[256]["denoised_relmse"] < res[256]["plain_relmse"], res[256]
