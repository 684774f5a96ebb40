"""The denoiser at image sizes where its tiles end: the smallest image, widths
past a 64-pixel segment by 8 pixels, a coarsest level of one pixel, batches,
a size whose full resolution takes two rows per wave with a ragged last segment,
and one whose every level does.  Same references and bounds as test_gpu_denoiser.py."""
import numpy as np
import pytest
import torch
from test_gpu_denoiser import inputs, random_params

from aurora_amd import denoiser as dn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W", [(8, 8), (40, 72), (128, 136), (512, 520)])
def test_forward_edges(ctx, H, W):
    net = dn.Denoiser(ctx, seed=1)
    p = random_params(net.n, 11)
    net.set_params(p)
    spp = 4
    rgb, alb, nrm, _ = inputs(1, H, W, seed=H + W, spp=spp)
    out = net.denoise(rgb[0].cuda(), alb[0].cuda(), nrm[0].cuda(), spp).cpu().numpy()
    out16, noisy_log = dn.torch_reference(torch.from_numpy(p), rgb, alb, nrm, spp)
    ref = torch.clamp(torch.expm1(noisy_log + out16[:, :3]), min=0).permute(0, 2, 3, 1)[0].numpy()
    err = np.abs(out - ref)
    assert np.allclose(out, ref, rtol=2e-2, atol=2e-2), err.max()
    assert err.mean() < 2e-3
    # in place: the image over its own input sums
    buf = rgb[0].cuda()
    net.denoise(buf, alb[0].cuda(), nrm[0].cuda(), spp, out=buf)
    assert np.array_equal(buf.cpu().numpy(), out)


@pytest.mark.parametrize("B,H,W", [(1, 8, 8), (3, 24, 72), (2, 40, 136)])
def test_gradient_edges(ctx, B, H, W):
    net = dn.Denoiser(ctx, seed=2)
    net.set_loss("log")
    p = random_params(net.n, 12)
    net.set_params(p)
    spp = 4
    rgb, alb, nrm, tgt = inputs(B, H, W, seed=B * H * W, spp=spp)
    args = [t.cuda() for t in (rgb, alb, nrm, tgt)]
    loss, g = net.loss_grad(*args, spp)
    pt = torch.from_numpy(p).to(torch.float64).requires_grad_(True)
    out16, noisy_log = dn.torch_reference(pt, rgb, alb, nrm, spp, emulate_bf16=False)
    pred = noisy_log + out16[:, :3]
    ((pred - torch.log1p(tgt.to(torch.float64).permute(0, 3, 1, 2))) ** 2).mean().backward()
    gr = pt.grad.numpy()
    assert g @ gr / (np.linalg.norm(g) * np.linalg.norm(gr)) > 0.995
    assert np.linalg.norm(g - gr) / np.linalg.norm(gr) < 0.1
    # fixed summation order: the same gradients again
    assert np.array_equal(net.loss_grad(*args, spp)[1], g)


def test_forward_pools_in_the_convolution_at_every_level(ctx):
    """The smallest square image whose level 2 (64 channels) pools in its
    convolution's epilogue (512 blocks of 8 rows x 64 pixels), and one 32 rows
    shorter, where a kernel of its own pools that level: crops of both match the
    reference, with the bounds of the other forward tests."""
    net = dn.Denoiser(ctx, seed=1)
    p = random_params(net.n, 13)
    net.set_params(p)
    spp, W = 4, 2048
    rgb, alb, nrm, _ = inputs(1, 2048, W, seed=21, spp=spp)
    for H in (2048, 2016):
        a = [t[0, :H].contiguous() for t in (rgb, alb, nrm)]
        out = net.denoise(*[t.cuda() for t in a], spp).cpu().numpy()
        # the receptive field of a pixel reaches less than 96 pixels: the reference on a crop
        # is the image's where the crop's edge is that far away or the image's own
        for y0, x0 in ((0, 0), (H - 384, W - 384), (H // 16 * 8, 1024)):
            y1, x1 = y0 + 384, x0 + 384
            crop = [t[None, y0:y1, x0:x1].contiguous() for t in a]
            out16, noisy_log = dn.torch_reference(torch.from_numpy(p), *crop, spp)
            ref = torch.clamp(torch.expm1(noisy_log + out16[:, :3]), min=0).permute(0, 2, 3, 1)[0].numpy()
            m = [0 if y0 == 0 else 96, 384 if y1 == H else 288, 0 if x0 == 0 else 96, 384 if x1 == W else 288]
            got, want = out[y0:y1, x0:x1][m[0]:m[1], m[2]:m[3]], ref[m[0]:m[1], m[2]:m[3]]
            err = np.abs(got - want)
            assert np.allclose(got, want, rtol=2e-2, atol=2e-2), (H, y0, err.max())
            assert err.mean() < 2e-3
