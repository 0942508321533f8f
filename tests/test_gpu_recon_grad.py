"""Gradients through the reconstruction of k-space on the GPU, against the same on the CPU.

Tolerance: float32 transforms of 1,024 values and back: 1e-5 of the largest gradient."""

import pytest
import torch

from blochparty_amd import recon


@pytest.mark.gpu
def test_gradient_through_the_reconstruction(gpu):
    g = torch.Generator().manual_seed(0)
    k = torch.randn(3, 32, 32, dtype=torch.complex64, generator=g)
    w = torch.rand(32, 32, generator=g)
    grads = []
    for dev in ("cpu", "cuda"):
        x = k.to(dev).requires_grad_()
        image = recon.rss(recon.ifftnc(x, 2))
        assert image.requires_grad
        grads.append(torch.autograd.grad((w.to(dev) * image).sum(), x)[0].cpu())
        with torch.no_grad():
            assert torch.allclose(recon.rss(recon.ifftnc(x, 2)), image.detach(), rtol=1e-5, atol=1e-6)
    assert float((grads[1] - grads[0]).abs().max()) <= 1e-5 * float(grads[0].abs().max())
