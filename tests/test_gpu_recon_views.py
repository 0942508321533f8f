"""Reconstruction of conjugated views of k-space on the GPU (a view that torch marks and does not write out: its memory
holds the values themselves), one pass per axis and planes, against torch's FFT of the values.

Tolerance: float32 transforms of at most 4,096 values: 1e-6 of the largest value (as the reconstruction's other tests)."""

import pytest
import torch

from blochparty_amd import recon

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(3, 64, 64), (2, 8, 32), (2, 4, 32, 32)])
def test_conjugated_views(gpu, shape):
    k = torch.randn(*shape, dtype=torch.complex64, generator=torch.Generator().manual_seed(len(shape)))
    view = k.cuda().conj()
    assert view.is_conj()
    axes = tuple(range(-(len(shape) - 1), 0))
    ref = torch.fft.fftshift(torch.fft.ifftn(torch.fft.ifftshift(k.conj().to(torch.complex128), dim=axes), dim=axes),
                             dim=axes)
    img = recon.ifftnc(view, len(shape) - 1)
    assert float((img.cpu() - ref).abs().max() / ref.abs().max()) < 1e-6
    out = recon.rss(img.conj())
    assert float((out.cpu() - (ref.abs() ** 2).sum(0).sqrt()).abs().max() / ref.abs().max()) < 1e-6
