"""hb_ifftc_plane (both of the last two axes in one pass) against one pass per axis and torch's FFT in float64, GPU: odd and
even log2 sides, every butterfly count, the smallest and largest sides and planes, in place and out of place, many planes
and none; and the rule that takes a transform there.

Tolerance: a float32 transform of N values rounds log2 N times a value (2^-24 each, in the root mean square): 1e-6 of the
largest value; the two routes do the same operations, so between them the same bound holds with room."""

import pytest
import torch

from blochparty_amd import recon
from blochparty_amd.engines import hip

CASES = [(16, 64, 5), (64, 16, 300), (32, 32, 1), (64, 64, 8), (128, 32, 3), (16, 512, 2), (64, 128, 2), (128, 128, 7),
         (1024, 16, 2), (16, 1024, 2)]


@pytest.mark.gpu
@pytest.mark.parametrize("A,B,planes", CASES)
@pytest.mark.parametrize("in_place", [False, True])
def test_plane(gpu, A, B, planes, in_place):
    x = torch.randn(planes, A, B, 2, generator=torch.Generator().manual_seed(A + B)).cuda()
    x = torch.view_as_complex(x)
    ref = recon.ifftnc(x.cpu().to(torch.complex128), 2)
    lib = gpu.lib()
    axis = torch.empty_like(x)
    lib.ifftc_axis(x.data_ptr(), axis.data_ptr(), planes, A, B)
    lib.ifftc_axis(axis.data_ptr(), axis.data_ptr(), planes * A, B, 1)
    out = x.clone() if in_place else torch.full_like(x, float("nan"))
    lib.ifftc_plane((out if in_place else x).data_ptr(), out.data_ptr(), planes, A, B)
    scale = float(ref.abs().max())
    assert float((out.cpu() - ref).abs().max()) <= 1e-6 * scale
    assert float((out - axis).abs().max()) <= 1e-6 * scale


@pytest.mark.gpu
def test_ifftnc_takes_the_plane_in_2d_and_3d(gpu):
    x = torch.view_as_complex(torch.randn(3, 8, 32, 64, 2, generator=torch.Generator().manual_seed(1)))
    for ndim in (1, 2, 3):
        for t in (x, x.transpose(-1, -2)):  # a strided view is laid out first
            ref = recon.ifftnc(t.to(torch.complex128), ndim)
            got = recon.ifftnc(t.cuda(), ndim).cpu()
            assert float((got - ref).abs().max()) <= 1e-6 * float(ref.abs().max())
    gpu.lib().ifftc_plane(x.cuda().data_ptr(), x.cuda().data_ptr(), 0, 32, 64)  # no planes: nothing launched
    with pytest.raises(RuntimeError):
        gpu.lib().ifftc_plane(x.cuda().data_ptr(), x.cuda().data_ptr(), 1, 8, 8)


def test_rule():
    takes = hip.load().hb_ifftc_plane_takes
    assert all(takes(a, b) and takes(b, a) for a, b, _ in CASES)
    assert not any(takes(a, b) for a, b in ((16, 32), (8, 1024), (128, 256), (2048, 16), (0, 64), (48, 64), (-16, -64)))
