"""Intervals of more segments than hb_adjoint_chunks reverses at a time (2,048): the workspace does not grow with them, and
the gradients are the same bit for bit as with short intervals, also beyond 65,535 chunks (a grid's y dimension)."""

import pytest
import torch

import blochparty_amd as bp
from blochparty_amd.engines import adjoint, driver, hip
from test_gpu_adjoint_chunks import table

f64 = torch.float64


def test_workspace_has_a_limit():
    ws = hip.load().hb_adjoint_chunks_workspace
    for blocks, nc in ((1, 0), (32, 8), (64, 16), (1024, 16)):
        assert 0 < ws(256 * blocks, 2048, nc) == ws(256 * blocks, 2112, nc) == ws(256 * blocks, 2**31 - 64, nc)
        assert ws(256 * blocks, 2048, nc) * 4 < 1.6e9


def test_where_one_walk_is_faster():
    """Up to two coils from 513 to 768 workgroups: not in chunks; on both sides and with more coils in chunks."""
    ws = hip.load().hb_adjoint_chunks_workspace
    for nc in (0, 1, 2):
        assert all(ws(256 * b, 384, nc) == 0 for b in (513, 600, 768))
        assert all(ws(256 * b, 384, nc) > 0 for b in (512, 769, 1024))
    assert all(ws(256 * b, 384, nc) > 0 for b in (513, 768) for nc in (4, 8, 16))


def gradients(ph, seq, c, every, need_seg):
    case = driver.prepare_case(ph, seq, c, chunk=every, aligned=True)
    ckpts = driver.run_forward(case, keep=True)
    nc = adjoint.adjoint_width(c.shape[1])
    g = torch.Generator().manual_seed(1)
    h = torch.randn(case.n_adc, nc, 2, generator=g).cuda()
    lam = torch.randn(3, case.n_pad, generator=g).cuda()
    out = adjoint.run_backward(case, ckpts, every, h, lam, adjoint.adjoint_sens(c, case.n_pad, nc).cuda(), nc, need_seg, True)
    return [t[..., : len(ph)].cpu() if i != 2 else t.cpu() for i, t in enumerate(out)]


def spins(n, coils):
    g = torch.Generator().manual_seed(n)
    u = lambda lo, hi: lo + (hi - lo) * torch.rand(n, generator=g, dtype=f64)
    ph = bp.Phantom(torch.stack([u(-0.1, 0.1), u(-0.1, 0.1), u(-0.1, 0.1)], 1), u(0.5, 1.5), u(0.3, 2.0), u(0.02, 0.3),
                    u(-60.0, 60.0), b1=u(0.8, 1.2))
    return ph, torch.complex(*torch.randn(2, n, coils, generator=g, dtype=f64))


@pytest.mark.gpu
@pytest.mark.parametrize("n_spins,coils,segments,need_seg", [(40, 1, 2048, 1), (300, 8, 2049, 2), (300, 3, 4500, 1),
                                                             (17000, 2, 4161, 0)])
def test_same_bits_in_batches(gpu, n_spins, coils, segments, need_seg):
    ph, c = spins(n_spins, coils)
    seq = table(n_spins, segments)
    long = gradients(ph, seq, c, -(-segments // 64) * 64, need_seg)
    for a, b in zip(long, gradients(ph, seq, c, 128, need_seg)):
        assert bool(torch.isfinite(a).all()) and torch.equal(a, b)


@pytest.mark.gpu
def test_more_chunks_than_a_grid_takes(gpu):
    """One interval of 8 x 65,536 + 64 segments on one workgroup (chunks of 8)."""
    segments = 8 * 65536 + 64
    ph, c = spins(16, 1)
    part = table(3, 4096)
    times = -(-segments // 4096)
    rep = lambda t: t.repeat(times, *(1,) * (t.ndim - 1))[:segments]
    flags = lambda f: (list(f) * times)[:segments]
    seq = bp.Sequence(rep(part.dt), rep(part.rf), rep(part.grad), rep(part.adc_phase), flags(part.is_rf), flags(part.adc),
                      flags(part.spoil))
    long = gradients(ph, seq, c, segments, 0)
    for a, b in zip(long, gradients(ph, seq, c, 16384, 0)):
        assert bool(torch.isfinite(a).all()) and torch.equal(a, b)
