"""hb_adjoint_chunks (an interval reversed in chunks of segments side by side) against hb_adjoint_interval (one walk) on
the same buffers, GPU: workgroup counts of every chunk length, intervals that end inside a chunk or are shorter than one,
coil counts and modes of the kernel's variants, spoils and samples at chunk ends.

Tolerance: both sum the same float32 terms, in other groups, with lambda carried by other instruction sequences: some
thousand roundings of 2^-24, 1e-5 of the largest of a row; the project's bound on gradients, 1e-4, is asserted."""

import ctypes

import numpy as np
import pytest
import torch

import blochparty_amd as bp
from blochparty_amd.engines import adjoint, driver, hip

f64 = torch.float64


def table(seed, segments):
    rng = np.random.default_rng(seed)
    kind = np.repeat(rng.integers(0, 3, segments), rng.integers(1, 14, segments))[:segments]  # RF, free, samples
    is_rf, adc = kind == 0, kind == 2
    t = lambda v: torch.tensor(v, dtype=f64)
    rf = rng.normal(0, 400, (segments, 2)) * is_rf[:, None]
    grad = rng.normal(0, 2e3, (segments, 3))
    for k in range(1, segments):  # equal neighbours, for the kept factors
        if kind[k] == kind[k - 1] and rng.random() < 0.7:
            grad[k] = grad[k - 1]
    dt = np.where(is_rf, 10e-6, np.where(adc, 20e-6, 1e-3))
    spoil = (rng.random(segments) < 0.05) & ~is_rf
    return bp.Sequence(t(dt), t(rf), t(grad), t(rng.uniform(0, 6, segments)), is_rf.tolist(), adc.tolist(), spoil.tolist())


@pytest.mark.gpu
@pytest.mark.parametrize("n_spins,coils,every,segments,mode", [
    (1, 1, 64, 64, 1), (300, 8, 64, 150, 2), (9000, 3, 128, 300, 1), (17000, 16, 192, 333, 2), (40000, 0, 64, 131, 1),
    (70000, 5, 128, 135, 0)])
def test_chunks_against_one_walk(gpu, n_spins, coils, every, segments, mode):
    g = torch.Generator().manual_seed(n_spins)
    u = lambda lo, hi: lo + (hi - lo) * torch.rand(n_spins, generator=g, dtype=f64)
    ph = bp.Phantom(torch.stack([u(-0.1, 0.1), u(-0.1, 0.1), u(-0.1, 0.1)], 1), u(0.5, 1.5), u(0.3, 2.0), u(0.02, 0.3),
                    u(-60.0, 60.0), b1=u(0.8, 1.2))
    seq = table(n_spins, segments)
    c = torch.complex(*torch.randn(2, n_spins, max(coils, 1), generator=g, dtype=f64))
    case = driver.prepare_case(ph, seq, c, chunk=every, aligned=True)
    ckpts = driver.run_forward(case, keep=True)
    nc = adjoint.adjoint_width(coils) if coils else 0
    sens = adjoint.adjoint_sens(c, case.n_pad, nc).cuda()
    h = torch.randn(max(case.n_adc, 1), max(nc, 1), 2, generator=g).cuda()
    lam0 = torch.randn(3, case.n_pad, generator=g).cuda()
    cs, lib, n_blocks = case.struct(), hip.HIP.lib(), case.n_pad // 256
    need = hip.load().hb_adjoint_chunks_workspace(case.n_pad, every, nc)
    assert need > 0
    outs = []
    for work in (None, torch.full((need,), float("nan"), device="cuda")):
        gs = torch.zeros(8, case.n_pad, dtype=f64, device="cuda")
        gc = torch.zeros(2 * max(nc, 1), case.n_pad, dtype=f64, device="cuda")
        lam = lam0.clone()
        gseg = torch.zeros(len(ckpts), n_blocks, every, 8, device="cuda")
        r8 = torch.empty((every + 7) // 8 * 3 * case.n_pad, device="cuda")
        for i in reversed(range(len(ckpts))):
            ad = hip.HbAdjoint(ckpts[i].data_ptr(), r8.data_ptr(), lam.data_ptr(), gs.data_ptr(), gc.data_ptr(),
                               gseg[i].data_ptr(), h.data_ptr(), sens.data_ptr(), None, None, None, None, None, nc, mode,
                               int(mode != 0), every)
            lib.adjoint_chunks(ctypes.byref(cs), ctypes.byref(ad), case.starts[i], case.ends[i],
                               None if work is None else work.data_ptr())
        torch.cuda.synchronize()
        outs.append([gs[:, :n_spins], gc[:, :n_spins], lam[:, :n_spins].double(), gseg.sum(1).reshape(-1, 8).T.double()])
    for a, b in zip(*outs):
        scale = a.abs().amax(-1, keepdim=True)
        assert bool(((a - b).abs() <= 1e-4 * scale).all())
    assert bool(torch.isfinite(outs[1][0]).all()) and float(outs[1][0].abs().max()) > 0


def test_workspace_rule():
    """0 doubles where the intervals are not taken in chunks (many spins), enough for every chunk elsewhere."""
    ws = hip.load().hb_adjoint_chunks_workspace
    assert ws(256 * 1025, 128, 8) == 0 and ws(255, 128, 8) == 0 and ws(256, 0, 8) == 0 and ws(256, 64, 17) == 0
    for blocks, chunk in ((1, 8), (32, 8), (63, 8), (64, 16), (127, 16), (128, 32), (255, 32), (256, 64), (1024, 64)):
        for k in (1, 64, 100, 384):
            assert ws(256 * blocks, k, 4) == -(-k // chunk) * (3 + 8 + 8) * 256 * blocks
