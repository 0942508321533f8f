"""The NUFFT runs' part of the reverse sweep (hb_adjoint_runs) where the coils' residuals differ by many powers of two,
GPU: each coil's gradients stand on that coil's own residual.

Tolerance: float16 pairs and float32 sums of at most 32 columns a run against the sweep's own float32 products and sums
(hb_adjoint_interval): some 30 roundings of 2^-23 of the coil's largest, 4e-6."""

import numpy as np
import pytest
import torch

import blochparty_amd as bp
from blochparty_amd.engines import adjoint, driver
from test_gpu_spread import scan

f64 = torch.float64


@pytest.mark.gpu
@pytest.mark.parametrize("coils", [2, 8, 16])
def test_weak_residuals(gpu, monkeypatch, coils):
    n_spins, g = 500, torch.Generator().manual_seed(coils)
    u = lambda lo, hi: lo + (hi - lo) * torch.rand(n_spins, generator=g, dtype=f64)
    ph = bp.Phantom(torch.stack([0.006 + u(0, 0.024), u(-2e-4, 2e-4), u(-2e-4, 2e-4)], 1), u(0.5, 2.0), u(0.3, 2.0),
                    u(0.02, 0.3), u(-60.0, 60.0))
    c = torch.complex(*torch.randn(2, n_spins, coils, generator=g, dtype=f64))
    seq = scan(24, 2, 1, 7, True)
    case = driver.prepare_case(ph, seq, c, chunk=128, reuse=True, nufft=(6, 3), aligned=True)
    assert case.nu is not None and case.nu["cols"] <= 32
    ckpts = driver.run_forward(case, keep=True)
    nc = adjoint.adjoint_width(coils)
    sens = adjoint.adjoint_sens(c[torch.from_numpy(np.ascontiguousarray(case.perm))], case.n_pad, nc).cuda()
    size = 2.0 ** -torch.linspace(0, 40, coils)
    h = (torch.randn(case.n_adc, nc, 2, generator=g) * size[None, :, None]).cuda()
    out = []
    for inline in (False, True):
        monkeypatch.setattr(adjoint, "runs_beside", lambda nc, cols, changes, beside=not inline: beside)
        lam = torch.zeros(3, case.n_pad, device="cuda")
        gs, gc, _, lam = adjoint.run_backward(case, ckpts, 128, h, lam, sens, nc, 0, True)
        out.append((gs.cpu(), gc.cpu().reshape(nc, -1), lam.cpu().double()))
    for name, a, b in zip(("spins", "coils", "lambda"), *out):
        e = (a - b).abs().amax(1) / b.abs().amax(1).clamp_min(1e-300)
        print(name, " ".join(f"{v:.1e}" for v in e.tolist()), flush=True)
    (_, a, _), (_, b, _) = out
    assert bool(((a - b).abs().amax(1) <= 4e-6 * b.abs().amax(1)).all()) and float(b.abs().amax(1).min()) > 0
