"""The NUFFT runs' part of the reverse sweep taken beside it (hb_adjoint_runs; windows of at most 32 columns) against the
sweep that takes it inline (hb_adjoint_interval, every window), GPU: alternating run kinds (the weights are formed anew at
each), windows on both sides of 16 columns, coil counts of every variant and tiles of 16 coils, partly filled
workgroups, intervals that cut between runs and hold none, spoiled and unspoiled run ends, one term (no decay nodes but 0).

Tolerance: the products take float16 pairs (2^-22 of the window's largest grid value) with float32 sums of at most 32
columns, the inline form float32 sums of the same terms: some 10 roundings of 2^-22, 3e-6 of a run's largest, and the
gradients sum runs; the project's bound on gradients, 1e-4 of a gradient's largest, is asserted."""

from dataclasses import replace

import pytest
import torch

import blochparty_amd as bp
from blochparty_amd.engines import driver, hip
from cases import rel, weighted_loss
from test_gpu_spread import scan

f64 = torch.float64


@pytest.mark.gpu
@pytest.mark.parametrize("n_spins,coils,n,kinds,pulses,nufft,every", [
    (1, 1, 16, 1, 1, (6, 3), 64), (255, 8, 17, 2, 1, (6, 3), 128), (700, 2, 64, 3, 2, (6, 3), 192),
    (3000, 16, 33, 2, 1, (6, 2), 64), (513, 3, 24, 1, 2, (5, 1), 512), (2000, 20, 40, 2, 1, (8, 3), 256)])
@pytest.mark.parametrize("spoil", [True, False])
def test_beside_against_inline(gpu, monkeypatch, n_spins, coils, n, kinds, pulses, nufft, every, spoil):
    g = torch.Generator().manual_seed(n_spins)
    u = lambda lo, hi: lo + (hi - lo) * torch.rand(n_spins, generator=g, dtype=f64)
    x = 0.006 + u(0, 0.012) * -(-n_spins // 256)  # narrow windows, as in test_gpu_spread.py
    ph = bp.Phantom(torch.stack([x, u(-2e-4, 2e-4), u(-2e-4, 2e-4)], 1), u(0.5, 2.0), u(0.3, 2.0), u(0.02, 0.3),
                    u(-60.0, 60.0))
    c = torch.complex(*torch.randn(2, n_spins, coils, generator=g, dtype=f64))
    seq = scan(n, kinds, pulses, 7, spoil)
    case = driver.prepare_case(ph, seq, c, chunk=every, reuse=True, nufft=nufft, aligned=True)
    assert case.nu is not None and case.nu["cols"] <= 32
    taken, out = [], []
    real = hip.load().hb_adjoint_runs_takes
    for takes in (real, lambda nc, cols: 0):
        monkeypatch.setattr(hip.load(), "hb_adjoint_runs_takes",
                            lambda nc, cols, f=takes: taken.append(f(nc, cols)) or taken[-1])
        leaves = {k: getattr(ph, k).clone().requires_grad_() for k in ("pos", "pd", "t1", "t2", "db0")}
        ck = c.clone().requires_grad_()
        r = bp.simulate(replace(ph, **leaves), seq, ck, engine="gpu", pulses="reuse", readouts="nufft",
                        nufft_width=nufft[0], nufft_terms=nufft[1], checkpoint_every=every)
        out.append(torch.autograd.grad(weighted_loss(r.signal, r.m), [*leaves.values(), ck]))
    assert taken[0] == 1 and taken[-1] == 0  # both routes ran
    for name, a, b in zip((*leaves, "coils"), *out):
        e = rel(a, b)
        print(name, f"{e:.1e}")
        assert bool(torch.isfinite(a.abs()).all()) and float(b.abs().max()) > 0
        assert e <= 1e-4, name


def test_rule():
    """The kernel's variants, and windows that one product takes."""
    takes = hip.load().hb_adjoint_runs_takes
    assert all(takes(nc, k) for nc in (1, 2, 4, 8, 16) for k in (1, 32))
    assert not any(takes(nc, 8) for nc in (0, 3, 17, 32)) and not any(takes(8, k) for k in (-1, 0, 33))
