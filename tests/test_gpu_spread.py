"""NUFFT runs spread as one matrix product per run (windows of at most 32 columns, up to 16 coils, no stepped RF in the
dispatch) against the staged spreading of the same dispatches, GPU: alternating run kinds (the weights are formed anew
at each), windows on both sides of 16 columns, samples staged before and after runs, coil counts at the tiles' edges,
partly filled workgroups, dispatch cuts, spoiled and unspoiled run ends, a single map and several.

Tolerance: both take the same float32 weights and magnetization, in float16 pairs (2^-24 relative) with float32 sums of
64 spins; what differs is the rounding of a product (S c) w against S (c w): a few 2^-24 of each term, 2e-6 of the
largest sample at most."""

import numpy as np
import pytest
import torch

import blochparty_amd as bp
from blochparty_amd.engines import driver
from cases import rel
from oracle import core

pytestmark = pytest.mark.gpu
f64 = torch.float64


def scan(n, kinds, pulses, reps, spoil=True):
    """reps repetitions: one of ``pulses`` two-step pulses with its own flip, a prephaser ending on a sample, a run of n
    samples with one of ``kinds`` gradients, two lone samples, a fill."""
    dt, rf, g, is_rf, adc, sp, psi = [], [], [], [], [], [], []
    for i in range(reps):
        ph, amp = 0.7 * i * i, 2000.0 * (1 + i % pulses)
        for k in range(2):
            dt.append(10e-6), rf.append((amp * (1 + k) * np.cos(ph), amp * (1 + k) * np.sin(ph)))
            g.append((0.0, 0.0, 0.0)), is_rf.append(True), adc.append(False), sp.append(False), psi.append(0.0)
        read = [(40.0 / n / 10e-6, 0.0, 0.0), (-40.0 / n / 10e-6, 2000.0, 0.0), (30.0 / n / 10e-6, 0.0, 500.0)][i % kinds]
        parts = [(5e-4, (-2e4, 300.0 * i, 0.0), False, False), (5e-6, read, True, False)]
        parts += [(10e-6, read, True, spoil and i % 3 == 2 and k == n - 1) for k in range(n)]
        parts += [(7e-6, (0.0, 100.0, 0.0), True, False), (9e-6, (50.0, 0.0, 0.0), True, False),
                  (3e-3, (0.0, 0.0, 100.0), False, spoil and i % 2 == 0)]
        for t, grad, a, s in parts:
            dt.append(t), rf.append((0.0, 0.0)), g.append(grad), is_rf.append(False), adc.append(a), sp.append(s)
            psi.append(0.1 * i)
    t = lambda v: torch.tensor(np.array(v), dtype=f64)
    return bp.Sequence(t(dt), t(rf), t(g), t(psi), is_rf, adc, sp)


@pytest.mark.parametrize("n_spins,coils,n,kinds,pulses,nufft,chunk", [
    (1, 1, 16, 1, 1, (6, 3), 32768), (255, 8, 17, 2, 1, (6, 3), 32768), (700, 9, 64, 3, 2, (6, 3), 32768),
    (3000, 16, 33, 2, 1, (6, 2), 90), (513, 5, 24, 1, 2, (5, 3), 70), (2000, 7, 40, 2, 1, (8, 3), 32768)])
@pytest.mark.parametrize("spoil", [True, False])
def test_spread_against_staged(gpu, n_spins, coils, n, kinds, pulses, nufft, chunk, spoil):
    g = torch.Generator().manual_seed(n_spins)
    u = lambda lo, hi: lo + (hi - lo) * torch.rand(n_spins, generator=g, dtype=f64)
    # about one grid cell per workgroup of sorted spins, away from phase 0 (a workgroup across it would span the grid)
    ph = bp.Phantom(torch.stack([0.006 + u(0, 0.012) * -(-n_spins // 256), u(-2e-4, 2e-4), u(-2e-4, 2e-4)], 1), u(0.5, 2.0), u(0.3, 2.0),
                    u(0.02, 0.3), u(-60.0, 60.0))
    c = torch.complex(*torch.randn(2, n_spins, coils, generator=g, dtype=f64))
    seq = scan(n, kinds, pulses, 7, spoil)
    case = driver.prepare_case(ph, seq, c, chunk=chunk, reuse=True, nufft=nufft)
    assert case.nu is not None and all(case.rf_free)
    assert case.nu["cols"] <= 32  # the matrix product's side of the rule
    driver.run_forward(case)
    spread = driver.read_result(case)
    case.rf_free = [False] * len(case.rf_free)  # always correct: the general variant
    driver.run_forward(case)
    staged = driver.read_result(case)
    assert rel(spread.m, staged.m) < 1e-5  # the same steps (two compiled variants), as against per-sample readouts
    assert rel(spread.signal, staged.signal) < 2e-6
    if nufft == (6, 3) and n_spins < 1000:
        ref, _ = core.simulate(ph, seq, c)
        assert rel(spread.signal.to(torch.complex128), ref) < 1e-4


def test_windows_too_wide_for_the_product(gpu):
    """More than 32 columns: the staged spreading, within the NUFFT's tolerance of the oracle."""
    n_spins, g = 300, torch.Generator().manual_seed(5)
    u = lambda lo, hi: lo + (hi - lo) * torch.rand(n_spins, generator=g, dtype=f64)
    ph = bp.Phantom(torch.stack([0.006 + u(0, 0.012) * -(-n_spins // 256), u(-2e-4, 2e-4), u(-2e-4, 2e-4)], 1), u(0.5, 2.0), u(0.3, 2.0),
                    u(0.05, 0.3), u(-60.0, 60.0))
    seq, c = scan(16, 1, 1, 4), torch.complex(*torch.randn(2, 300, 3, generator=g, dtype=f64))
    case = driver.prepare_case(ph, seq, c, reuse=True, nufft=(8, 4))
    assert case.nu is not None and case.nu["cols"] > 32
    driver.run_forward(case)
    ref, _ = core.simulate(ph, seq, c)
    assert rel(driver.read_result(case).signal.to(torch.complex128), ref) < 1e-4
