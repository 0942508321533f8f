"""NUFFT runs spread as one matrix product with the largest operands the scales allow, GPU: full transverse
magnetization (90 degree pulses; m_init along x without RF, a run as the first record) under coils whose parts sit at a
power of two or just below one (modulus up to sqrt(2) after scaling), and magnetization above PD (T2 far above 2 T1).

Tolerance: against the oracle the NUFFT's own bound, 1e-4 of the largest sample at (6, 3); against the staged spreading
2e-6 (a few 2^-24 of each term, as the spreading's other tests)."""

import math

import numpy as np
import pytest
import torch

import blochparty_amd as bp
from blochparty_amd.engines import driver
from cases import rel
from oracle import core
from test_gpu_spread import scan

f64 = torch.float64


def spins(n, t1=(0.5, 2.0), t2=(0.3, 0.5)):
    g = torch.Generator().manual_seed(n)
    u = lambda lo, hi: lo + (hi - lo) * torch.rand(n, generator=g, dtype=f64)
    return bp.Phantom(torch.stack([0.006 + u(0, 0.012) * -(-n // 256), u(-2e-4, 2e-4), u(-2e-4, 2e-4)], 1),
                      torch.ones(n, dtype=f64), u(*t1), u(*t2), u(-5.0, 5.0))


def both_routes(ph, seq, coils, m_init=None):
    case = driver.prepare_case(ph, seq, coils, m_init, reuse=True, nufft=(6, 3))
    assert case.nu is not None and all(case.rf_free) and 20 < case.nu["cols"] <= 32
    case.nu["kind_changes"] = 0  # the matrix product, also for kinds in turn
    driver.run_forward(case)
    spread = driver.read_result(case)
    case.rf_free = [False] * len(case.rf_free)  # always correct: the general variant
    driver.run_forward(case)
    return spread, driver.read_result(case)


def check(ph, seq, coils, m_init=None):
    spread, staged = both_routes(ph, seq, coils, m_init)
    c = torch.ones(len(ph), 1, dtype=torch.complex128) if coils is None else coils
    ref, _ = core.simulate(ph, seq, c, m_init=m_init)
    e = rel(spread.signal.to(torch.complex128), ref), rel(spread.signal, staged.signal)
    print(f"oracle {e[0]:.1e}, staged {e[1]:.1e}", flush=True)
    assert bool(torch.isfinite(torch.view_as_real(spread.signal)).all())
    assert e[0] < 1e-4 and e[1] < 2e-6


@pytest.mark.gpu
@pytest.mark.parametrize("coil", [None, 1.0, 1 + 1j, 0.9 + 0.9j, -0.999 - 0.999j, 1.01 + 0.5j])
@pytest.mark.parametrize("coils", [1, 9])
def test_quarter_turn(gpu, coil, coils):
    """90 degree pulses (two substeps of 10 us)."""
    if coil is None and coils > 1:
        pytest.skip("no coils is one coil")
    n = 500
    seq = scan(24, 2, 1, 5, spoil=True)
    amp = 1 / (4 * 10e-6 * 3)  # 2 pi (a + 2 a) 10 us = pi / 2
    seq = bp.Sequence(seq.dt, seq.rf * (amp / 2000.0), seq.grad, seq.adc_phase, seq.is_rf, seq.adc, seq.spoil)
    check(spins(n), seq, None if coil is None else torch.full((n, coils), complex(coil), dtype=torch.complex128))


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [1.0, 0.5, 1e4])
def test_run_first(gpu, scale):
    """No RF: the run is the first record and the spins start transverse, |M| = |m_init| the case's bound."""
    n, N = 300, 32
    t = lambda v: torch.tensor(np.array(v), dtype=f64)
    seq = bp.Sequence(t([10e-6] * N + [1e-3]), t([(0.0, 0.0)] * (N + 1)), t([(40.0 / N / 10e-6, 0, 0)] * N + [(0, 0, 0)]),
                      t([0.0] * (N + 1)), [False] * (N + 1), [True] * N + [False], [False] * (N + 1))
    m0 = torch.zeros(n, 3, dtype=f64)
    m0[:, 0] = scale
    check(spins(n), seq, torch.full((n, 1), 1 + 1j, dtype=torch.complex128), m0)


def balanced(reps, n=16, t=1.9e-3):
    """Turns by pi - 0.25 about +x and -x, a run between, every gradient refocused: magnetization near +-y is turned onto
    its mirror image and gains along z in between, so with T2 >> T1 it grows far above PD."""
    dt, rf, g, is_rf, adc = [], [], [], [], []
    amp, gx = (math.pi - 0.25) / (2 * math.pi * 3 * 10e-6), 40.0 / n / 10e-6
    for i in range(reps):
        parts = [(10e-6, (1 + k) * (-amp if i % 2 else amp), 0.0, False) for k in range(2)]
        back = [(t, 0.0, -gx * n * 10e-6 / 2 / t, False)]
        parts += back + [(10e-6, 0.0, gx, True)] * n + back
        for d, w, x, a in parts:
            dt.append(d), rf.append((w, 0.0)), g.append((x, 0.0, 0.0)), is_rf.append(w != 0.0), adc.append(a)
    v = lambda x: torch.tensor(np.array(x, dtype=np.float64))
    return bp.Sequence(v(dt), v(rf), v(g), v([0.0] * len(dt)), is_rf, adc, [False] * len(dt))


@pytest.mark.gpu
def test_magnetization_above_pd(gpu):
    """T2 = 10^6 T1: balanced pulses take the magnetization above four times PD."""
    n = 256
    ph = spins(n, t1=(0.05, 0.06), t2=(5e4, 6e4))
    ph = bp.Phantom(ph.pos, ph.pd, ph.t1, ph.t2, torch.zeros(n, dtype=f64))
    m0 = torch.tensor([[0.0, -math.cos(0.125), math.sin(0.125)]], dtype=f64).expand(n, 3)
    seq, coils = balanced(500), torch.full((n, 1), 1 + 1j, dtype=torch.complex128)
    _, m = core.simulate(ph, seq, coils, m_init=m0)
    assert float(m.norm(dim=1).max()) > 4.0
    check(ph, seq, coils, m0)


def test_bound_of_the_magnetization():
    """driver.magnetization_bound: PD for T2 <= 2 T1; above it, no sequence of rotations and relaxation passes it
    (random ones, and the climb along Mz = PD R1 / (2 (R1 - R2)), in float64)."""
    rng = np.random.default_rng(0)
    one = lambda v: torch.tensor([v], dtype=f64)
    for r in (0.05, 1.0, 2.0):
        assert driver.magnetization_bound(one(0.8), one(1.0), one(r), one(0.5), 100.0) == 0.8
        assert driver.magnetization_bound(one(0.8), one(1.0), one(r), one(3.0), 100.0) == 3.0
    assert driver.magnetization_bound(one(0.8), one(1.0), one(math.inf), one(0.8), 0.0) == pytest.approx(0.8)
    assert driver.magnetization_bound(one(-0.8), one(math.inf), one(math.inf), one(0.0), 5.0) == 0.8
    assert driver.magnetization_bound(*(torch.zeros(0, dtype=f64),) * 4, 5.0) == 0.0
    for t2, total in ((3.0, 50.0), (40.0, 200.0), (1e4, 60.0), (math.inf, 30.0)):
        bound = driver.magnetization_bound(one(1.0), one(1.0), one(t2), one(1.0), total)
        steps = 20000
        h, rho, best = total / steps, 1.0, 1.0
        r2 = 1 / t2
        for k in range(steps):  # turned to the best Mz before each step (or a random one)
            z = min(rho, 1 / (2 * (1 - r2))) if rng.random() < 0.98 else rho * rng.uniform(-1, 1)
            xy = math.sqrt(max(rho * rho - z * z, 0.0)) * math.exp(-h * r2)
            z = 1 + (z - 1) * math.exp(-h)
            rho = math.hypot(xy, z)
            best = max(best, rho)
        assert best <= bound * (1 + 1e-9) and best > 0.7 * bound, (t2, best, bound)
