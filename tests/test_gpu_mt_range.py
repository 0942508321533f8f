"""The full variant's signal where coils, spins or the scales of a case differ by many powers of two, against the FP64
oracle, GPU: a coil far below another, dim spins beside a bright one that no coil sees, and a caller of the C interface who
leaves the plain kernels' scales at 0.

Tolerance: float32 steps, some 1,000 per case, against float64 on the same inputs: 1e-5 of a coil's largest value, as the
other cases of this kernel."""

from dataclasses import replace

import pytest
import torch

from blochparty_amd.engines import driver
from cases import rel
from oracle import exchange as E
from test_gpu_mt_routes import SPANS, TRAINS, blocks, pooled

pytestmark = pytest.mark.gpu
f64 = torch.float64


def run(ph, seq, c, **scales):
    case = driver.prepare_case(ph, seq, c)
    assert case.extra.get("mt") is not None
    for k, v in scales.items():
        setattr(case, k, v)
    driver.run_forward(case)
    out = driver.read_result(case).signal.to(torch.complex128)
    ref, _ = E.simulate_bound(ph, seq, c)
    e = [rel(a, b) for a, b in zip(out, ref)]  # coil by coil
    print(" ".join(f"{v:.1e}" for v in e), flush=True)
    assert max(e) < 1e-5


def coils(n, count, seed=0):
    g = torch.Generator().manual_seed(seed)
    return torch.complex(*torch.randn(2, n, count, generator=g, dtype=f64))


@pytest.mark.parametrize("count", [2, 8, 16, 17])
def test_weak_coils(gpu, count):
    ph = pooled(300, 1)
    c = coils(300, count) * 2.0 ** -torch.linspace(0, 40, count, dtype=f64)
    run(ph, blocks(SPANS, TRAINS), c)


@pytest.mark.parametrize("count", [3, 9])
def test_dim_spins(gpu, count):
    ph = pooled(300, 2)
    ph = replace(ph, pd=ph.pd * torch.where(torch.arange(300) == 7, 2.0**24, 1.0))
    c = coils(300, count)
    c[7] = 0
    run(ph, blocks(SPANS, TRAINS), c)


@pytest.mark.parametrize("count", [3, 9])
def test_no_scales(gpu, count):
    ph = pooled(300, 3)
    run(replace(ph, pd=ph.pd * 1e5), blocks(SPANS, TRAINS), coils(300, count) * 1e3, sens_scale=0.0, x_scale=0.0)
