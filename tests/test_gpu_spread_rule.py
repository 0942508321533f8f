"""Which spreading NUFFT runs take (hb_forward_product): by the windows' columns, the coil tiles and how often the runs' kind
changes; and the matrix product on kinds in turn with one and two tiles, which the rule no longer sends there, against the
staged spreading (as test_gpu_spread.py, with its tolerance). The same for the runs' part of the reverse sweep
(adjoint.runs_beside; as test_gpu_nufft_back.py, with its tolerance)."""

from dataclasses import replace

import pytest
import torch

import blochparty_amd as bp
from blochparty_amd.engines import adjoint, driver, hip
from blochparty_amd.engines import nufft as nu_mod
from cases import rel, weighted_loss
from test_gpu_spread import scan

f64 = torch.float64


def test_rule():
    """Kinds in turn (1,024 changes in 1,024 runs) are staged, one kind takes the product where its windows are wide
    enough; never above 32 columns or two tiles."""
    takes = hip.load().hb_forward_product
    for tiles, base in ((1, 4), (2, 20)):
        for cols in range(1, 33):
            assert takes(cols, tiles, 0) == (cols >= base)
            line = 16 * (cols - base)
            if line > 0:
                assert takes(cols, tiles, line) and not takes(cols, tiles, line + 1)
        assert not takes(21, tiles, 1024) and not takes(33, tiles, 0)
    assert not takes(21, 3, 0)


@pytest.mark.parametrize("kinds,reps,changes", [(1, 7, 0), (2, 7, 6 / 7), (3, 9, 8 / 9), (2, 1, 0)])
def test_changes_of_kind(kinds, reps, changes):
    plan = nu_mod.make_plan(scan(24, kinds, 1, reps), 6, 3)
    assert plan.kind_changes == -(-1024 * round(changes * reps) // reps)


@pytest.mark.gpu
@pytest.mark.parametrize("n_spins,coils,kinds,nufft,chunk", [
    (255, 8, 2, (6, 3), 32768), (700, 9, 3, (6, 3), 32768), (3000, 16, 2, (5, 4), 90), (513, 3, 2, (5, 4), 70),
    (1, 16, 3, (7, 3), 32768)])
@pytest.mark.parametrize("spoil", [True, False])
def test_product_on_kinds_in_turn(gpu, n_spins, coils, kinds, nufft, chunk, spoil):
    g = torch.Generator().manual_seed(n_spins)
    u = lambda lo, hi: lo + (hi - lo) * torch.rand(n_spins, generator=g, dtype=f64)
    ph = bp.Phantom(torch.stack([0.006 + u(0, 0.012) * -(-n_spins // 256), u(-2e-4, 2e-4), u(-2e-4, 2e-4)], 1), u(0.5, 2.0),
                    u(0.3, 2.0), u(0.02, 0.3), u(-60.0, 60.0))
    c = torch.complex(*torch.randn(2, n_spins, coils, generator=g, dtype=f64))
    case = driver.prepare_case(ph, scan(33, kinds, 1, 7, spoil), c, chunk=chunk, reuse=True, nufft=nufft)
    assert case.nu is not None and all(case.rf_free) and 20 < case.nu["cols"] <= 32
    out = []
    for changes in (0, 1024):
        assert hip.load().hb_forward_product(case.nu["cols"], case.n_tiles, changes) == (changes == 0)
        case.nu["kind_changes"] = changes
        driver.run_forward(case)
        out.append(driver.read_result(case))
    assert rel(out[0].m, out[1].m) < 1e-5
    assert rel(out[0].signal, out[1].signal) < 2e-6


def test_rule_of_the_reverse():
    """Beside the sweep with one kind from 7 columns on (6 with 8 coils, 5 with 16), inside it for kinds in turn unless the
    coils pay for the weights, and wherever the kernel refuses."""
    beside = adjoint.runs_beside
    for nc, first in ((1, 7), (2, 7), (4, 7), (8, 6), (16, 5)):
        assert all(beside(nc, cols, 0) == (cols >= first) for cols in range(1, 33))
        assert not beside(nc, 33, 0) and beside(nc, 21, 100) and beside(nc, 21, 1024) == (nc == 16)
    assert not beside(3, 21, 0)


@pytest.mark.parametrize("kinds,reps,interval", [(1, 7, 256), (1, 40, 512), (2, 40, 512)])
def test_weights_formed_in_the_reverse(kinds, reps, interval):
    """Every change of kind and every default interval forms them, whatever interval is asked for."""
    from types import SimpleNamespace

    seq = scan(200, kinds, 1, reps)
    plan = nu_mod.make_plan(seq, 6, 3)
    assert adjoint.default_checkpoint_every(len(seq), True) == interval
    case = SimpleNamespace(n_segments=len(seq), nu=dict(plan=plan))
    changes = reps - 1 if kinds > 1 else 0
    assert adjoint._weights_formed(case) == -(-1024 * changes // reps) + -(-1024 * -(-len(seq) // interval) // reps)


@pytest.mark.gpu
@pytest.mark.parametrize("n_spins,coils,kinds,every", [(255, 1, 2, 128), (700, 2, 3, 64), (300, 4, 2, 192)])
def test_beside_on_kinds_in_turn(gpu, monkeypatch, n_spins, coils, kinds, every):
    g = torch.Generator().manual_seed(n_spins)
    u = lambda lo, hi: lo + (hi - lo) * torch.rand(n_spins, generator=g, dtype=f64)
    x = 0.006 + u(0, 0.012) * -(-n_spins // 256)
    ph = bp.Phantom(torch.stack([x, u(-2e-4, 2e-4), u(-2e-4, 2e-4)], 1), u(0.5, 2.0), u(0.3, 2.0), u(0.02, 0.3),
                    u(-60.0, 60.0))
    c = torch.complex(*torch.randn(2, n_spins, coils, generator=g, dtype=f64))
    seq, taken, out = scan(24, kinds, 1, 7), [], []
    for beside in (True, False):
        monkeypatch.setattr(adjoint, "runs_beside", lambda nc, cols, changes, b=beside: taken.append((cols, changes)) or b)
        leaves = {k: getattr(ph, k).clone().requires_grad_() for k in ("pos", "pd", "t1", "t2", "db0")}
        ck = c.clone().requires_grad_()
        r = bp.simulate(replace(ph, **leaves), seq, ck, engine="gpu", pulses="reuse", readouts="nufft",
                        checkpoint_every=every)
        out.append(torch.autograd.grad(weighted_loss(r.signal, r.m), [*leaves.values(), ck]))
    assert taken and all(cols <= 32 and changes > 800 for cols, changes in taken)
    for name, a, b in zip((*leaves, "coils"), *out):
        assert bool(torch.isfinite(a.abs()).all()) and float(b.abs().max()) > 0
        assert rel(a, b) <= 1e-4, name
