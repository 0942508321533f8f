"""Which spreading NUFFT runs take (hb_forward_product): by the windows' columns, the coil tiles and how often the runs' kind
changes; and the matrix product on kinds in turn with one and two tiles, which the rule no longer sends there, against the
staged spreading (as test_gpu_spread.py, with its tolerance)."""

import pytest
import torch

import blochparty_amd as bp
from blochparty_amd.engines import driver, hip
from blochparty_amd.engines import nufft as nu_mod
from cases import rel
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
