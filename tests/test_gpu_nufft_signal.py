"""hb_nufft_signal on both sides of its rule (one sample a workgroup, four a workgroup) against the same sums in NumPy, GPU:
sample counts around multiples of four, coil counts around groups of eight, one term and several, slots in another order
than the runs.

Tolerance: float64 sums of at most 3 x 256 products in another order, a few hundred roundings of 2^-53: 1e-12 of the
largest value."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,slots,coils,terms", [
    (1, 1, 1, 1), (17, 3, 3, 3), (64, 15, 8, 3), (64, 16, 8, 3), (33, 40, 9, 2), (66, 30, 16, 3), (67, 20, 5, 1)])
def test_signal(gpu, n, slots, coils, terms):
    rng = np.random.default_rng(n + slots)
    ng, tiles, rows0 = 2 * n, -(-coils // 8), 5
    vals, runs = 16 * tiles, slots + 2
    grid = rng.normal(size=(slots, terms, ng, vals))
    run_of = rng.permutation(runs)[:slots].astype(np.int32)
    row_of = (rows0 + n * rng.permutation(runs)).astype(np.int32)
    tw, lw = rng.normal(size=(n, ng, 2)), rng.normal(size=(terms, n))
    psi = rng.uniform(0, 6, rows0 + n * runs)
    dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (grid, run_of, row_of, tw, lw, psi)]
    sig = torch.full((len(psi), coils, 2), float("nan"), dtype=torch.float64, device="cuda")
    g, ro, rw, t, w, ps = (d.data_ptr() for d in dev)
    gpu.lib().nufft_signal(g, slots, ro, rw, n, ng, terms, tiles, coils, t, w, ps, sig.data_ptr())
    got = torch.view_as_complex(sig).cpu().numpy()
    gc = grid[..., 0:2 * coils:2] + 1j * grid[..., 1:2 * coils:2]  # (slots, terms, ng, coils)
    twc = tw[..., 0] + 1j * tw[..., 1]
    ref = np.full(got.shape, np.nan, dtype=complex)
    for s in range(slots):
        rows = row_of[run_of[s]] + np.arange(n)
        y = sum(lw[m][:, None] * (twc @ gc[s, m]) for m in range(terms))
        ref[rows] = y * np.exp(-1j * psi[rows])[:, None]
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.nanmax(np.abs(got - ref)) <= 1e-12 * np.nanmax(np.abs(ref))
