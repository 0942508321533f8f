"""RF trains stepped with several records in flight, GPU: every length around the loop's group, alone and after one
another, equal and changing dt, against the FP64 oracle: the signal and final state, and every gradient (the replay's
trains, the walk of lambda back through RF segments, which ends a group at samples, spoils and interval starts).

Tolerance: the steps are those of any stepped RF segment; the project's bounds on them (1e-5 on m, 1e-4 on the signal and
on gradients)."""

import numpy as np
import pytest
import torch

import blochparty_amd as bp
from cases import random_phantom, rel
from oracle import core
from test_gpu_adjoint import compare

pytestmark = pytest.mark.gpu
f64 = torch.float64


def trains(lengths, seed, ends):
    """A train of each length, then a sample (ends[i] = 1), a spoil (2) or a plain free segment (0)."""
    rng = np.random.default_rng(seed)
    dt, rf, is_rf, adc, spoil = [], [], [], [], []
    for i, n in enumerate(lengths):
        for k in range(n):
            dt.append(10e-6 if rng.random() < 0.8 else 14e-6), rf.append(rng.normal(0, 300, 2))
            is_rf.append(True), adc.append(False), spoil.append(False)
        dt.append(1e-3), rf.append(np.zeros(2)), is_rf.append(False)
        adc.append(ends[i % len(ends)] == 1), spoil.append(ends[i % len(ends)] == 2)
    t = lambda v: torch.tensor(np.array(v), dtype=f64)
    grad = rng.normal(0, 500, (len(dt), 3))
    return bp.Sequence(t(dt), t(rf), t(grad), t(rng.uniform(0, 6, len(dt))), is_rf, adc, spoil)


@pytest.mark.parametrize("lengths,ends,every", [
    ((1, 2, 3, 4, 5, 6, 7, 8, 9, 10), (1, 0), 64), ((66, 3, 61, 1, 2), (1, 2, 0), 64), ((130, 64), (1,), 128)])
def test_train_lengths(gpu, lengths, ends, every):
    ph, seq = random_phantom(300, seed=len(lengths)), trains(lengths, len(lengths), ends)
    coils = bp.birdcage_sensitivities(ph.pos, 3)
    r = bp.simulate(ph, seq, coils, engine="gpu")
    ref_sig, ref_m = core.simulate(ph, seq, coils)
    assert rel(r.m, ref_m) < 1e-5 and rel(r.signal, ref_sig) < 1e-4
    compare(ph, seq, coils, checkpoint_every=every)
