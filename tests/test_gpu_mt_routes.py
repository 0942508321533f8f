"""The full-variant forward kernel's own routes against the FP64 oracle, GPU: readout runs and RF trains at the lengths
where their loops end (a lone segment, the shortest marked run, around the eight staged samples), cut by dispatches,
ended by spoils; RF segments whose offset factors may and may not be kept; exchange steps on both sides of the series'
limit and at a double eigenvalue; coil counts of every kernel variant. And the marks themselves on the CPU.

Tolerance: float32 steps, some 1,000 per case, against float64 on the same inputs: 1e-5 of the largest value, as the
other cases of this kernel."""

from dataclasses import replace

import numpy as np
import pytest
import torch

import blochparty_amd as bp
from cases import rel
from oracle import exchange as E

f64 = torch.float64


def pooled(n_spins, seed, lineshape="superlorentzian", **pool):
    g = torch.Generator().manual_seed(seed)
    u = lambda lo, hi: lo + (hi - lo) * torch.rand(n_spins, generator=g, dtype=f64)
    p = dict(f=u(0.0, 0.2), k=u(5.0, 60.0), t1=u(0.5, 1.5), t2=u(8e-6, 14e-6), dw=u(-300.0, 100.0))
    p.update(pool)
    pos = torch.stack([u(-0.1, 0.1), u(-0.1, 0.1), u(-3e-3, 3e-3)], 1)
    return bp.Phantom(pos, u(0.5, 1.0), u(0.3, 2.0), u(0.02, 0.3), u(-80.0, 80.0), b1=u(0.8, 1.2),
                      bound=bp.BoundPool(lineshape=lineshape, **p))


def blocks(spans, trains, seed=0):
    """RF trains of the given lengths (gradient, RF frequency and phase changing inside every third) and readouts of
    the given numbers of samples, free segments between, some ends spoiled."""
    rng = np.random.default_rng(seed)
    dt, rf, g, is_rf, adc, spoil, freq = [], [], [], [], [], [], []

    def add(t, w=(0.0, 0.0), grad=(0.0, 0.0, 0.0), r=False, a=False, sp=False, fr=0.0):
        dt.append(t), rf.append(w), g.append(grad), is_rf.append(r), adc.append(a), spoil.append(sp), freq.append(fr)

    for i, (span, train) in enumerate(zip(spans, trains)):
        for j in range(train):
            a = 300.0 * np.sin((j + 1) / (train + 1) * np.pi)
            ph = 0.4 * i + (np.pi if i % 3 == 2 and j > train // 2 else 0.0)
            add(20e-6 if i % 2 else 12e-6, (a * np.cos(ph), a * np.sin(ph)),
                (0.0, 0.0, 1e5 if i % 3 == 1 and j >= train // 2 else 2e5), r=True,
                fr=500.0 if i % 3 == 2 and j % 2 else 0.0)
        add(1e-3, grad=(-300.0, 150.0, -100.0))
        add(4e-4, grad=(200.0, 0.0, 50.0))
        for j in range(span):
            add(10e-6, grad=(4e4, 1e3 * (i % 2), 0.0), a=True, sp=(i % 4 == 3 and j == span - 1))
        add(8e-3, grad=(100.0, 0.0, float(rng.uniform(0, 400))), sp=i % 2 == 0)
    S = len(dt)
    t = lambda v: torch.tensor(np.array(v), dtype=f64)
    psi = t(rng.uniform(0, 6, S))
    return bp.Sequence(t(dt), t(rf), t(g), psi, is_rf, adc, spoil, rf_freq=t(freq))


SPANS, TRAINS = (1, 3, 4, 7, 8, 9, 16, 17, 30), (1, 2, 3, 4, 5, 12, 4, 3, 9)


def check(ph, seq, coils, tol=1e-5, **kw):
    ref_s, ref_m = E.simulate_bound(ph, seq, coils)
    out = bp.simulate(ph, seq, coils, engine="gpu", **kw)
    m4 = torch.cat([out.m, out.m_bound[:, None]], 1).double()
    e = rel(out.signal.to(torch.complex128), ref_s), rel(m4, ref_m)
    print(f"signal {e[0]:.1e}, m {e[1]:.1e}", flush=True)
    assert max(e) < tol, e
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("n_spins,coils,chunk", [(1, 1, 32768), (255, 8, 32768), (257, 9, 37), (300, 16, 50),
                                                 (260, 17, 32768), (64, 33, 41)])
def test_runs_and_trains(gpu, n_spins, coils, chunk):
    ph = pooled(n_spins, n_spins)
    g = torch.Generator().manual_seed(coils)
    c = torch.complex(*(torch.randn(2, n_spins, coils, generator=g, dtype=f64)))
    check(ph, blocks(SPANS, TRAINS), c, chunk=chunk)


@pytest.mark.gpu
@pytest.mark.parametrize("pool", [dict(k=400.0, t1=0.02), dict(k=0.0, f=0.1, t1=1.0), dict(f=0.0, k=30.0),
                                  dict(k=3000.0, f=0.3)], ids=["fast", "double", "none", "stiff"])
def test_exchange_steps(gpu, pool):
    ph = pooled(130, 7, "lorentzian", **pool)
    if pool["k"] == 0.0:  # R1 = R1b: a double eigenvalue
        ph = replace(ph, t1=torch.ones(130, dtype=f64))
    check(ph, blocks((8, 5), (6, 4)), bp.birdcage_sensitivities(ph.pos, 2))


@pytest.mark.gpu
def test_bound_pool_larger_than_the_free_pool_at_the_start(gpu):
    """m_init's Mzb may pass into the free pool and exceed PD: the contraction's scale covers it."""
    ph = pooled(70, 8, k=2000.0, f=torch.full((70,), 0.5, dtype=f64))
    m0 = torch.zeros(70, 4, dtype=f64)
    m0[:, 3] = 4000.0
    seq, coils = blocks((9,), (5,)), bp.birdcage_sensitivities(ph.pos, 3)
    ref_s, _ = E.simulate_bound(ph, seq, coils, m_init=m0)
    out = bp.simulate(ph, seq, coils, engine="gpu", m_init=m0)
    assert rel(out.signal.to(torch.complex128), ref_s) < 1e-5


def test_marks():
    from blochparty_amd.engines import driver, mt

    seq = blocks(SPANS, TRAINS)
    S = len(seq)
    for chunk in (S, 37):
        starts = list(range(0, S, chunk))
        rec = driver.segment_table(seq, starts)
        mt.mark_records(rec, seq, starts, seq.rf_freq.float())
        rf = np.asarray(seq.is_rf)
        prev = None
        for s in range(S):
            if s in starts:
                prev = None
            key = (float(seq.dt[s]), *seq.grad[s].tolist(), float(seq.rf_freq[s]))
            if rf[s]:
                assert bool(rec["flags"][s] & mt.SAME_RF_OFFSET) == (key == prev), s
                prev = key
        runs = [(s, int(rec["pad"][s, 3])) for s in np.flatnonzero(rec["flags"] & driver.RUN)]
        for s, n in runs:
            assert n >= driver.MIN_RUN and len({k // chunk for k in range(s, s + n)}) == 1
            assert all(seq.adc[s:s + n]) and not any(seq.spoil[s:s + n]) and not rf[s:s + n].any()
            assert torch.equal(seq.grad[s:s + n], seq.grad[s].expand(n, 3))
        if chunk == S:
            assert [n for _, n in runs] == [n - (i % 4 == 3) for i, n in enumerate(SPANS) if n - (i % 4 == 3) >= 4]


@pytest.mark.gpu
@pytest.mark.parametrize("n_spins,coils,every", [(40, 1, 64), (300, 5, 64), (600, 16, 192), (256, 0, 128)])
@pytest.mark.parametrize("lineshape", ["superlorentzian", "none"])
def test_reverse_in_chunks(gpu, n_spins, coils, every, lineshape):
    """hb_adjoint_full_chunks with a workspace (the interval reversed in chunks side by side) against hb_adjoint_full
    (one walk): the same float64 sums in another grouping, lambda carried in float64 either way, so 1e-9 of the largest
    (per-segment sums: the float32 partials' rounding, 1e-6)."""
    import ctypes

    from blochparty_amd.engines import adjoint, driver, full_adjoint, hip, mt

    if lineshape == "none":
        ph = replace(pooled(n_spins, 3), bound=None)
    else:
        ph = pooled(n_spins, 3, lineshape)
    seq = blocks(SPANS, TRAINS)
    g = torch.Generator().manual_seed(1)
    conc = (1e-7 * torch.randn(n_spins, 6, generator=g, dtype=f64), 1)
    c = torch.complex(*torch.randn(2, n_spins, max(coils, 1), generator=g, dtype=f64))
    case = driver.prepare_case(ph, seq, c, chunk=every, aligned=True, conc=conc)
    ckpts = driver.run_forward(case, keep=True)
    nc = adjoint.adjoint_width(coils) if coils else 0
    sens = adjoint.adjoint_sens(c, case.n_pad, nc).cuda()
    h = torch.randn(case.n_adc, max(nc, 1), 2, generator=g).cuda()
    h[:, coils:] = 0
    lam0 = torch.randn(4, case.n_pad, generator=g).cuda()
    lam0[:, n_spins:] = 0
    lib = hip.load()
    mt.bind(lib)
    cs, mts = case.struct(), mt.struct(case.extra["mt"])
    z = lambda *s: torch.zeros(*s, dtype=f64, device="cuda")
    outs = []
    for chunks in (False, True):
        gs, gc, lam = z(20, case.n_pad), z(2 * max(nc, 1), case.n_pad), lam0.clone()
        n_blocks = case.n_pad // 256
        traj = torch.empty(every * 4 * case.n_pad, device="cuda")
        gseg = torch.zeros(len(ckpts), n_blocks, every, 8, device="cuda")
        need = lib.hb_adjoint_full_workspace(case.n_pad, every, nc)
        assert need > 0
        work = torch.full((need,), float("nan"), dtype=f64, device="cuda")
        for i in reversed(range(len(ckpts))):
            ad = full_adjoint.HbFullAdjoint(ckpts[i].data_ptr(), ckpts[i][6].data_ptr() if ph.bound else None,
                                            traj.data_ptr(), lam.data_ptr(), gs.data_ptr(), gc.data_ptr(),
                                            gseg[i].data_ptr(), h.data_ptr(), sens.data_ptr(), nc, every, 1, 1)
            rc = lib.hb_adjoint_full_chunks(ctypes.byref(cs), ctypes.byref(mts), ctypes.byref(ad), case.starts[i],
                                            case.ends[i], work.data_ptr() if chunks else None, None)
            assert rc == 0
        torch.cuda.synchronize()
        outs.append((gs[:, :n_spins].cpu(), gc[:, :n_spins].cpu(), lam[:, :n_spins].cpu().double(),
                     gseg.sum(1).cpu().double()))
    for a, b, tol in zip(*outs, (1e-9, 1e-9, 1e-6, 1e-6)):
        scale = a.abs().amax(-1, keepdim=True).clamp_min(1e-300)
        assert bool(((a - b).abs() <= tol * scale.max() if a.ndim > 2 else (a - b).abs() <= tol * scale).all())
