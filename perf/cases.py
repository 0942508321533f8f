"""The framework's work as measured cases: what a user has it do, through its public entry points, over the range of
sizes, coil counts, pulses, readouts and directions it is used with.

A case is a dict of plain values. ``path`` names what runs:

- ``call``: ``simulate`` forward, the whole call on host tensors;
- ``call_grad``: ``simulate`` with gradients and its backward, the whole call (a map fit: pd, t1, t2 and coils);
- ``forward``: a prepared case run forward on resident buffers (``driver.prepare_case`` once, ``run_forward`` per pass),
  as a program does that simulates one scan setup again and again;
- ``adjoint``: the same with checkpoints, then the reverse sweep of sum |signal - data|^2 (spin maps, coils and RF);
- ``full``, ``full_adjoint``: the same two for the full variant (a bound pool and concomitant fields);
- ``recon``: Cartesian coil images and their root-sum-of-squares from k-space on the GPU.

Sequences: ``gre2d`` (hard pulses, ideal spoiling, dummy TRs), ``tse`` (16-echo trains by default), ``gre3d`` (sinc slab
of 200 substeps), ``multislice`` (300-substep slice pulses, one slice after another), ``mt`` (RF-spoiled slice-selective
GRE). Spins, coils and data come from the seed: tissue maps and off-resonance of another seed are other maps.
"""

import math

import numpy as np
import torch

import blochparty_amd as bp
from blochparty_amd import fields, recon
from blochparty_amd import workloads as W
from blochparty_amd.engines import adjoint, driver, full_adjoint
from blochparty_amd.exchange import BoundPool

FOV = 0.22


def listed():
    return [
        # one small 2D scan, called as a notebook does: 2,039 spins, 4,752 segments; launches and host work count
        dict(name="gre2d_64_call", path="call", seq="gre2d", n=64, coils=8, dummies=200),
        # one iteration of a quantitative map fit on a turbo spin echo, checkpoints every 64 segments
        dict(name="tse_128_call_grad", path="call_grad", seq="tse", n=128, coils=8, etl=16),
        # the default options (every RF substep stepped, every sample taken) on a mid-sized 3D scan
        dict(name="gre3d_32_step", path="forward", seq="gre3d", n=32, iso=4, coils=8, pulses="step", readouts="direct"),
        # the flagship 3D workload: a million spins, learned pulse maps, NUFFT readouts
        dict(name="gre3d_64_surrogate_nufft", path="forward", seq="gre3d", n=64, iso=4, coils=8, pulses="surrogate",
             readouts="nufft"),
        # a large array coil on a matrix that is no power of two: two coil tiles, 96-sample readouts
        dict(name="gre3d_96_reuse_nufft", path="forward", seq="gre3d", n=96, iso=1, coils=16, pulses="reuse",
             readouts="nufft"),
        # multi-slice 2D with exact maps of one pulse per slice, every sample taken; 12 coils (a ragged tile)
        dict(name="multislice_128_reuse_direct", path="forward", seq="multislice", n=128, slices=3, iso=8, coils=12,
             pulses="reuse", readouts="direct"),
        # gradients with every RF substep stepped: pulse design and fits where no pulse recurs
        dict(name="gre3d_24_step_adjoint", path="adjoint", seq="gre3d", n=24, iso=4, coils=8, pulses="step",
             readouts="direct"),
        # gradients of a large scan: maps and NUFFT readouts in both sweeps
        dict(name="gre3d_64_reuse_nufft_adjoint", path="adjoint", seq="gre3d", n=64, iso=1, coils=8, pulses="reuse",
             readouts="nufft"),
        # magnetization transfer and a low-field scanner's concomitant fields, 65,536 spins
        dict(name="mt_128_full", path="full", seq="mt", n=128, iso=4, coils=8),
        # and its gradients (a fit of pool and tissue maps) at a fit's usual matrix
        dict(name="mt_64_full_adjoint", path="full_adjoint", seq="mt", n=64, iso=4, coils=8),
        # images: one small 2D slice, and the largest 3D matrix with 16 coils
        dict(name="recon_64_2d", path="recon", dims=2, n=64, coils=8),
        dict(name="recon_128_3d", path="recon", dims=3, n=128, coils=16),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    cap = max(work(c)["flops"] for c in listed())
    while True:
        path = rng.choice(["call", "call_grad", "forward", "forward", "forward", "adjoint", "adjoint", "full",
                           "full_adjoint", "recon"])
        coils = rng.choice([1, 2, 3, 5, 8, 8, 8, 11, 16, 16])
        if path == "call":
            case = dict(path=path, seq="gre2d", n=_log_int(rng, 16, 96), coils=coils, dummies=rng.randrange(0, 201))
        elif path == "call_grad":
            etl = rng.choice([4, 8, 16])
            case = dict(path=path, seq="tse", n=etl * _log_int(rng, 32 // etl, 144 // etl), coils=coils, etl=etl)
        elif path in ("forward", "adjoint"):
            pulses, readouts = rng.choice(["step", "reuse", "reuse"]), rng.choice(["direct", "nufft"])
            if path == "forward" and rng.random() < 0.3:
                case = dict(path=path, seq="multislice", n=_log_int(rng, 32, 192), slices=rng.randrange(1, 6),
                            iso=rng.randrange(1, 9), coils=coils, pulses=pulses, readouts=readouts)
            else:
                big = 80 if path == "forward" and pulses == "reuse" else 48 if pulses == "reuse" else 28
                case = dict(path=path, seq="gre3d", n=_log_int(rng, 12, big), iso=rng.choice([1, 2, 4]), coils=coils,
                            pulses=pulses, readouts=readouts)
                if case["n"] < 17 and readouts == "nufft":  # shorter readouts than a NUFFT takes
                    continue
        elif path in ("full", "full_adjoint"):
            case = dict(path=path, seq="mt", n=_log_int(rng, 24, 160 if path == "full" else 80),
                        iso=rng.randrange(1, 7), coils=coils)
        else:
            dims = rng.choice([2, 3])
            n = _log_int(rng, 16, 1024 if dims == 2 else 128)
            if rng.random() < 0.7:  # matrices are mostly powers of two
                n = 1 << round(math.log2(n))
            case = dict(path=path, dims=dims, n=n, coils=coils)
        if _seconds(case) <= 1.2 and work(case)["flops"] <= cap:
            return case


def _sizes(case):
    """(spins, segments stepped as RF, occurrences of a pulse, readout runs, samples) of a simulated case."""
    n = case["n"]
    if case["seq"] == "gre2d":
        return round(0.498 * n * n), n + case["dummies"], n + case["dummies"], n, n * n
    if case["seq"] == "tse":
        return round(0.498 * n * n), 60 * n, n, n, n * n
    if case["seq"] == "gre3d":
        return n**3 * case["iso"], 200 * n * n, n * n, n * n, n**3
    if case["seq"] == "multislice":
        trs = n * case["slices"]
        return n * n * case["iso"] * case["slices"], 300 * trs, trs, trs, n * trs
    return n * n * case["iso"], 100 * n, n, n, n * n


def work(case):
    """Spins, coils, records, data read once, signal, state and gradients written once; per spin 48 flops per RF
    substep (30 per occurrence of a pulse taken as a map), 12 per free event, 8 per coil and sample (a NUFFT run:
    18 grid columns in place of its samples); twice that and 16 per coil and sample for a gradient."""
    n, c = case["n"], case["coils"]
    if case["path"] == "recon":
        v = n ** case["dims"]
        return dict(bytes=16.0 * c * v + 4.0 * v, flops=5.0 * c * v * math.log2(v) + 4.0 * c * v)
    spins, rf, occ, runs, samples = _sizes(case)
    maps = case.get("pulses", "step") != "step"
    nufft = case.get("readouts") == "nufft"
    events = 6 * occ + (runs if nufft else samples)
    columns = (18 * runs + runs) if nufft else samples
    flops = spins * ((30.0 * occ if maps else 48.0 * rf) + 12.0 * events + 8.0 * c * columns)
    pool = 6 if case["seq"] == "mt" else 0
    nbytes = spins * (4.0 * (14 + pool) + 8.0 * c + 12.0) + samples * 8.0 * c
    if case["path"] in ("call_grad", "adjoint", "full_adjoint"):
        flops = 3.0 * flops + 16.0 * c * spins * columns
        nbytes += spins * (4.0 * (8 + 2 * pool) + 8.0 * c) + samples * 8.0 * c
    return dict(bytes=nbytes, flops=flops)


def _seconds(case):
    """About how long a pass takes (for draw): launches of one wave per SIMD are bound by their chain of segments."""
    if case["path"] == "recon":
        return 1e-3
    spins, rf, occ, runs, samples = _sizes(case)
    rounds = max(1.0, spins / 65536)
    maps = case.get("pulses", "step") != "step"
    chain = (2 * occ if maps else rf) + (20 * runs if case.get("readouts") == "nufft" else samples) + 8 * occ
    per = dict(call=2e-7, call_grad=3e-6, forward=2e-7, adjoint=2e-6, full=1.2e-6, full_adjoint=6e-6)[case["path"]]
    return chain * rounds * per


# ---- inputs


def _gen(seed, salt):
    return torch.Generator().manual_seed(1000003 * (seed % 1000003) + salt)


def _vary(ph, seed, db0_max):
    """Tissue values a few per cent about their classes, and a smooth off-resonance map that reaches +-db0_max."""
    g = _gen(seed, 1)
    jitter = lambda: 1 + 0.1 * (torch.rand(len(ph), generator=g, dtype=torch.float64) - 0.5)
    p = ph.pos / FOV
    k = 4 * (torch.rand(3, 3, generator=g, dtype=torch.float64) - 0.5)
    phase = 2 * math.pi * torch.rand(3, generator=g, dtype=torch.float64)
    db0 = torch.cos(2 * math.pi * p @ k + phase).sum(1) * (db0_max / 3)
    db0[int(db0.argmin())], db0[int(db0.argmax())] = -db0_max, db0_max
    b1 = None if ph.b1 is None else ph.b1
    return bp.Phantom(ph.pos, ph.pd * jitter(), ph.t1 * jitter(), ph.t2 * jitter(), db0, b1=b1)


def _coils(pos, count, seed):
    """Birdcage sensitivities, each coil with a gain and phase of its own."""
    g = _gen(seed, 2)
    gain = 0.8 + 0.4 * torch.rand(count, generator=g, dtype=torch.float64)
    return bp.birdcage_sensitivities(pos, count) * torch.polar(gain, 6.28 * torch.rand(count, generator=g,
                                                                                    dtype=torch.float64))


_ISO = {1: (1, 1, 1), 2: (1, 1, 2), 4: (1, 2, 2)}
_TISSUE = torch.tensor([(0.7, 0.8, 0.080), (0.8, 1.3, 0.110), (1.0, 4.0, 2.0)], dtype=torch.float64)


def _slices(n, slices, iso, seed):
    """Voxels of ``slices`` slices (3 mm, centres 6 mm apart), ``iso`` isochromats through each, three classes in
    smooth patches, B1 in 0.7-1.3."""
    g = _gen(seed, 3)
    plane = bp.grid_positions(n, FOV).reshape(-1, 3)
    z = torch.tensor(W.slice_centres(slices), dtype=torch.float64)[:, None] + \
        ((torch.arange(iso, dtype=torch.float64) + 0.5) / iso - 0.5) * W.SLICE_THICKNESS
    pos = plane[None, :, None, :].expand(slices, n * n, iso, 3).clone()
    pos[..., 2] = z[:, None, :].expand(slices, n * n, iso)
    vox = pos[:, :, 0].reshape(-1, 3) / FOV
    k = 6 * (torch.rand(3, 2, generator=g, dtype=torch.float64) - 0.5)
    label = ((vox @ k).sin().sum(1) * 1.5).clamp(-1, 1).round().long() + 1
    props = _TISSUE[label].repeat_interleave(iso, 0)
    b1 = (0.7 + 0.6 * torch.rand(len(vox), generator=g, dtype=torch.float64)).repeat_interleave(iso)
    return bp.Phantom(pos.reshape(-1, 3), props[:, 0] / iso, props[:, 1], props[:, 2], torch.zeros(len(b1)).double(),
                      b1=b1)


def _inputs(case, seed):
    """(phantom, sequence, coils, scanner or None), host float64."""
    n, kind, scanner = case["n"], case["seq"], None
    if kind == "gre2d":
        ph = _vary(bp.shepp_logan(n, FOV), seed, 40.0)
        seq = bp.gre_2d(n, FOV, n_dummy=case["dummies"], te=5e-3, flip_deg=15.0, tr=10e-3)
    elif kind == "tse":
        ph = _vary(bp.shepp_logan(n, FOV), seed, 40.0)
        seq = bp.tse_2d(n, FOV, etl=case["etl"], tr=1.5, refocus_flip_deg=[150.0] * case["etl"])
    elif kind == "gre3d":
        iso = _ISO[case["iso"]]
        label = torch.randint(0, 3, (max(2, n // 4),) * 3, generator=_gen(seed, 4)).double()
        label = torch.nn.functional.interpolate(label[None, None], size=(n,) * 3, mode="trilinear")[0, 0].round()
        maps = _TISSUE[label.long()]
        ph = _vary(bp.phantom_from_maps(maps[..., 0], maps[..., 1], maps[..., 2], FOV, spins_per_voxel=iso), seed,
                   100.0)
        seq = W.gre3d_sequence(n)
    elif kind == "multislice":
        ph = _vary(_slices(n, case["slices"], case["iso"], seed), seed, 200.0)
        seq = W.multislice_sequence(n, slices=case["slices"])
    else:
        ph = _vary(_slices(n, 1, case["iso"], seed), seed, 100.0)
        f = 0.15 * torch.rand(len(ph), generator=_gen(seed, 5), dtype=torch.float64)
        full = lambda v: torch.full((len(ph),), v, dtype=torch.float64)
        ph.bound = BoundPool(f=f, k=full(30.0), t1=full(1.0), t2=full(12e-6), dw=full(-200.0))
        seq = bp.gre_cartesian((n, n), FOV, flip_deg=20.0, tr=12e-3, slice_thickness=W.SLICE_THICKNESS,
                               rf_duration=2e-3, time_bw_product=4.0, spoiling="rf", system=bp.System(rf_raster=20e-6))
        seq.rf_freq = torch.zeros(len(seq), dtype=torch.float64)
        scanner = bp.Scanner(field_strength=0.55)
    return ph, seq, _coils(ph.pos, case["coils"], seed), scanner


def _data(spins, samples, coils, seed):
    g = _gen(seed, 6)
    return 0.05 * math.sqrt(spins) * torch.complex(torch.randn(samples, coils, generator=g),
                                                   torch.randn(samples, coils, generator=g))


def _kspace(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed % (1 << 31))
    shape = (case["coils"],) + (case["n"],) * case["dims"]
    return torch.view_as_complex(torch.randn(*shape, 2, generator=g, device="cuda"))


def _options(case):
    pulses = case.get("pulses", "step")
    return dict(reuse=pulses == "reuse", surrogate=pulses == "surrogate",
                nufft=(6, 3) if case.get("readouts") == "nufft" else None)


def _single(ph, coils):
    """The inputs in float32, as a fit keeps its parameters."""
    return ph.to(dtype=torch.float32), coils.to(torch.complex64)


class _Grid:
    """What ``reconstruct`` reads of a sequence: the k-space grid of its samples."""

    def __init__(self, shape):
        self.meta = {"kspace_shape": shape}


def prepare(case, seed):
    path = case["path"]
    if path == "recon":
        k = _kspace(case, seed)
        return dict(path=path, signal=k.reshape(k.shape[0], -1), grid=_Grid(tuple(k.shape[1:])))
    ph, seq, coils, scanner = _inputs(case, seed)
    if path == "call":
        return dict(path=path, phantom=ph, seq=seq, coils=coils)
    if path == "call_grad":
        ph, coils = _single(ph, coils)
        for t in (ph.pd, ph.t1, ph.t2, coils):
            t.requires_grad_()
        return dict(path=path, phantom=ph, seq=seq, coils=coils,
                    data=_data(len(ph), seq.n_adc, case["coils"], seed).T.contiguous())
    conc = None
    if scanner is not None:
        spin = fields.spin_fields(scanner, ph.pos)
        conc = (spin.conc, spin.mode)
    if path in ("forward", "full"):
        dev = driver.prepare_case(ph, seq, coils, conc=conc, **_options(case))
        state = dict(path=path, case=dev)
    else:
        opts = _options(case)
        every = adjoint.default_checkpoint_every(len(seq), bodies=opts["reuse"] or opts["nufft"] is not None)
        dev = driver.prepare_case(ph, seq, coils, chunk=every, aligned=True, conc=conc, **opts)
        nc = adjoint.adjoint_width(case["coils"])
        order = coils if dev.perm is None else coils[torch.from_numpy(dev.perm)]
        where = dev.spins.device
        state = dict(path=path, case=dev, every=every, nc=nc, sens=adjoint.adjoint_sens(order, dev.n_pad, nc).to(where),
                     data=torch.view_as_real(_data(dev.n, dev.n_adc, case["coils"], seed)).double().to(where))
    state["inverse"] = None
    if dev.perm is not None:  # NUFFT readouts sort the spins: back to the caller's order
        inverse = torch.empty(dev.n, dtype=torch.int64)
        inverse[torch.from_numpy(dev.perm)] = torch.arange(dev.n)
        state["inverse"] = inverse.to(dev.spins.device)
    return state


def _ordered(state, rows):
    """(k, n) float32 rows of the n spins in the caller's order."""
    rows = rows[:, : state["case"].n].float()
    return rows if state["inverse"] is None else rows[:, state["inverse"]]


def _signal(dev):
    return torch.view_as_complex(dev.sig[: dev.n_adc]).T.to(torch.complex64)


def run(state):
    path = state["path"]
    if path == "recon":
        images = recon.reconstruct(state["signal"], state["grid"])
        return dict(images=images, rss=recon.rss(images))
    if path == "call":
        res = bp.simulate(state["phantom"], state["seq"], state["coils"], engine="gpu")
        return dict(signal=res.signal, m=res.m)
    if path == "call_grad":
        ph, coils = state["phantom"], state["coils"]
        res = bp.simulate(ph, state["seq"], coils, engine="gpu", checkpoint_every=64)
        loss = (res.signal - state["data"]).abs().square().sum()
        g = torch.autograd.grad(loss, [ph.pd, ph.t1, ph.t2, coils])
        return dict(signal=res.signal.detach(), pd=g[0], t1=g[1], t2=g[2], coils=g[3])
    dev = state["case"]
    if path in ("forward", "full"):
        driver.run_forward(dev)
        out = dict(signal=_signal(dev), m=_ordered(state, dev.state[:3] + dev.state[3:]))
        if path == "full":
            out["m_bound"] = dev.extra["mt"]["mb"].sum(0)[: dev.n]
        return out
    ckpts = driver.run_forward(dev, keep=True)
    nc, c = state["nc"], dev.n_coils
    back = 2 * (dev.sig[: dev.n_adc] - state["data"])  # dL/dsignal of sum |signal - data|^2, turned by exp(i psi)
    cp, sp = torch.cos(dev.psi_rows)[:, None], torch.sin(dev.psi_rows)[:, None]
    h = torch.zeros(dev.n_adc, nc, 2, dtype=torch.float32, device=back.device)
    h[:, :c, 0] = (back[..., 0] * cp - back[..., 1] * sp).float()
    h[:, :c, 1] = (back[..., 0] * sp + back[..., 1] * cp).float()
    lam = torch.zeros(3 if path == "adjoint" else 4, dev.n_pad, dtype=torch.float32, device=back.device)
    if path == "adjoint":
        gs, gc, seg, lam = adjoint.run_backward(dev, ckpts, state["every"], h, lam, state["sens"], nc, 2, True)
    else:
        gs, gc, seg, lam = full_adjoint.run_backward(dev, ckpts, state["every"], h, lam, state["sens"], nc, True, True)
    grads = _ordered(state, gs)
    return dict(signal=_signal(dev), coils=_ordered(state, gc)[: 2 * c], m0=_ordered(state, lam), seg=seg.float(),
                **{name: grads[i] for i, name in enumerate(_GRADS[: len(grads)])})


_GRADS = ("px", "py", "pz", "db0", "pd", "r1", "r2", "b1", "c0", "c1", "c2", "c3", "c4", "c5", "c6", "f", "k", "r1b",
          "t2b", "dw")


# ---- the same in 64 bits: torch alone, from the segments


def exact(case, seed):
    if case["path"] == "recon":
        k = _kspace(case, seed).to(torch.complex128)
        axes = tuple(range(1, k.ndim))
        img = torch.fft.fftshift(torch.fft.ifftn(torch.fft.ifftshift(k, dim=axes), dim=axes), dim=axes)
        return dict(images=img, rss=img.abs().square().sum(0).sqrt())
    ph, seq, coils, scanner = _inputs(case, seed)
    grad = case["path"] in ("call_grad", "adjoint", "full_adjoint")
    if case["path"] == "call_grad":
        ph, coils = _single(ph, coils)
    dev = lambda t: t.detach().double().cuda()
    P = dict(pos=dev(ph.pos), pd=dev(ph.pd), r1=1 / dev(ph.t1), r2=1 / dev(ph.t2), db0=dev(ph.db0),
             b1=torch.ones(len(ph), dtype=torch.float64, device="cuda") if ph.b1 is None else dev(ph.b1),
             coils=coils.detach().to(torch.complex128).cuda().T.contiguous())
    if ph.bound is not None:
        b = ph.bound
        P.update(f=dev(b.f), k=dev(b.k), r1b=1 / dev(b.t1), t2b=dev(b.t2), dw=dev(b.dw))
        P["conc"] = dev(fields.spin_fields(scanner, ph.pos).conc)
    if grad:
        for t in P.values():
            t.requires_grad_()
    m0 = torch.stack([torch.zeros_like(P["pd"]), torch.zeros_like(P["pd"]), P["pd"]] +
                     ([P["f"] * P["pd"]] if "f" in P else [])).detach()
    m0.requires_grad_(grad)
    signal, m = _bloch(P, seq, m0, grad)
    if not grad:
        out = dict(signal=signal, m=m[:3])
        if case["path"] == "call":
            out["m"] = m[:3].T
        if case["path"] == "full":
            out["m_bound"] = m[3]
        return out
    data = _data(len(ph), seq.n_adc, case["coils"], seed).to(torch.complex128).cuda().T
    loss = (signal - data).abs().square().sum()
    if case["path"] == "call_grad":  # the starting magnetization is pd's, the rates the times'
        g = torch.autograd.grad(loss, [P["pd"], P["r1"], P["r2"], P["coils"], m0])
        return dict(signal=signal.detach(), pd=g[0] + g[4][2], t1=-g[1] * P["r1"].detach() ** 2,
                    t2=-g[2] * P["r2"].detach() ** 2, coils=g[3].T)
    names = ["pos", "db0", "pd", "r1", "r2", "b1", "coils"] + (["conc", "f", "k", "r1b", "t2b", "dw"] if "f" in P else [])
    g = dict(zip(names + ["m0"], torch.autograd.grad(loss, [P[x] for x in names] + [m0])))
    gc = torch.view_as_real(g["coils"]).permute(0, 2, 1).reshape(-1, len(ph))
    out = dict(signal=signal.detach(), coils=gc, m0=g["m0"], seg=None, px=g["pos"][:, 0], py=g["pos"][:, 1],
               pz=g["pos"][:, 2], **{x: g[x] for x in ("db0", "pd", "r1", "r2", "b1")})
    if "f" in P:
        out.update({f"c{i}": g["conc"][:, i] for i in range(6)}, c6=None, **{x: g[x] for x in ("f", "k", "r1b", "t2b", "dw")})
    return out


def _super_lorentzian(x):
    """sqrt(2 pi) int_0^1 exp(-2 x^2 / (3 u^2 - 1)^2) / |3 u^2 - 1| du, by Gauss-Legendre on both sides of the magic
    angle (u = sin(a) / sqrt 3 and u = cosh(a) / sqrt 3)."""
    t, w = (torch.tensor(v, device=x.device) for v in np.polynomial.legendre.leggauss(160))
    total = torch.zeros_like(x)
    top = math.acosh(math.sqrt(3.0))
    for ti, wi in zip(t, w):
        c = torch.cos(0.25 * math.pi * (ti + 1))
        s = torch.sinh(0.5 * top * (ti + 1))
        total = total + 0.25 * math.pi * wi * torch.exp(-2 * x * x / c**4) / c \
            + 0.5 * top * wi * torch.exp(-2 * x * x / s**4) / s
    return math.sqrt(2 * math.pi / 3) * total


def _bloch(P, seq, m, grad):
    """(signal (C, samples), final state): each distinct pulse composed once into an affine map per spin, free
    precession in closed form, each readout run one product with its phasors."""
    from torch.utils.checkpoint import checkpoint

    pi2 = 2 * math.pi
    dt, rf, g = (t.detach().double().numpy() for t in (seq.dt, seq.rf, seq.grad))
    psi = seq.adc_phase.detach().double()
    is_rf, adc, spoil = (np.asarray(v, dtype=bool) for v in (seq.is_rf, seq.adc, seq.spoil))
    N, pool = P["pd"].shape[0], "f" in P
    again = (lambda fn, *a: checkpoint(fn, *a, use_reentrant=False)) if grad else (lambda fn, *a: fn(*a))
    held = {}

    def once(key, make):
        if key not in held:
            held[key] = make()
        return held[key]

    def offset(gs):
        lin = P["pos"] @ torch.tensor(gs, dtype=torch.float64, device="cuda") + P["db0"]
        if "conc" in P and any(gs):
            x, y, z = gs
            lin = lin + P["conc"] @ torch.tensor([x * x, y * y, z * z, x * y, x * z, y * z], dtype=torch.float64,
                                               device="cuda")
        return lin

    def recover(z, t, sat):
        """Longitudinal relaxation (and exchange) over t of the rows z; z[..., -1, :] columns are affine."""
        if not pool:
            e = torch.exp(-t * P["r1"])
            return z * e, P["pd"] * (1 - e)
        a11, a12, a21 = -(P["r1"] + P["k"] * P["f"]), P["k"], P["k"] * P["f"]
        a22 = -(P["r1b"] + P["k"] + sat)
        c1, c2 = P["r1"] * P["pd"], P["r1b"] * P["f"] * P["pd"]
        det = a11 * a22 - a12 * a21
        s1, s2 = (a12 * c2 - a22 * c1) / det, (a21 * c1 - a11 * c2) / det
        mid, h = 0.5 * (a11 + a22), 0.5 * (a11 - a22)
        q = torch.sqrt(h * h + a12 * a21)
        ea, eb = torch.exp((mid + q) * t), torch.exp((mid - q) * t)
        p, r = 0.5 * (ea + eb), 0.5 * (ea - eb) / q
        k11, k12, k21, k22 = p + r * h, r * a12, r * a21, p - r * h
        lin = torch.stack([k11 * z[0] + k12 * z[1], k21 * z[0] + k22 * z[1]])
        return lin, torch.stack([s1 - k11 * s1 - k12 * s2, s2 - k21 * s1 - k22 * s2])

    def longitudinal(M, t, sat, affine):
        z, add = recover(M[2:] if pool else M[2], t, sat)
        if affine:  # only the last column carries the constant
            z = torch.cat([z[..., :-1, :], (z[..., -1, :] + add)[..., None, :]], dim=-2)
        else:
            z = z + add
        return torch.cat([M[:2], z if pool else z[None]])

    def lineshape(s):
        x = pi2 * (offset(g[s].tolist()) + P["dw"]).abs().clamp_min(1e3) * P["t2b"]
        return P["t2b"] * _super_lorentzian(x)

    def substep(M, s, rx, ry):
        t, w_off = float(dt[s]), offset(g[s].tolist())
        sat = (pi2 * P["b1"]) ** 2 * (rx * rx + ry * ry) * held["line", g[s].tobytes()] if pool else None
        e2 = torch.exp(-0.5 * t * P["r2"])
        half = lambda A: longitudinal(torch.cat([A[:2] * e2, A[2:]]), 0.5 * t, sat, True)
        M = half(M)
        w = [-pi2 * t * P["b1"] * rx, -pi2 * t * P["b1"] * ry, -pi2 * t * w_off]
        p2 = w[0] * w[0] + w[1] * w[1] + w[2] * w[2]
        tiny = p2 < 1e-12  # there the angle's square adds under 1e-13
        phi = torch.sqrt(torch.where(tiny, torch.ones_like(p2), p2))
        a = torch.where(tiny, 1 - p2 / 6, torch.sin(phi) / phi)
        b = torch.where(tiny, 0.5 - p2 / 24, 2 * (torch.sin(phi / 2) / phi) ** 2)
        cross = lambda v: torch.stack([w[1] * v[2] - w[2] * v[1], w[2] * v[0] - w[0] * v[2], w[0] * v[1] - w[1] * v[0]])
        c = cross(M[:3])
        return half(torch.cat([M[:3] + a * c + b * cross(c), M[3:]]))

    def pulse(s, e):
        """(map, phase) of segments [s, e): the map of the pulse turned back by its largest sample's phase."""
        z = rf[s:e, 0] + 1j * rf[s:e, 1]
        turn = float(np.angle(z[np.argmax(np.abs(z))])) if np.abs(z).max() > 0 else 0.0
        z = z * np.exp(-1j * turn)
        key = ("pulse", e - s, np.round(z, 7).tobytes(), np.round(g[s:e], 7).tobytes(), np.round(dt[s:e], 13).tobytes())

        def make():
            D = 3 + pool
            M = torch.zeros(D, D + 1, N, dtype=torch.float64, device="cuda")
            for i in range(D):
                M[i, i] = 1.0
            for i in range(s, e if pool else s):
                once(("line", g[i].tobytes()), lambda: lineshape(i))
            for a in range(s, e, 8):
                def steps(M, a=a):
                    for i in range(a, min(e, a + 8)):
                        M = substep(M, i, float(z[i - s].real), float(z[i - s].imag))
                    return M
                M = again(steps, M)
            return M

        return once(key, make), turn

    def turned(m, a):
        c, s = math.cos(a), math.sin(a)
        return torch.cat([torch.stack([c * m[0] - s * m[1], s * m[0] + c * m[1]]), m[2:]])

    def factors(s, L):
        """Phasor of one segment like s to the powers 1..L, (N, L)."""
        t = float(dt[s])
        rate = torch.complex(-P["r2"], -pi2 * offset(g[s].tolist())) * t
        return torch.exp(rate[:, None] * torch.arange(1, L + 1, device="cuda"))

    def free(m, s, L, E=None):
        if E is None:
            t = float(dt[s])
            E = torch.exp(torch.complex(-P["r2"], -pi2 * offset(g[s].tolist())) * t)
            xy = torch.complex(m[0], m[1]) * E
        else:
            xy = torch.complex(m[0], m[1]) * E[:, -1]
        m = torch.cat([torch.stack([xy.real, xy.imag]), m[2:]])
        return longitudinal(m, float(dt[s]) * L, torch.zeros_like(P["pd"]) if pool else None, False)

    # the segments as pulses, free segments and readout runs
    ops, s, S = [], 0, len(dt)
    same = np.zeros(S, dtype=bool)
    same[1:] = (np.abs(np.diff(dt)) < 1e-13) & (np.abs(np.diff(g, axis=0)) < 1e-6).all(1) & ~spoil[:-1]
    while s < S:
        e = s + 1
        if is_rf[s]:
            while e < S and is_rf[e] and not spoil[e - 1]:
                e += 1
        elif adc[s]:
            while e < S and adc[e] and not is_rf[e] and same[e]:
                e += 1
        ops.append((s, e))
        s = e
    kinds = {}
    for s, e in ops:  # what is composed once and read by every block
        if is_rf[s]:
            pulse(s, e)
        elif adc[s]:
            key = (e - s, round(float(dt[s]), 13), tuple(np.round(g[s], 6)))
            kinds[s] = once(("read",) + key, lambda: factors(s, e - s))
    pad = -N % 2048
    C = P["coils"].shape[0]
    split = lambda t: torch.nn.functional.pad(torch.view_as_real(t), (0, 0, 0, pad)).reshape(*t.shape[:-1], -1, 2048, 2)
    rows = []

    def block(m, *span):
        pend, out = {}, []
        for s, e in span:
            if is_rf[s]:
                M, turn = pulse(s, e)
                u = turned(m, -turn)
                m = turned((M[:, :-1] * u[None]).sum(1) + M[:, -1], turn)
            elif adc[s]:
                pend.setdefault(id(kinds[s]), (kinds[s], []))[1].append((s, torch.complex(m[0], m[1])))
                m = free(m, s, e - s, kinds[s])
            else:
                m = free(m, s, 1)
            if spoil[e - 1]:
                m = torch.cat([torch.zeros_like(m[:2]), m[2:]])
        sc = torch.view_as_complex(split(P["coils"]))  # (C, chunks, 2048)
        for E, runs in pend.values():
            xy = torch.view_as_complex(split(torch.stack([v for _, v in runs])))  # (runs, chunks, 2048)
            left = (xy[:, None] * sc[None]).reshape(-1, *xy.shape[1:]).transpose(0, 1).contiguous()
            right = torch.nn.functional.pad(torch.view_as_real(E), (0, 0, 0, 0, 0, pad))
            right = torch.view_as_complex(right.contiguous()).reshape(-1, 2048, E.shape[1])
            got = torch.bmm(left, right).sum(0).reshape(len(runs), C, -1)
            out += [(s, got[i]) for i, (s, _) in enumerate(runs)]
        out.sort(key=lambda v: v[0])
        return (m,) + tuple(v for _, v in out)

    reads = np.cumsum([bool(adc[s]) and not is_rf[s] for s, _ in ops])
    per = 32
    for b in range(0, int(reads[-1]) // per + 1):
        span = [op for op, k in zip(ops, reads) if k // per == b]
        if span:
            m, *got = again(block, m, *span)
            rows += got
    signal = torch.cat(rows, dim=1)
    return signal * torch.exp(-1j * psi[torch.from_numpy(adc)]).cuda()[None], m
