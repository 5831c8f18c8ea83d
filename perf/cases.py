"""Timed cases of the framework: particles -> density -> power spectrum / bispectrum / gradients.

``listed()`` are the cases, ``draw(rng)`` gives others of the same ranges, ``prepare(case, seed)`` makes the
inputs a program has in hand on the GPU, ``run(state)`` is one pass through the public entry points,
``work(case)`` the bytes and operations a pass cannot do without, and ``exact(case, seed)`` the same
results in float64 from plain torch.

Kinds of case
* ``pk``     PkParticles: particles to every P(k) output in one call (the pipeline a survey or simulation
             analysis repeats for each snapshot, realisation and redshift);
* ``ma``     MAS_library.MA: a density grid from particles, 3-D or 2-D (projected mass maps);
* ``pkf``    Pk_library.Pk of a field that is in memory already;
* ``xpk``    Pk_library.XPk: auto and cross spectra of several fields (CDM, gas, neutrinos);
* ``bk``     overdensity + Pk_library.Bk: bispectrum of a particle set over angles theta;
* ``grad``   autograd.pk0: P0(k) forward and d loss / d positions backward;
* ``batch``  PkBatch: many uneven realisations in one launch, results read back;
* ``field``  smoothing, window correction, correlation function, FFT there and back, interpolation.
"""
import math
import random

import numpy as np
import torch

BOX = 1000.0     # Mpc/h
HUBBLE = 100.0   # (km/s)/(Mpc/h)
SCHEMES = ("NGP", "CIC", "TSC", "PCS")
ORDER = {"NGP": 1, "CIC": 2, "TSC": 3, "PCS": 4}
FFT_SIZES = (16, 20, 24, 32, 40, 48, 64, 80, 96, 128, 160, 192, 256, 320, 384, 512)
NTHETA = 20


# ---------------------------------------------------------------------------------------------- cases
def listed():
    return [
        # the smallest call: a test box; launches and the host's part of a call are all there is
        {"name": "pk_small_box", "kind": "pk", "n": 32 ** 3, "order": "lattice", "dims": 32, "MAS": "CIC", "axis": 0,
         "weights": False, "rsd": False, "precision": "fp32"},
        # the benchmark workload: a 512^3 simulation snapshot, one particle per cell, every output
        {"name": "pk_snapshot_512", "kind": "pk", "n": 512 ** 3, "order": "lattice", "dims": 512, "MAS": "CIC",
         "axis": 0, "weights": False, "rsd": False, "precision": "fp32"},
        # a halo catalogue: unordered, clustered, weighted by mass, in redshift space along z; odd count
        {"name": "pk_halos_rsd_tsc", "kind": "pk", "n": 3000017, "order": "halos", "dims": 320, "MAS": "TSC",
         "axis": 2, "weights": True, "rsd": True, "precision": "fp32"},
        # the double precision pipeline (convergence checks), a radix-3 grid, high-order scheme
        {"name": "pk_double_384", "kind": "pk", "n": 256 ** 3, "order": "lattice", "dims": 384, "MAS": "PCS",
         "axis": 1, "weights": False, "rsd": False, "precision": "fp64"},
        # a large density grid with the highest-order scheme (64 cells per particle)
        {"name": "ma_pcs_400", "kind": "ma", "n": 400 ** 3, "order": "lattice", "dims": 400, "axes": 3, "MAS": "PCS",
         "weights": False},
        # gas particles with masses onto a grid whose edge is no multiple of anything convenient
        {"name": "ma_weighted_250", "kind": "ma", "n": 10000019, "order": "halos", "dims": 250, "axes": 3,
         "MAS": "CIC", "weights": True},
        # a projected map: 2-D positions onto an image
        {"name": "ma_map_1000", "kind": "ma", "n": 5000011, "order": "halos", "dims": 1000, "axes": 2, "MAS": "TSC",
         "weights": False},
        # matter components of one snapshot and their crosses, line of sight z (the default axis)
        {"name": "xpk_components_384", "kind": "xpk", "fields": 3, "dims": 384, "axis": 2, "MAS": "CIC",
         "double": False},
        # one realisation of a bispectrum covariance: particles -> delta -> B(theta)
        {"name": "bk_realisation_256", "kind": "bk", "n": 256 ** 3, "order": "lattice", "dims": 256, "MAS": "CIC",
         "k1": 0.1, "k2": 0.2},
        # field-level inference: P0 and the gradient of a loss with respect to every position
        {"name": "grad_256", "kind": "grad", "n": 256 ** 3, "order": "lattice", "dims": 256, "MAS": "CIC",
         "nbins": 64},
        # mock realisations of uneven sizes, one launch for all, spectra read back
        {"name": "batch_mocks_12", "kind": "batch", "jobs": 12, "mix": 5, "n_max": 192 ** 3, "MAS": "CIC", "axis": 0},
        # smoothing of a large field with a filter that is kept
        {"name": "smooth_512", "kind": "field", "op": "smooth", "dims": 512, "MAS": "CIC", "axis": 2, "n": 0,
         "double": False},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _count(rng, MAS, order, hi=None):
    """A particle count: a lattice side cubed, or any number (odd ones among them)."""
    top = hi or {"NGP": 2 ** 27, "CIC": 2 ** 27, "TSC": 2 ** 25, "PCS": 2 ** 24}[MAS]
    n = _logint(rng, 2 ** 12, top)
    return max(16, int(n ** (1.0 / 3.0))) ** 3 if order == "lattice" else n


def draw(rng):
    kind = rng.choice(("pk", "pk", "ma", "ma", "pkf", "xpk", "bk", "grad", "batch", "field"))
    MAS = rng.choice(SCHEMES)
    order = rng.choice(("lattice", "halos"))
    axis = rng.randrange(3)
    fft = [n for n in FFT_SIZES if n <= 320]
    if kind == "pk":
        double = rng.random() < 0.25
        dims = rng.choice(fft if double else FFT_SIZES)
        return {"kind": kind, "n": _count(rng, MAS, order, 2 ** 24 if double else None), "order": order, "dims": dims,
                "MAS": MAS, "axis": axis, "weights": rng.random() < 0.4, "rsd": rng.random() < 0.4,
                "precision": "fp64" if double else "fp32"}
    if kind == "ma":
        axes = 2 if rng.random() < 0.25 else 3
        return {"kind": kind, "n": _count(rng, MAS, order, 2 ** 23 if axes == 2 else 2 ** 24),
                "order": "halos" if axes == 2 else order,
                "dims": _logint(rng, 64, 2000) if axes == 2 else _logint(rng, 24, 400), "axes": axes, "MAS": MAS,
                "weights": rng.random() < 0.5}
    if kind == "pkf":
        double = rng.random() < 0.5
        return {"kind": kind, "dims": rng.choice(fft if double else FFT_SIZES), "axis": axis,
                "MAS": rng.choice(SCHEMES + ("None",)), "double": double, "keep": rng.random() < 0.3,
                "amp": rng.uniform(0.2, 2.0)}
    if kind == "xpk":
        double = rng.random() < 0.3
        return {"kind": kind, "fields": rng.randint(2, 4), "dims": rng.choice([n for n in fft if n <= 256]),
                "axis": axis, "MAS": MAS, "double": double}
    if kind == "bk":
        dims = rng.choice([n for n in fft if 64 <= n <= 256])
        kn = math.pi * dims / BOX
        k1 = rng.uniform(0.15, 0.3) * kn
        return {"kind": kind, "n": _count(rng, "CIC", order, 2 ** 25), "order": order, "dims": dims, "MAS": MAS,
                "k1": k1, "k2": k1 * rng.uniform(1.2, 2.0)}
    if kind == "grad":
        dims = rng.choice([n for n in fft if n >= 32])
        MAS = rng.choice(SCHEMES[1:])   # NGP has no gradient
        return {"kind": kind, "n": _count(rng, MAS, order, 2 ** 23), "order": order, "dims": dims, "MAS": MAS,
                "nbins": rng.randint(4, dims // 2)}
    if kind == "batch":
        return {"kind": kind, "jobs": rng.randint(3, 12), "mix": rng.randrange(1 << 16),
                "n_max": _logint(rng, 2 ** 16, 2 ** 22), "MAS": MAS, "axis": axis}
    op = rng.choice(("smooth", "correct_MAS", "Xi", "fft", "interp"))
    double = op not in ("smooth", "interp") and rng.random() < 0.3
    return {"kind": "field", "op": op, "dims": rng.choice([n for n in FFT_SIZES if n <= (256 if double else 384)]),
            "MAS": MAS, "axis": axis, "n": _count(rng, "CIC", "halos", 2 ** 23) if op == "interp" else 0,
            "double": double}


# --------------------------------------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _smooth_modes(m, g, slope, kc):
    """Half spectrum of a Gaussian random field with P(k) ~ k^-slope exp(-(k/kc)^2) and its wavenumbers."""
    wk = torch.fft.rfftn(torch.randn((m, m, m), generator=g, device="cuda"))
    kf = 2.0 * math.pi / BOX
    f = torch.fft.fftfreq(m, 1.0 / m, device="cuda") * kf
    fz = torch.arange(m // 2 + 1, device="cuda", dtype=torch.float32) * kf
    ks = (f[:, None, None], f[None, :, None], fz[None, None, :])
    k2 = ks[0] ** 2 + ks[1] ** 2 + ks[2] ** 2
    k2[0, 0, 0] = 1.0
    amp = torch.exp(-0.5 * k2 / (kc * kc)) * k2 ** (-0.5 * slope)
    amp[0, 0, 0] = 0.0
    return wk * amp, ks, k2


def _lattice(side, g):
    """Particles of a simulation in the order of their lattice (z fastest): Zel'dovich displacements of
    5 Mpc/h rms."""
    wk, ks, k2 = _smooth_modes(side, g, 1.0, 0.5)
    pos = torch.empty((side ** 3, 3), device="cuda")
    q = (torch.arange(side, device="cuda", dtype=torch.float64) + 0.5) * (BOX / side)
    disp = [torch.fft.irfftn(wk * (1j * k / k2), s=(side,) * 3) for k in ks]
    rms = math.sqrt(sum(float(torch.mean(d.double() ** 2)) for d in disp))
    for a in range(3):
        shape = [1, 1, 1]
        shape[a] = side
        pos[:, a] = torch.remainder(disp[a].double() * (5.0 / rms) + q.reshape(shape), BOX).reshape(-1).float()
    return pos


def _halos(n, g, axes=3):
    """Clustered points in no spatial order: clumps of about 8 with a scatter of 3 Mpc/h."""
    nc = max(1, n // 8)
    cen = torch.rand((nc, axes), generator=g, device="cuda") * BOX
    pos = cen[torch.randint(nc, (n,), generator=g, device="cuda")]
    pos += 3.0 * torch.randn((n, axes), generator=g, device="cuda")
    return torch.remainder(pos, BOX).contiguous()


def _points(case, g):
    if case["order"] == "lattice":
        return _lattice(int(round(case["n"] ** (1.0 / 3.0))), g)
    return _halos(case["n"], g, case.get("axes", 3))


def _field(dims, g, double, amp=1.0):
    """An overdensity field: a smooth Gaussian field plus white noise."""
    wk, _, _ = _smooth_modes(dims, g, 1.5, 0.3)
    f = torch.fft.irfftn(wk, s=(dims,) * 3)
    f = f * (amp / float(f.std())) + 0.3 * torch.randn((dims,) * 3, generator=g, device="cuda")
    return f.double() if double else f.contiguous()


def _batch_sizes(case):
    r = random.Random(case["mix"])
    return [(_logint(r, 2 ** 14, case["n_max"]), r.choice((64, 96, 128, 192, 256)), r.uniform(250.0, 1000.0))
            for _ in range(case["jobs"])]


def _inputs(case, seed):
    """The inputs of a case: tensors on the GPU, from the seed alone."""
    g = _gen(seed)
    kind = case["kind"]
    if kind in ("pk", "ma"):
        s = {"pos": _points(case, g), "W": None, "vel": None}
        n = int(s["pos"].shape[0])
        if case["weights"]:
            s["W"] = torch.exp(0.5 * torch.randn((n,), generator=g, device="cuda"))
        if case.get("rsd"):
            s["vel"] = 300.0 * torch.randn((n, 3), generator=g, device="cuda")
        return s
    if kind == "pkf":
        return {"delta": _field(case["dims"], g, case["double"], case["amp"])}
    if kind == "xpk":
        a = _field(case["dims"], g, case["double"])
        return {"deltas": [a] + [(0.6 * a + 0.5 * _field(case["dims"], g, case["double"])).contiguous()
                                 for _ in range(case["fields"] - 1)]}
    if kind == "bk":
        return {"pos": _points(case, g)}
    if kind == "grad":
        pos = _points(case, g)
        return {"pos": pos, "w": torch.rand((case["nbins"],), generator=g, device="cuda", dtype=torch.float64)}
    if kind == "batch":
        return {"jobs": [(torch.rand((n, 3), generator=g, device="cuda") * np.float32(L), dims, L)
                         for n, dims, L in _batch_sizes(case)]}
    s = {"field": _field(case["dims"], g, case["double"])}
    if case["op"] == "interp":
        s["pos"] = _halos(case["n"], g)
    return s


def _radius(case):
    """Smoothing radius: three cells."""
    return 3.0 * BOX / case["dims"]


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    if case["kind"] == "batch":
        from pylians_amd import batch
        jobs = [{"pos": p, "BoxSize": L, "dims": d, "MAS": case["MAS"], "axis": case["axis"]} for p, d, L in s["jobs"]]
        s["batch"] = batch.PkBatch(jobs, flags=0)
    elif case["kind"] == "grad":
        s["pos"].requires_grad_(True)
    elif case["kind"] == "field" and case["op"] == "smooth":
        from pylians_amd import smoothing_library
        s["filter"] = torch.from_numpy(smoothing_library.FT_filter(BOX, _radius(case), case["dims"], "Gaussian")).cuda()
    return s


# ----------------------------------------------------------------------------------------------- run
PK_NAMES = ("k1D", "Pk1D", "Nmodes1D", "kpar", "kper", "Pk2D", "Nmodes2D", "k3D", "Pk", "Pkphase", "Nmodes3D")
XPK_NAMES = ("k1D", "Pk1D", "PkX1D", "Nmodes1D", "kpar", "kper", "Pk2D", "PkX2D", "Nmodes2D", "k3D", "Pk", "XPk",
             "Nmodes3D")


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "pk":
        from pylians_amd.pipeline import PkParticles
        rsd = {"vel": s["vel"], "Hubble": HUBBLE, "redshift": 0.5} if case["rsd"] else {}
        p = PkParticles(s["pos"], BOX, case["dims"], MAS=case["MAS"], axis=case["axis"], W=s["W"],
                        precision=case["precision"], **rsd)
        return {k: getattr(p, k) for k in PK_NAMES}
    if kind == "ma":
        from pylians_amd import MAS_library
        grid = torch.zeros((case["dims"],) * case["axes"], device="cuda")
        MAS_library.MA(s["pos"], grid, BOX, case["MAS"], W=s["W"])
        return grid
    if kind == "pkf":
        from pylians_amd import Pk_library
        p = Pk_library.Pk(s["delta"], BOX, axis=case["axis"], MAS=case["MAS"], keep_deltak=case["keep"])
        return {k: getattr(p, k) for k in PK_NAMES + (("delta_k",) if case["keep"] else ())}
    if kind == "xpk":
        from pylians_amd import Pk_library
        p = Pk_library.XPk(s["deltas"], BOX, axis=case["axis"], MAS=[case["MAS"]] * case["fields"])
        return {k: getattr(p, k) for k in XPK_NAMES}
    if kind == "bk":
        from pylians_amd import Pk_library
        from pylians_amd.pipeline import overdensity
        delta = overdensity(s["pos"], BOX, case["dims"], MAS=case["MAS"])
        b = Pk_library.Bk(delta, BOX, case["k1"], case["k2"], np.linspace(0.0, np.pi, NTHETA), MAS=case["MAS"])
        return {"B": b.B, "Q": b.Q, "k": b.k, "Pk": b.Pk, "delta": delta}
    if kind == "grad":
        from pylians_amd.autograd import pk0
        P0 = pk0(s["pos"], BOX, case["dims"], MAS=case["MAS"], nbins=case["nbins"])
        grad, = torch.autograd.grad((s["w"] * P0).sum(), s["pos"])
        return {"P0": P0.detach(), "grad": grad}
    if kind == "batch":
        s["batch"].run()
        res = s["batch"].results()
        return {"Pk": [r.Pk for r in res], "k3D": [r.k3D for r in res], "Nmodes3D": [r.Nmodes3D for r in res]}
    from pylians_amd import MAS_library, Pk_library, smoothing_library
    op = case["op"]
    if op == "smooth":
        return smoothing_library.field_smoothing(s["field"], s["filter"])
    if op == "correct_MAS":
        return Pk_library.correct_MAS(s["field"], BOX, MAS=case["MAS"])
    if op == "Xi":
        x = Pk_library.Xi(s["field"], BOX, MAS=case["MAS"], axis=case["axis"])
        return {"r3D": x.r3D, "xi": x.xi, "Nmodes3D": x.Nmodes3D}
    if op == "fft":
        if case["double"]:
            k = Pk_library.FFT3Dr_d(s["field"])
            return {"k": k, "x": Pk_library.IFFT3Dr_d(k)}
        k = Pk_library.FFT3Dr_f(s["field"])
        return {"k": k, "x": Pk_library.IFFT3Dr_f(k)}
    out = torch.empty((case["n"],), device="cuda")
    MAS_library.CIC_interp(s["field"], BOX, s["pos"], out)
    return out


# ---------------------------------------------------------------------------------------------- work
def _fft_flops(N):
    return 2.5 * N ** 3 * 3 * math.log2(N)


def _spectrum_len(N):
    kp, kq, km = N // 2, math.isqrt(2 * (N // 2) ** 2), math.isqrt(3 * (N // 2) ** 2)
    return 6 * km + 3 * kp + 4 * (kp + 1) * (kq + 1)


def work(case):
    kind = case["kind"]
    N = case.get("dims", 0)
    if kind == "ma":
        n, ax, S = case["n"], case["axes"], ORDER[case["MAS"]]
        return {"bytes": n * (4 * ax + (4 if case["weights"] else 0)) + 4 * N ** ax, "flops": n * 2 * S ** ax}
    if kind == "pk":
        n, S = case["n"], ORDER[case["MAS"]]
        per = 12 + (4 if case["weights"] else 0) + (4 if case["rsd"] else 0)
        return {"bytes": n * per + 8 * _spectrum_len(N), "flops": n * 2 * S ** 3 + _fft_flops(N) + 10 * N ** 3}
    if kind == "pkf":
        b = 8 if case["double"] else 4
        out = 8 * _spectrum_len(N) + (2 * b * N * N * (N // 2 + 1) if case["keep"] else 0)
        return {"bytes": b * N ** 3 + out, "flops": _fft_flops(N) + 10 * N ** 3}
    if kind == "xpk":
        F, b = case["fields"], 8 if case["double"] else 4
        return {"bytes": F * b * N ** 3 + 4 * F * (F + 1) * _spectrum_len(N),
                "flops": F * _fft_flops(N) + 4 * F * (F + 1) * N ** 3}
    if kind == "bk":
        S = ORDER[case["MAS"]]
        return {"bytes": 12 * case["n"] + 4 * N ** 3, "flops": case["n"] * 2 * S ** 3 + 4 * _fft_flops(N)}
    if kind == "grad":
        S = ORDER[case["MAS"]]
        return {"bytes": 24 * case["n"], "flops": case["n"] * 8 * S ** 3 + 2 * _fft_flops(N)}
    if kind == "batch":
        S = ORDER[case["MAS"]]
        return {"bytes": sum(12 * n + 8 * _spectrum_len(d) for n, d, _ in _batch_sizes(case)),
                "flops": sum(n * 2 * S ** 3 + _fft_flops(d) + 10 * d ** 3 for n, d, _ in _batch_sizes(case))}
    b, op = 8 if case["double"] else 4, case["op"]
    half = 2 * b * N * N * (N // 2 + 1)
    if op == "smooth":
        return {"bytes": 2 * b * N ** 3 + half, "flops": 2 * _fft_flops(N)}
    if op == "correct_MAS":
        return {"bytes": 2 * b * N ** 3, "flops": 2 * _fft_flops(N)}
    if op == "Xi":
        return {"bytes": b * N ** 3, "flops": 2 * _fft_flops(N) + 10 * N ** 3}
    if op == "fft":
        return {"bytes": 2 * b * N ** 3 + half, "flops": 2 * _fft_flops(N)}
    return {"bytes": 4 * N ** 3 + 16 * case["n"], "flops": 16 * case["n"]}


# --------------------------------------------------------------------------------------------- exact
def _axis_weights(d, MAS, N):
    """[(cell index, weight)] of one coordinate in cell units (float64), differentiable in d."""
    if MAS == "NGP":
        return [(torch.floor(d.detach() + 0.5).long() % N, torch.ones_like(d))]
    if MAS == "CIC":
        b = torch.floor(d.detach())
        return [(b.long() % N, 1.0 - (d - b)), ((b.long() + 1) % N, d - b)]
    lo = torch.floor(d.detach() - (1.5 if MAS == "TSC" else 2.0))
    out = []
    for j in range(1, 4 if MAS == "TSC" else 5):
        t = torch.abs(lo + j - d)
        if MAS == "TSC":
            w = torch.where(t < 0.5, 0.75 - t * t, torch.where(t < 1.5, 0.5 * (1.5 - t) ** 2, torch.zeros_like(t)))
        else:
            w = torch.where(t < 1.0, (4.0 - 6.0 * t * t + 3.0 * t ** 3) / 6.0,
                            torch.where(t < 2.0, (2.0 - t) ** 3 / 6.0, torch.zeros_like(t)))
        out.append(((lo.long() + j) % N, w))
    return out


def _stencil(pos, MAS, N, L):
    """(flat cell, weight) pairs of every stencil cell of (n, axes) float64 positions."""
    ax = [_axis_weights(pos[:, a] * (N / L), MAS, N) for a in range(pos.shape[1])]
    if len(ax) == 2:
        for i0, w0 in ax[0]:
            for i1, w1 in ax[1]:
                yield i0 * N + i1, w0 * w1
        return
    for i0, w0 in ax[0]:
        for i1, w1 in ax[1]:
            i01, w01 = (i0 * N + i1) * N, w0 * w1
            for i2, w2 in ax[2]:
                yield i01 + i2, w01 * w2


def _density(pos, MAS, N, L, W=None):
    axes = int(pos.shape[1])
    rho = torch.zeros(N ** axes, device="cuda", dtype=torch.float64)
    for a in range(0, pos.shape[0], 1 << 24):
        p = pos[a:a + (1 << 24)].double()
        for i, w in _stencil(p, MAS, N, L):
            rho.index_add_(0, i, w if W is None else w * W[a:a + (1 << 24)].double())
    return rho.reshape((N,) * axes)


def _signed(N):
    k = torch.arange(N, device="cuda")
    return torch.where(k > N // 2, k - N, k)


def _window(N, MAS):
    x = _signed(N).double() * (math.pi / N)
    return torch.where(x == 0, torch.ones_like(x), (x / torch.sin(x)) ** ORDER.get(MAS, 0))


def _modes(N):
    """Signed wavenumbers, broadcastable to the half spectrum, and the independent-mode mask."""
    k, h = _signed(N), N // 2
    kx, ky, kz = k[:, None, None], k[None, :, None], torch.arange(h + 1, device="cuda")[None, None, :]
    plane = (kz == 0) | ((kz == h) & (N % 2 == 0))
    edge = (kx == 0) | ((kx == h) & (N % 2 == 0))
    return kx, ky, kz, ~(plane & ((kx < 0) | (edge & (ky < 0))))


def _factor(N, MAS):
    w = _window(N, MAS)
    return w[:, None, None] * w[None, :, None] * w[None, None, :N // 2 + 1]


def _hist(idx, w, n):
    return torch.bincount(idx, weights=w, minlength=n)[:n]


def _spectra(dks, N, L, axis, MAS, pairs):
    """The binned outputs of Pk_library.Pk / XPk for the pairs of half spectra, float64."""
    kx, ky, kz, ok = _modes(N)
    shape = (N, N, N // 2 + 1)
    ok = ok.expand(shape)
    h, kf = N // 2, 2.0 * math.pi / L
    kper_max, kmax = math.isqrt(2 * h * h), math.isqrt(3 * h * h)
    k2 = (kx * kx + ky * ky + kz * kz).expand(shape)[ok]
    kpar = (kx, ky, kz)[axis].expand(shape)[ok].abs()
    k = torch.sqrt(k2.double())
    b3 = torch.floor(k).long()
    b2 = torch.floor(torch.sqrt((k2 - kpar * kpar).double())).long() * (h + 1) + kpar
    in1 = k2 <= h * h
    b1 = kpar[in1]
    mu2 = torch.where(k2 == 0, torch.zeros_like(k), (kpar / torch.clamp(k, min=1e-30)) ** 2)
    n2 = (h + 1) * (kper_max + 1)
    one = torch.ones_like(k)
    N3, N1, N2 = _hist(b3, one, kmax + 1)[1:], _hist(b1, one[in1], h + 1)[1:], _hist(b2, one, n2)
    unit = (L / N ** 2) ** 3
    k1 = torch.arange(1, h + 1, device="cuda").double() * kf
    i2 = torch.arange(n2, device="cuda")
    out = {"k3D": _hist(b3, k, kmax + 1)[1:] / N3 * kf, "Nmodes3D": N3, "k1D": k1, "Nmodes1D": N1, "Nmodes2D": N2,
           "kpar": 0.5 * (2 * (i2 % (h + 1)) + 1).double() * kf, "kper": 0.5 * (2 * (i2 // (h + 1)) + 1).double() * kf}
    dk = [d[ok] * _factor(N, MAS)[ok] for d in dks]
    P3, P1, P2 = [], [], []
    for a, b in pairs:
        v = dk[a].real * dk[b].real + dk[a].imag * dk[b].imag
        L2, L4 = (3.0 * mu2 - 1.0) / 2.0, (35.0 * mu2 * mu2 - 30.0 * mu2 + 3.0) / 8.0
        P3.append(torch.stack([_hist(b3, v, kmax + 1)[1:] / N3 * unit, _hist(b3, v * L2, kmax + 1)[1:] * 5.0 / N3 * unit,
                               _hist(b3, v * L4, kmax + 1)[1:] * 9.0 / N3 * unit], dim=1))
        area = math.pi * torch.clamp((h * kf) ** 2 - k1 * k1, min=0.0)
        P1.append(_hist(b1, v[in1], h + 1)[1:] * unit * (area / N1) / (2.0 * math.pi) ** 2)
        P2.append(_hist(b2, v, n2) * unit / N2)
    if len(pairs) == 1:
        ph = torch.atan2(dk[0].real, torch.abs(dk[0]))
        out.update(Pk=P3[0], Pk1D=P1[0], Pk2D=P2[0], Pkphase=_hist(b3, ph * ph, kmax + 1)[1:] / N3 * unit)
        return out
    F = len(dks)
    for name, cross, v in (("Pk", "XPk", torch.stack(P3, dim=2)), ("Pk1D", "PkX1D", torch.stack(P1, dim=1)),
                           ("Pk2D", "PkX2D", torch.stack(P2, dim=1))):
        out[name], out[cross] = v[..., :F], v[..., F:]
    return out


def _delta(pos, MAS, N, L, W=None):
    mass = float(pos.shape[0]) if W is None else float(W.double().sum())
    return _density(pos, MAS, N, L, W) * (N ** 3 / mass) - 1.0


def _redshift_space(pos, vel, axis):
    """The shift of the redshift-space positions, which are float32 like the positions."""
    L = np.float32(BOX)
    fac = float(np.float32(1.5 / HUBBLE))
    p = pos.clone()
    x = p[:, axis] + vel[:, axis] * fac
    p[:, axis] = torch.where((x > L) | (x < 0), torch.fmod(x + float(L), float(L)), x)
    return p


def _bispectrum(delta, N, L, k1, k2, MAS):
    kf = 2.0 * math.pi / L
    theta = np.linspace(0.0, np.pi, NTHETA)
    kall = np.concatenate([[k1, k2], np.sqrt((k2 * np.sin(theta)) ** 2 + (k2 * np.cos(theta) + k1) ** 2)])
    dk = torch.fft.rfftn(delta) * _factor(N, MAS)
    kx, ky, kz, _ = _modes(N)
    k = torch.sqrt((kx * kx + ky * ky + kz * kz).double())

    def shell(i):
        m = ((k >= (kall[i] - kf) / kf) & (k < (kall[i] + kf) / kf)).double()
        return torch.fft.irfftn(dk * m, s=(N,) * 3), torch.fft.irfftn(m + 0j, s=(N,) * 3)

    uP, uB = (L / N ** 2) ** 3, (L ** 2 / N ** 3) ** 3
    (d1, i1), (d2, i2) = shell(0), shell(1)
    Pk = [float((d * d).sum() / (i * i).sum()) * uP for d, i in ((d1, i1), (d2, i2))]
    B, Q = [], []
    for j in range(NTHETA):
        d3, i3 = shell(j + 2)
        Pk.append(float((d3 * d3).sum() / (i3 * i3).sum()) * uP)
        B.append(float((d1 * d2 * d3).sum() / (i1 * i2 * i3).sum()) * uB)
        Q.append(B[-1] / (Pk[0] * Pk[1] + Pk[0] * Pk[-1] + Pk[1] * Pk[-1]))
    return {"B": np.array(B), "Q": np.array(Q), "k": kall, "Pk": np.array(Pk)}


def _gradient(pos, w, N, L, MAS):
    p = pos.detach().double().requires_grad_(True)
    rho = torch.zeros(N ** 3, device="cuda", dtype=torch.float64)
    for i, wt in _stencil(p, MAS, N, L):
        rho = rho.index_add(0, i, wt)
    dk = torch.fft.rfftn(rho.reshape((N,) * 3) * (N ** 3 / float(p.shape[0])) - 1.0)
    kx, ky, kz, ok = _modes(N)
    shape = (N, N, N // 2 + 1)
    ok = ok.expand(shape)
    bins = torch.floor(torch.sqrt((kx * kx + ky * ky + kz * kz).expand(shape)[ok].double())).long()
    f = _factor(N, MAS)[ok] ** 2
    power = (dk.real ** 2 + dk.imag ** 2)[ok] * f
    nb = math.isqrt(3 * (N // 2) ** 2) + 1
    sums = torch.zeros(nb, device="cuda", dtype=torch.float64).index_add(0, bins, power)
    cnt = torch.bincount(bins, minlength=nb).double()
    P0 = (sums / cnt * (L / N ** 2) ** 3)[1:1 + w.numel()]
    grad, = torch.autograd.grad((w * P0).sum(), p)
    return {"P0": P0.detach(), "grad": grad}


def _xi(field, N, L, MAS, axis):
    dk = torch.fft.rfftn(field) * _factor(N, MAS)
    xi = torch.fft.irfftn((dk.real ** 2 + dk.imag ** 2) + 0j, s=(N,) * 3).reshape(-1)
    o = _signed(N)
    X, Y, Z = o[:, None, None], o[None, :, None], o[None, None, :]
    r = torch.sqrt((X * X + Y * Y + Z * Z).double())
    mu = torch.where(r == 0, torch.zeros_like(r), (X, Y, Z)[axis] / torch.clamp(r, min=1e-30)).reshape(-1)
    r = r.reshape(-1)
    b, nb = torch.floor(r).long(), math.isqrt(3 * (N // 2) ** 2) + 1
    m2 = mu * mu
    n = _hist(b, torch.ones_like(r), nb)[1:]
    x = [_hist(b, xi * f, nb)[1:] * c / n / N ** 3 for c, f in
         ((1.0, torch.ones_like(r)), (5.0, (3.0 * m2 - 1.0) / 2.0), (9.0, (35.0 * m2 * m2 - 30.0 * m2 + 3.0) / 8.0))]
    return {"r3D": _hist(b, r, nb)[1:] / n * (L / N), "xi": torch.stack(x, dim=1), "Nmodes3D": n}


def exact(case, seed):
    s = _inputs(case, seed)
    kind, N, MAS = case["kind"], case.get("dims"), case.get("MAS")
    if kind == "ma":
        return _density(s["pos"], MAS, N, BOX, s["W"])
    if kind == "pk":
        pos = _redshift_space(s["pos"], s["vel"], case["axis"]) if case["rsd"] else s["pos"]
        dk = torch.fft.rfftn(_delta(pos, MAS, N, BOX, s["W"]))
        return _spectra([dk], N, BOX, case["axis"], MAS, [(0, 0)])
    if kind == "pkf":
        dk = torch.fft.rfftn(s["delta"].double())
        out = _spectra([dk], N, BOX, case["axis"], MAS, [(0, 0)])
        if case["keep"]:
            out["delta_k"] = torch.where(_modes(N)[3], dk * _factor(N, MAS), dk)
        return out
    if kind == "xpk":
        F = case["fields"]
        pairs = [(i, i) for i in range(F)] + [(i, j) for i in range(F) for j in range(i + 1, F)]
        return _spectra([torch.fft.rfftn(d.double()) for d in s["deltas"]], N, BOX, case["axis"], MAS, pairs)
    if kind == "bk":
        delta = _delta(s["pos"], MAS, N, BOX)
        return dict(_bispectrum(delta, N, BOX, case["k1"], case["k2"], MAS), delta=delta)
    if kind == "grad":
        return _gradient(s["pos"], s["w"], N, BOX, MAS)
    if kind == "batch":
        res = []
        for pos, d, L in s["jobs"]:
            dk = torch.fft.rfftn(_delta(pos, MAS, d, L))
            res.append(_spectra([dk], d, L, case["axis"], MAS, [(0, 0)]))
        return {name: [r[name] for r in res] for name in ("Pk", "k3D", "Nmodes3D")}
    f, op = s["field"].double(), case["op"]
    if op == "smooth":
        o = _signed(N)
        d2 = (o[:, None, None] ** 2 + o[None, :, None] ** 2 + o[None, None, :] ** 2).double()
        w = torch.exp(-d2 / (2.0 * (_radius(case) * N / BOX) ** 2))
        return torch.fft.irfftn(torch.fft.rfftn(f) * torch.fft.rfftn(w / w.sum()), s=(N,) * 3)
    if op == "correct_MAS":
        dk = torch.fft.rfftn(f)
        return torch.fft.irfftn(torch.where(_modes(N)[3], dk * _factor(N, MAS), dk), s=(N,) * 3)
    if op == "Xi":
        return _xi(f, N, BOX, MAS, case["axis"])
    if op == "fft":
        return {"k": torch.fft.rfftn(f), "x": f}
    out = torch.zeros(case["n"], device="cuda", dtype=torch.float64)
    flat = f.reshape(-1)
    for i, w in _stencil(s["pos"].double(), "CIC", N, BOX):
        out += flat[i] * w
    return out
