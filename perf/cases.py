"""Performance cases of the power-spectrum path: what a user's program has
it do, over the sizes, precisions and options it is used with.

A case is a dict; its ``kind`` names the call sequence:

* ``power``    clear + deposit + fused r2c/binning through a kept ``Plan``
               (the step of the throughput benchmark);
* ``cross``    two species through two plans, one fused binning of both auto
               spectra and the cross spectrum;
* ``density``  clear + deposit + export of the real-space density;
* ``spectrum`` clear + deposit + r2c with the spectrum kept, then binning;
* ``grad``     forward and backward of the band-power chi^2 loss through
               ``genpk_amd.autograd``;
* ``batch``    one launch of a captured batch of uneven realisations;
* ``host``     the reference's host call surface on numpy arrays: fieldize,
               in-place FFT, powerspectrum.

``dims`` is the grid, ``n`` the particle count, ``points`` the particles'
distribution: "clumps" (half uniform, half in Gaussian clumps of power-law
size; any n) or "waves" (an n_side^3 lattice displaced by random plane
waves, n = n_side^3).  ``masses`` gives every particle its own mass.

``exact`` is the same computation in float64 with plain torch: CIC weights
added with index_add_, torch.fft.rfftn, and bins, mode weights and window
factors from their formulas (a window factor is a float by definition, as
in the reference's invwindow).
"""
import math

import numpy as np
import torch

BOX = 1000.0


def listed():
    return [
        # the smallest call: a toy box in a test or a notebook, all latency
        dict(name="power_f64_64", kind="power", precision="f64", dims=64, n=32 ** 3, points="waves", masses=False),
        # the reference's driver switched over as it is: host arrays in and out
        dict(name="host_f64_128", kind="host", precision="f64", dims=128, n=64 ** 3, points="waves", masses=False),
        # one snapshot of a small simulation, grid as fine as the particles
        dict(name="power_f32_256", kind="power", precision="f32", dims=256, n=256 ** 3, points="waves", masses=False),
        # a gas or star species: ragged count, a mass per particle, a grid that is no power of two
        dict(name="power_f64_200_masses", kind="power", precision="f64", dims=200, n=1234567, points="clumps",
             masses=True),
        # the density alone, for a map or another tool
        dict(name="density_f32_384_masses", kind="density", precision="f32", dims=384, n=20000003, points="clumps",
             masses=True),
        # the modes themselves are wanted beside the bins
        dict(name="spectrum_f64_360", kind="spectrum", precision="f64", dims=360, n=240 ** 3, points="waves",
             masses=False),
        # an ordinary large snapshot in the reference's precision
        dict(name="power_f64_512", kind="power", precision="f64", dims=512, n=512 ** 3, points="waves", masses=False),
        # two species of one snapshot and their cross spectrum
        dict(name="cross_f32_512", kind="cross", precision="f32", dims=512, n=512 ** 3, points="waves", masses=False),
        # the largest: the headline workload of the benchmark
        dict(name="power_f32_1024", kind="power", precision="f32", dims=1024, n=1024 ** 3, points="clumps",
             masses=False),
        # one step of a fit of particle positions and masses to a target spectrum
        dict(name="grad_f32_256", kind="grad", precision="f32", dims=256, n=256 ** 3, points="waves", masses=True,
             recompute="auto"),
        # the same at a larger size with the field recomputed instead of kept
        dict(name="grad_f32_512", kind="grad", precision="f32", dims=512, n=100000007, points="clumps", masses=False,
             recompute="always"),
        # a suite of uneven mock catalogues, one launch for all
        dict(name="batch_f32_20", kind="batch", precision="f32", dims=512, n=256 ** 3, points="waves", masses=False,
             count=20),
    ]


def _smooth(lo, hi, even):
    """Grid sizes in [lo, hi]: even 2^a 3^b 5^c for transforms, else any."""
    out = []
    for d in range(lo, hi + 1):
        m = d
        for p in (2, 3, 5):
            while m % p == 0:
                m //= p
        if not even or (m == 1 and d % 2 == 0):
            out.append(d)
    return out


def _near(rng, values, lo, hi):
    """A value at a log-uniform place of [lo, hi]."""
    t = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(values, key=lambda v: abs(math.log(v / t)))


def draw(rng):
    kind = rng.choice(["power", "power", "power", "cross", "density", "spectrum", "grad", "grad", "batch", "host"])
    c = dict(kind=kind, precision=rng.choice(["f32", "f64"]), points=rng.choice(["clumps", "waves"]),
             masses=rng.random() < 0.4)
    lo, hi = 32, {"power": 900, "host": 160, "batch": 384}.get(kind, 640)
    most = {"host": 1 << 21, "batch": 1 << 22}.get(kind, 1 << 28)
    if kind == "density":
        c["dims"] = _near(rng, _smooth(lo, hi, False), lo, hi)
    else:
        c["dims"] = _near(rng, _smooth(lo, hi, True), lo, hi)
    # particles per cell between 1/16 and 16, as samplings of a grid go
    d3 = c["dims"] ** 3
    n = int(math.exp(rng.uniform(math.log(max(4096, d3 // 16)), math.log(min(most, max(8192, 16 * d3))))))
    c["n"] = round(n ** (1 / 3)) ** 3 if c["points"] == "waves" else n
    if kind == "host":
        c["precision"] = "f64"
    if kind == "grad":
        c["recompute"] = rng.choice(["auto", "always"])
    if kind == "batch":
        c["count"] = rng.randint(3, 20)
        c["points"], c["masses"], c["n"] = "waves", False, round(n ** (1 / 3)) ** 3
    return c


# ------------------------------------------------------------------ inputs

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _generator(seed, device):
    g = torch.Generator(device=device)
    g.manual_seed(int(seed))
    return g


def _clumps(n, dims, seed, device, chunk=1 << 26):
    """n particles, half uniform, half in Gaussian clumps of 0.5 to 4 cells
    radius whose sizes follow a power law."""
    g = _generator(seed, device)
    f64 = dict(dtype=torch.float64, device=device)
    pos = torch.empty((n, 3), dtype=torch.float32, device=device)
    nu, k = n // 2, int(min(100000, max(8, n // 2000)))
    nc = n - nu
    for s in range(0, nu, chunk):
        e = min(nu, s + chunk)
        pos[s:e] = (torch.rand((e - s, 3), generator=g, **f64) * BOX).float()
    u = torch.rand(k, generator=g, **f64)
    size = torch.cumsum((1 - u) ** (-1 / 0.9), 0)
    edge = torch.round(size / size[-1] * nc).long()
    centre = torch.rand((k, 3), generator=g, **f64) * BOX
    radius = (0.5 + 3.5 * torch.rand((k, 1), generator=g, **f64)) * (BOX / dims)
    for s in range(0, nc, chunk):
        e = min(nc, s + chunk)
        own = torch.searchsorted(edge, torch.arange(s, e, device=device), right=True).clamp_(max=k - 1)
        x = centre[own] + torch.randn((e - s, 3), generator=g, **f64) * radius[own]
        pos[nu + s:nu + e] = torch.remainder(x, BOX).float()
    return pos


def _waves(n, dims, seed, device, modes=24):
    """A lattice displaced by plane waves of random direction and phase and
    amplitude ~ k / k^2, one cell rms per component."""
    m = round(n ** (1 / 3))
    g = _generator(seed, device)
    f64 = dict(dtype=torch.float64, device=device)
    k = torch.round(torch.randn((modes, 3), generator=g, **f64) * (m / 8))
    phase = 2 * math.pi * torch.rand(modes, generator=g, **f64)
    amp = k * (torch.randn(modes, generator=g, **f64) / k.square().sum(1).clamp(min=1.0))[:, None]
    amp *= (BOX / dims) / (amp.square().sum(0) / 2).sqrt().clamp(min=1e-9)
    at = torch.arange(m, **f64) / m
    pos = torch.empty((m, m, m, 3), dtype=torch.float32, device=device)
    step = max(1, (1 << 23) // (m * m))
    for x0 in range(0, m, step):
        x = at[x0:x0 + step]
        d = torch.zeros((x.shape[0], m, m, 3), **f64)
        for j in range(modes):
            plane = 2 * math.pi * (k[j, 1] * at[:, None] + k[j, 2] * at[None, :]) + phase[j]
            d += torch.sin(plane[None] + 2 * math.pi * k[j, 0] * x[:, None, None])[..., None] * amp[j]
        d[..., 0] += BOX * x[:, None, None]
        d[..., 1] += BOX * at[None, :, None]
        d[..., 2] += BOX * at[None, None, :]
        pos[x0:x0 + step] = torch.remainder(d, BOX).float()
    return pos.reshape(-1, 3)


def _particles(c, seed, device):
    make = _clumps if c["points"] == "clumps" else _waves
    pos = make(c["n"], c["dims"], seed, device)
    masses = None
    if c["masses"]:
        # gas and star particles: masses within a factor of a few
        masses = 0.5 + 1.5 * torch.rand(pos.shape[0], generator=_generator(seed + 7, device), device=device)
    return pos, masses


def _species(c, seed, device):
    """The second species of a cross spectrum: other points of a tenth of the mass."""
    return _particles(c, seed + 1000003, device)


def _jobs(c, seed):
    """Sizes of a batch: the largest as given, the others smaller, uneven, on four grid sizes."""
    rng = np.random.default_rng(1000 + c["count"])
    d0 = c["dims"]
    grids = [d for d in (d0, 3 * d0 // 4, d0 // 2, d0 // 4) if d in _smooth(16, d0, True)]
    m0 = round(c["n"] ** (1 / 3))
    out = []
    for r in range(c["count"]):
        m = max(8, int(round(m0 * math.exp(-rng.uniform(0, math.log(4)))))) if r else m0
        d = int(grids[int(rng.integers(len(grids)))]) if r else d0
        out.append(dict(c, dims=d, n=m ** 3, seed=seed + 31 * r))
    return out


def _total(pos, masses, mass=1.0):
    return float(masses.double().sum()) if masses is not None else mass * pos.shape[0]


def prepare(case, seed):
    import genpk_amd
    from genpk_amd.batch import Batch
    c, dev = case, _device()
    kind = c["kind"]
    if kind == "batch":
        b = Batch(8)
        for j in _jobs(c, seed):
            pos, _ = _particles(j, j["seed"], dev)
            b.add(pos, BOX, j["dims"], precision=c["precision"])
        return dict(kind=kind, batch=b.build())
    pos, masses = _particles(c, seed, dev)
    s = dict(kind=kind, dims=c["dims"], pos=pos, masses=masses, M=_total(pos, masses))
    if kind == "host":
        d = c["dims"]
        s.update(pos=pos.cpu().numpy(), masses=None if masses is None else masses.cpu().numpy(),
                 grid=np.zeros((d, d, 2 * (d // 2 + 1)), np.float64))
        return s
    s["plan"] = genpk_amd.Plan(c["dims"], c["precision"])
    if kind == "cross":
        pos2, masses2 = _species(c, seed, dev)
        s.update(pos2=pos2, masses2=masses2, M2=_total(pos2, masses2, 0.1),
                 plan2=genpk_amd.Plan(c["dims"], c["precision"]))
    elif kind == "density":
        s["out"] = torch.zeros_like(s["plan"].grid)
    elif kind == "grad":
        target, count = _target(c, s["M"], dev)
        s.update(target=target, count=count, recompute=c["recompute"])
        pos.requires_grad_(True)
        if masses is not None:
            masses.requires_grad_(True)
    return s


def _target(c, M, dev):
    """A measured spectrum to fit to: clustering over a noise level, with
    the mode counts of the bins."""
    _, count, keffs = _bins(c["dims"], c["dims"], dev)
    k = keffs.clamp(min=1.0)
    return 1.0 / c["n"] + 1e-4 * k ** -1.5, count


def run(state):
    import genpk_amd
    from genpk_amd import autograd
    s = state
    kind = s["kind"]
    if kind == "batch":
        s["batch"].launch()
        return s["batch"].results()
    d, pos, masses = s["dims"], s["pos"], s["masses"]
    if kind == "host":
        grid = s["grid"]
        grid[:] = 0
        genpk_amd.fieldize(BOX, d, grid, pos, masses)
        spec = genpk_amd.fft_r2c_3d_inplace(grid)
        power, count, keffs = genpk_amd.powerspectrum(d, spec, spec, d, s["M"], s["M"])
        return dict(spectrum=spec, power=power, count=count, keffs=keffs)
    plan = s["plan"]
    if kind == "grad":
        P = autograd.power_spectrum(pos, BOX, d, masses=masses, total_mass=s["M"], plan=plan,
                                    recompute=s["recompute"])
        loss = autograd.chi2_loss(P, s["target"], s["count"])
        wanted = (pos,) if masses is None else (pos, masses)
        return dict(power=P.detach(), grads=torch.autograd.grad(loss, wanted))
    plan.clear()
    plan.deposit(pos, BOX, masses)
    if kind == "density":
        return plan.export_density(s["out"])
    if kind == "spectrum":
        spec = plan.r2c()
        power, count, keffs = plan.bin(mass=s["M"])
        return dict(spectrum=spec, power=power, count=count, keffs=keffs)
    if kind == "cross":
        s["plan2"].clear()
        s["plan2"].deposit(s["pos2"], BOX, s["masses2"], mass=0.1)
        power, count, keffs = plan.power(other=s["plan2"], mass=s["M"], other_mass=s["M2"])
        return dict(power=power, count=count, keffs=keffs)
    power, count, keffs = plan.power(mass=s["M"])
    return dict(power=power, count=count, keffs=keffs)


# -------------------------------------------------------------------- work

def _one(c, d, n, kind):
    """Bytes in and out and operations of one job: positions (and masses)
    read once, results written once; CIC at about 60 operations a particle,
    5 N log2 N / 2 of a real transform."""
    cb = 4 if c["precision"] == "f32" else 8
    cells = d * d * 2 * (d // 2 + 1)
    b = (16 if c["masses"] else 12) * n + 20 * d
    f = 60.0 * n
    if kind == "density":
        return b + cb * cells, f
    f += 2.5 * d ** 3 * math.log2(float(d) ** 3) + 10.0 * cells / 2
    if kind in ("spectrum", "host"):
        b += cb * cells
    if kind == "grad":
        b += (28 if c["masses"] else 24) * n  # particles read again in the backward, gradients written
        f = 2 * f + 60.0 * n
    return b, f


def work(case):
    c = case
    if c["kind"] == "batch":
        parts = [_one(c, j["dims"], j["n"], "power") for j in _jobs(c, 0)]
    else:
        parts = [_one(c, c["dims"], c["n"], c["kind"])] * (2 if c["kind"] == "cross" else 1)
    return {"bytes": sum(b for b, _ in parts), "flops": sum(f for _, f in parts)}


# ------------------------------------------------------------------- exact

def _q_bins(d, nrbins):
    """Bin of every |k|^2 = q >= 1 up to 3 (d/2)^2."""
    per = (nrbins - 1) / math.log(math.sqrt(3.0) * d / 2.0)
    return [0] + [int(math.floor(per * math.log(math.sqrt(q)))) for q in range(1, 3 * (d // 2) ** 2 + 1)]


def _bins(d, nrbins, dev):
    """(bin of q, mode counts, mean |k| per bin), the counts from the number
    of modes of every q of the half spectrum, doubled off its two planes."""
    h = d // 2
    bin_of = torch.tensor(_q_bins(d, nrbins), device=dev)
    k2 = torch.minimum(torch.arange(d, device=dev), d - torch.arange(d, device=dev)) ** 2
    count = torch.zeros(nrbins, dtype=torch.float64, device=dev)
    ksum = torch.zeros(nrbins, dtype=torch.float64, device=dev)
    modes = torch.zeros(3 * h * h + 1, dtype=torch.int64, device=dev)
    plane = (k2[:, None] + k2[None, :]).reshape(-1)
    cnt2 = torch.bincount(plane, minlength=2 * h * h + 1)
    for kz in range(h + 1):
        modes[kz * kz:kz * kz + 2 * h * h + 1] += cnt2 * (1 if kz in (0, h) else 2)
    modes[0] = 0
    q = torch.arange(modes.numel(), device=dev, dtype=torch.float64)
    count.index_add_(0, bin_of, modes.double())
    ksum.index_add_(0, bin_of, modes.double() * q.sqrt())
    return bin_of, count.to(torch.int32), torch.where(count > 0, ksum / count.clamp(min=1), ksum)


def _window(d, dev):
    k = np.arange(d)
    k = np.where(k <= d // 2, k, k - d).astype(np.float64)
    with np.errstate(invalid="ignore", divide="ignore"):
        w = np.pi * k / (d * np.sin(np.pi * k / d))
    w[0] = 1.0
    return torch.from_numpy(w.astype(np.float32)).to(dev)


def _cic(pos, d):
    """Floor cells and fractions of a chunk of positions."""
    u = pos.double() * (d / BOX)
    f = u.floor()
    return torch.remainder(f.long(), d), u - f


def _chunks(n, step=1 << 24):
    return [slice(s, min(n, s + step)) for s in range(0, n, step)]


def _corners(i, f, d):
    for c in range(8):
        b = [(c >> a) & 1 for a in range(3)]
        at = [torch.remainder(i[:, a] + 1, d) if b[a] else i[:, a] for a in range(3)]
        w = [f[:, a] if b[a] else 1 - f[:, a] for a in range(3)]
        yield b, (at[0] * d + at[1]) * d + at[2], w


def _density(pos, masses, mass, d):
    """The CIC density, its sums formed in two integers of 2^-30 and 2^-60
    units (exact to 2^-61 a term; integer atomics also take many particles
    of one cell much faster than float64 ones)."""
    hi = torch.zeros(d ** 3, dtype=torch.int64, device=pos.device)
    lo = torch.zeros_like(hi)
    for s in _chunks(pos.shape[0]):
        i, f = _cic(pos[s], d)
        m = mass if masses is None else masses[s].double()
        for _, at, w in _corners(i, f, d):
            v = w[0] * w[1] * w[2] * m
            h = torch.round(v * 2.0 ** 30)
            hi.index_add_(0, at, h.long())
            lo.index_add_(0, at, torch.round((v - h * 2.0 ** -30) * 2.0 ** 60).long())
    return (hi.double() * 2.0 ** -30 + lo.double() * 2.0 ** -60).reshape(d, d, d)


def _planes(d, bin_of, wt, dev):
    """Per x-plane of the half spectrum: bins and mode weights (Hermitian
    weight times deconvolution; 0 at k = 0), window weight alone."""
    h = d // 2
    k2 = torch.minimum(torch.arange(d, device=dev), d - torch.arange(d, device=dev)) ** 2
    herm = torch.full((h + 1,), 2.0, dtype=torch.float64, device=dev)
    herm[0] = herm[h] = 1.0
    for x in range(d):
        q = k2[x] + k2[:, None] + k2[None, :h + 1]
        g = ((wt[x] * wt[:, None]) * wt[None, :h + 1]).double() ** 4
        g = torch.where(q == 0, torch.zeros_like(g), g)
        yield x, bin_of[q], g, herm


def _power(fields, totals, d, dev):
    """(P of each pair, count, keffs) of one or two spectra."""
    bin_of, count, keffs = _bins(d, d, dev)
    wt = _window(d, dev)
    pairs = [(0, 0)] if len(fields) == 1 else [(0, 0), (1, 1), (0, 1)]
    sums = [torch.zeros(d, dtype=torch.float64, device=dev) for _ in pairs]
    for x, b, g, herm in _planes(d, bin_of, wt, dev):
        for (i, j), s in zip(pairs, sums):
            t = (fields[i][x] * fields[j][x].conj()).real * g * herm
            s.index_add_(0, b.reshape(-1), t.reshape(-1))
    out = [torch.where(count > 0, s / (totals[i] * totals[j]) / count.clamp(min=1), s)
           for (i, j), s in zip(pairs, sums)]
    return out, count, keffs


def _exact_power(c, seed, dev):
    pos, masses = _particles(c, seed, dev)
    F = torch.fft.rfftn(_density(pos, masses, 1.0, c["dims"]))
    (P,), count, keffs = _power([F], [_total(pos, masses)], c["dims"], dev)
    return F, P, count, keffs


def exact(case, seed):
    c, dev, d = case, _device(), case["dims"]
    kind = c["kind"]
    if c["n"] > 1 << 28:
        return None  # too long
    if kind == "batch":
        return [(P, count, keffs) for _, P, count, keffs in (_exact_power(j, j["seed"], dev) for j in _jobs(c, seed))]
    if kind in ("power", "spectrum", "host"):
        F, P, count, keffs = _exact_power(c, seed, dev)
        out = dict(power=P, count=count, keffs=keffs)
        if kind != "power":
            out["spectrum"] = F
        return out
    pos, masses = _particles(c, seed, dev)
    if kind == "density":
        out = torch.zeros((d, d, 2 * (d // 2 + 1)), dtype=torch.float64, device=dev)
        out[..., :d] = _density(pos, masses, 1.0, d)
        return out
    M = _total(pos, masses)
    F = torch.fft.rfftn(_density(pos, masses, 1.0, d))
    if kind == "cross":
        pos2, masses2 = _species(c, seed, dev)
        F2 = torch.fft.rfftn(_density(pos2, masses2, 0.1, d))
        P, count, keffs = _power([F, F2], [M, _total(pos2, masses2, 0.1)], d, dev)
        return dict(power=tuple(P), count=count, keffs=keffs)
    # gradient: dL/dP of the chi^2 loss, then dL/drho = inverse transform of
    # 2 dL/dP_b g F / (M^2 C_b), interpolated at the particles
    (P,), count, _ = _power([F], [M], d, dev)
    target, cnt = _target(c, M, dev)
    occ = (cnt > 0) & (target > 0)
    sig2 = target ** 2 * 2.0 / cnt.double().clamp(min=1)
    lam = torch.where(occ, 2 * (P - target) / sig2, torch.zeros_like(P)) * 2 / (M * M) / count.double().clamp(min=1)
    for x, b, g, _ in _planes(d, _bins(d, d, dev)[0], _window(d, dev), dev):
        F[x] *= lam[b] * g
    G = torch.fft.irfftn(F, s=(d, d, d), norm="forward").reshape(-1)
    del F
    gpos = torch.empty(pos.shape, dtype=torch.float64, device=dev)
    gm = None if masses is None else torch.empty(pos.shape[0], dtype=torch.float64, device=dev)
    for s in _chunks(pos.shape[0]):
        i, f = _cic(pos[s], d)
        acc = torch.zeros((i.shape[0], 4), dtype=torch.float64, device=dev)
        for b, at, w in _corners(i, f, d):
            v = G[at]
            sign = [1.0 if t else -1.0 for t in b]
            acc[:, 0] += sign[0] * w[1] * w[2] * v
            acc[:, 1] += sign[1] * w[0] * w[2] * v
            acc[:, 2] += sign[2] * w[0] * w[1] * v
            acc[:, 3] += w[0] * w[1] * w[2] * v
        m = 1.0 if masses is None else masses[s].double()[:, None]
        gpos[s] = acc[:, :3] * m * (d / BOX)
        if gm is not None:
            gm[s] = acc[:, 3]
    return dict(power=P, grads=(gpos,) if gm is None else (gpos, gm))
