"""Performance cases of the estimators: the calls a user's program makes, over the sizes they are made at.

A case is a dict of plain values.  ``kind`` names the entry point:

  estimate   correlations.estimate(x, y, z[, w])          one call, particles -> P_0,2,4(k)
  estimator  correlations.Estimator(...).run(x, y, z)     the same with everything preallocated
  assign     mas.cic_mas_vec / tsc_mas_vec                particles -> mesh
  powspec    correlations.powspec_vec[_fundamental]       mesh -> P_0,2,4(k)
  xi         correlations.xi_vec                          mesh -> xi_0,2,4(s)
  bispec     correlations.bispec                          mesh -> P, B, Q of triangles
  grad       autodiff.estimate_ad + backward()            dLoss/dpositions (and /dweights)
  mock       gauss_field.lognormal_mock, then estimate()  seed -> fields, catalogue size and its P_0,2,4(k)
  batch      batch.BatchEstimator.set(...).run()          many uneven catalogues per launch

Particles are drawn from a lognormal field with a redshift-space scatter along z, so the
cells' occupation is as uneven as a real catalogue's; ``order`` is 'shuffled' (survey and
simulation catalogues, in no order) or 'cells' (what a mock generator writes).  ``aos``
gives the positions as columns of one (N, 3) array, else as three vectors.
"""
import math

import numpy as np
import torch

from jax_powspec_amd import autodiff, batch, correlations, gauss_field, mas

DEVICE = "cuda"
BIAS, GROWTH = 1.1, 0.8
# mesh sides with a compiled transform: 2^a and 3 2^a
SIDES = (32, 48, 64, 96, 128, 192, 256, 384, 512, 768, 1024)


def _particles(name, kind, n, particles, *, box=1000.0, scheme="CIC_REF", bins="half", weights=False, aos=True,
               order="shuffled", **more):
    return dict(name=name, kind=kind, n=n, particles=particles, box=box, scheme=scheme, bins=bins, weights=weights,
                aos=aos, order=order, **more)


def listed():
    return [
        # the smallest call: a few thousand objects of a small box (tests, quick looks);
        # launches and host work are all there is
        _particles("estimate-32", "estimate", 32, 20_000, box=500.0),
        # one simulation snapshot's halo catalogue, bins in k_F up to Nyquist
        _particles("estimate-128", "estimate", 128, 1_000_000, bins="kf"),
        # a weighted galaxy catalogue on a 3 2^a mesh: TSC, separate columns, an odd count
        _particles("estimate-384-tsc", "estimate", 384, 3_141_593, box=1200.0, scheme="TSC", weights=True, aos=False),
        # the headline: a survey-sized mock catalogue, repeated estimates with one estimator
        _particles("estimator-512", "estimator", 512, 20_000_000, box=1500.0),
        # the largest mesh, with the largest catalogue the serving mix holds
        _particles("estimate-1024", "estimate", 1024, 30_000_000, box=1500.0),
        # the drop-in mass assignment of a reference script (its mesh goes on to the user)
        _particles("assign-512", "assign", 512, 20_000_000, box=1500.0),
        # the drop-in P(k) of a mesh in fundamental bins (several hundred of them)
        dict(name="powspec-512", kind="powspec", n=512, box=1500.0, bins="fundamental", scheme="CIC"),
        # fitting particle positions to a target P(k): one forward and backward
        _particles("grad-256", "grad", 256, 2_000_000, scheme="CIC"),
        # the correlation function out to 200 Mpc/h in 5 Mpc/h bins
        dict(name="xi-512", kind="xi", n=512, box=1500.0, bins="s200", scheme="CIC"),
        # the bispectrum of k1 = 0.1, k2 = 0.2 at 20 angles
        dict(name="bispec-256", kind="bispec", n=256, box=1000.0, angles=20, scheme="CIC"),
        # one mock of a covariance: a survey-sized redshift-space catalogue and its P(k)
        dict(name="mock-512", kind="mock", n=512, box=1500.0, particles=20_000_000, growth=True),
        # a covariance set: uneven mocks of one mesh side, CIC and TSC in turn
        _particles("batch-128", "batch", 128, 500_000, bins="kf", jobs=16),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges above: any kind, mesh side, catalogue size and option."""
    kind = rng.choice(["estimate", "estimate", "estimator", "assign", "powspec", "xi", "bispec", "grad", "mock", "batch"])
    limits = {"estimate": (32, 1024), "estimator": (32, 1024), "assign": (32, 512), "powspec": (32, 512),
              "xi": (48, 512), "bispec": (64, 512), "grad": (32, 384), "mock": (64, 512), "batch": (64, 256)}
    lo, hi = limits[kind]
    n = rng.choice([s for s in SIDES if lo <= s <= hi])
    box = round(rng.uniform(500.0, 1500.0), 1)
    case = dict(kind=kind, n=n, box=box)
    if kind in ("powspec", "xi", "bispec"):
        case["scheme"] = rng.choice(["CIC", "CIC", "NONE"])
        if kind == "powspec":
            case["bins"] = rng.choice(["half", "kf", "fundamental"])
        elif kind == "xi":
            case["bins"] = rng.choice(["s200", "s100"])
        else:
            case["angles"] = rng.randint(5, 24)
        return case
    # catalogues: from about one object per 16 cells to sixteen per cell, 1e4 .. 3e7 of them
    cells = n ** 3
    most = {"grad": 5_000_000, "assign": 20_000_000, "mock": 20_000_000, "batch": 1_000_000}.get(kind, 30_000_000)
    top = min(most, max(40_000, 16 * cells))
    case["particles"] = _log_int(rng, min(max(10_000, cells // 16), top // 2), top)
    if kind == "mock":
        return dict(case, growth=rng.random() < 0.5)
    schemes = ["CIC_REF", "TSC"] if kind == "assign" else ["CIC_REF", "CIC", "TSC"]
    case.update(scheme=rng.choice(schemes if n < 768 else schemes[:2]), bins=rng.choice(["half", "kf", "fundamental"]),
                weights=rng.random() < 0.4 and n < 768, aos=rng.random() < 0.6 or n >= 768,
                order=rng.choice(["shuffled", "cells"]))
    if kind == "grad":
        case.update(aos=True, bins=rng.choice(["half", "kf"]))
    if kind == "batch":
        case["jobs"] = rng.randint(4, 20)
    return case


# ------------------------------------------------------------------------------------
# inputs
# ------------------------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _power(k):
    return 2e4 * (np.maximum(k, 1e-12) / 0.05) ** -1.5 * np.exp(-(k / 0.5) ** 2)


def _density(n, box, g):
    """A lognormal density mesh of unit mean, float32 (n, n, n)."""
    kf = 2 * math.pi / box
    ki = torch.fft.fftfreq(n, d=1.0 / n, device=DEVICE)
    kz = torch.fft.rfftfreq(n, d=1.0 / n, device=DEVICE)
    k = kf * torch.sqrt(ki[:, None, None] ** 2 + ki[None, :, None] ** 2 + kz[None, None, :] ** 2)
    k.clamp_(min=1e-12)
    amp = torch.sqrt(2e4 / (box / n) ** 3 * (k / 0.05) ** -1.5 * torch.exp(-(k / 0.5) ** 2))
    amp[0, 0, 0] = 0.0
    wk = torch.fft.rfftn(torch.randn((n, n, n), device=DEVICE, generator=g))
    wk *= amp
    rho = torch.exp(torch.fft.irfftn(wk, s=(n, n, n)))
    return rho / rho.mean()


def _catalogue(case, particles, g):
    """(positions, weights): float32 (N, 3) in [0, box) and float32 (N) or None."""
    m = min(case["n"], 256)
    box = case["box"]
    # whole numbers, so that the same seed gives the same cells whatever the scan's order
    cdf = torch.cumsum((_density(m, box, g).reshape(-1).double() * 2.0 ** 24).long(), 0)
    u = (torch.rand(particles, device=DEVICE, generator=g, dtype=torch.float64) * cdf[-1]).long()
    if case["order"] == "cells":
        u = u.sort().values
    cell = torch.searchsorted(cdf, u, right=True).clamp_(max=m ** 3 - 1)
    del cdf, u
    pos = torch.stack((cell // (m * m), (cell // m) % m, cell % m), 1).float()
    del cell
    pos += torch.rand((particles, 3), device=DEVICE, generator=g)
    pos *= box / m
    pos[:, 2] += 4.0 * torch.randn(particles, device=DEVICE, generator=g)
    pos = torch.remainder(pos, box).clamp_(0.0, box * (1.0 - 2e-6))
    w = None
    if case["weights"]:
        w = 0.5 + torch.rand(particles, device=DEVICE, generator=g)
    return pos, w


def _columns(case, pos):
    if case["aos"]:
        return [pos[:, 0], pos[:, 1], pos[:, 2]]
    return [pos[:, a].contiguous() for a in range(3)]


def _k_edges(case):
    """k bin edges in h/Mpc; None selects the fundamental bins."""
    n, kf = case["n"], 2 * math.pi / case["box"]
    if case["bins"] == "half":
        return kf * (0.5 + np.arange(n // 2 + 1))
    if case["bins"] == "kf":   # off the integers by an irrational amount: no mode lies on an edge
        return kf * (np.arange(1, n // 2 + 1) - 1e-3 * math.sqrt(2))
    return None


def _s_edges(case):
    top = 200.0 if case["bins"] == "s200" else 100.0
    return np.arange(1e-3, min(top, 0.45 * case["box"]), 5.0)


def _jobs(case):
    """Catalogue sizes of a batch: uneven, from a fifth of case['particles'] to three times it."""
    j = case["jobs"]
    return [max(1000, int(case["particles"] * 0.2 * 15.0 ** (i / max(1, j - 1)))) for i in range(j)]


def _batch_case(case, i):
    return dict(case, scheme="CIC" if i % 2 == 0 else "TSC")


def prepare(case, seed):
    kind, n, box = case["kind"], case["n"], case["box"]
    g = _generator(seed)
    s = dict(case=case)
    if kind in ("powspec", "xi", "bispec"):
        s["delta"] = _density(n, box, g) - 1.0
        if kind == "powspec":
            s["edges"] = _k_edges(case)
        elif kind == "xi":
            s["edges"] = _s_edges(case)
        else:
            s["theta"] = np.linspace(0.1, math.pi - 0.1, case["angles"])
        return s
    if kind == "mock":
        s["k"] = np.geomspace(1e-4, 50.0, 512)
        s["pk"] = _power(s["k"])
        s["seed"] = seed
        s["edges"] = 2 * math.pi / box * (0.5 + np.arange(n // 2 + 1))
        return s
    if kind == "batch":
        s["catalogues"] = []
        for i, particles in enumerate(_jobs(case)):
            pos, w = _catalogue(case, particles, g)
            x, y, z = _columns(case, pos)
            s["catalogues"].append(dict(x=x, y=y, z=z, w=w, box_size=box, n_bins=n, mas=_batch_case(case, i)["scheme"],
                                        k_edges=_k_edges(case), shot_noise=box ** 3 / particles))
        bins = len(_exact_edges(case)) - 1
        s["batch"] = batch.BatchEstimator(n, case["jobs"], max(_jobs(case)), bins)
        return s
    pos, w = _catalogue(case, case["particles"], g)
    s["edges"] = _k_edges(case)
    s["shot"] = box ** 3 / case["particles"]
    if kind == "grad":
        s["pos"] = pos.requires_grad_()
        s["w"] = None if w is None else w.requires_grad_()
        s["target"] = _target(case)
        return s
    s["xyz"], s["w"] = _columns(case, pos), w
    if kind == "estimator":
        s["estimator"] = correlations.Estimator(box_size=box, n_bins=n, max_particles=case["particles"],
                                                k_edges=s["edges"], mas=case["scheme"], shot_noise=s["shot"])
    if kind == "assign":
        s["delta"] = torch.zeros((n, n, n), device=DEVICE)
        if w is None:
            s["w"] = torch.ones(case["particles"], device=DEVICE)
    return s


def _target(case, dtype=torch.float32):
    e = _k_edges(case)
    k = 0.5 * (e[1:] + e[:-1])
    p = _power(k) + case["box"] ** 3 / case["particles"]
    return torch.as_tensor(p, device=DEVICE, dtype=dtype)


def _loss(pk, target):
    return (((pk[:, 0] - target) / (0.05 * target)) ** 2).mean()


# ------------------------------------------------------------------------------------
# one pass
# ------------------------------------------------------------------------------------
def run(s):
    case = s["case"]
    kind, n, box = case["kind"], case["n"], case["box"]
    if kind == "estimate":
        x, y, z = s["xyz"]
        return correlations.estimate(x, y, z, s["w"], box_size=box, n_bins=n, k_edges=s["edges"], mas=case["scheme"],
                                     shot_noise=s["shot"])
    if kind == "estimator":
        x, y, z = s["xyz"]
        e = s["estimator"]
        pk = e.run(x, y, z, s["w"])
        return e.k(), pk, e.out.nmodes, e.out.counts
    if kind == "assign":
        x, y, z = s["xyz"]
        f = mas.tsc_mas_vec if case["scheme"] == "TSC" else mas.cic_mas_vec
        return f(s["delta"], x, y, z, s["w"], case["particles"], 0.0, 0.0, 0.0, box, n, True)
    if kind == "powspec":
        if s["edges"] is None:
            return correlations.powspec_vec_fundamental(s["delta"], box, mas=case["scheme"])
        return correlations.powspec_vec(s["delta"], box, s["edges"], mas=case["scheme"])
    if kind == "xi":
        return correlations.xi_vec(s["delta"], box, s["edges"], mas=case["scheme"])
    if kind == "bispec":
        return correlations.bispec(s["delta"], box, *_legs(case), s["theta"], mas=case["scheme"])
    if kind == "grad":
        pos, w = s["pos"], s["w"]
        pos.grad = None
        if w is not None:
            w.grad = None
        _, pk, _ = autodiff.estimate_ad(pos, w, box_size=box, n_bins=n, k_edges=s["edges"], mas=case["scheme"])
        _loss(pk, s["target"]).backward()
        return (pk.detach(), pos.grad) if w is None else (pk.detach(), pos.grad, w.grad)
    if kind == "mock":
        pos, delta, psi = gauss_field.lognormal_mock(n, s["k"], s["pk"], box, case["particles"] / box ** 3, BIAS,
                                                     s["seed"], growth_rate=GROWTH if case["growth"] else 0.0,
                                                     return_fields=True)
        found = pos.shape[0]
        k, pk, nmodes = correlations.estimate(pos[:, 0], pos[:, 1], pos[:, 2], box_size=box, n_bins=n,
                                              k_edges=s["edges"], shot_noise=box ** 3 / found)
        return found, delta, psi, k, pk, nmodes
    return s["batch"].set(s["catalogues"]).run().results()


def _legs(case):
    """k1 = 0.1, k2 = 0.2, or the same ratio below the mesh's Nyquist wavenumber."""
    k1 = min(0.1, 0.2 * math.pi * case["n"] / case["box"])
    return k1, 2 * k1


def work(case):
    """Inputs read once, outputs written once; flops of the transforms, stencils and bins."""
    kind, n = case["kind"], case["n"]
    fft = 2.5 * n ** 3 * math.log2(n ** 3)
    if kind in ("powspec", "xi", "bispec"):
        transforms = {"powspec": 1, "xi": 2, "bispec": 4}[kind]
        return dict(bytes=4 * n ** 3, flops=transforms * fft + 15 * n ** 3)
    if kind == "mock":
        fields = 2 if case["growth"] else 1
        return dict(bytes=fields * 4 * n ** 3, flops=(fields + 1) * fft + 75 * n ** 3 + 100 * case["particles"])
    corners = 27 if case["scheme"] == "TSC" else 8
    record = 16 if case["weights"] else 12
    particles = case["particles"]
    if kind == "assign":
        return dict(bytes=16 * particles + 8 * n ** 3, flops=4 * corners * particles)
    if kind == "batch":
        total = sum(_jobs(case))
        return dict(bytes=record * total, flops=4 * 17 * total + case["jobs"] * (fft + 15 * n ** 3))
    if kind == "grad":
        return dict(bytes=2 * record * particles, flops=14 * corners * particles + 2 * fft + 30 * n ** 3)
    return dict(bytes=record * particles, flops=4 * corners * particles + fft + 15 * n ** 3)


# ------------------------------------------------------------------------------------
# the same results in 64 bits, with torch alone
# ------------------------------------------------------------------------------------
def _cells(pos, case):
    """Cell coordinates, float32 products as the estimators define them, then 64 bits."""
    inv = np.float32(1.0) / (np.float32(case["box"]) / np.float32(case["n"]))
    return (pos.detach() * float(inv)).double(), float(inv)


def _exact_mesh(p, w, n, scheme):
    """Mass assignment of cell coordinates p (N, 3): float64 (n, n, n), differentiable."""
    mesh = torch.zeros(n ** 3, device=DEVICE, dtype=torch.float64)
    if scheme == "TSC":
        base = torch.floor(p.detach() + 0.5)
        d = p - base
        f = [0.5 * (0.5 - d) ** 2, 0.75 - d * d, 0.5 * (0.5 + d) ** 2]
        offsets = (-1, 0, 1)
    else:
        base = torch.floor(p.detach())
        d = p - base
        f = [1.0 - d, d]
        offsets = (0, 1)
    base = base.long()
    r = range(len(offsets))
    for i in r:
        ix = (base[:, 0] + offsets[i]) % n
        for j in r:
            iy = (base[:, 1] + offsets[j]) % n
            for k in r:
                iz = (base[:, 2] + offsets[k]) % n
                # the reference stencil gives its (0, 1, 1) corner the y factor of row 0
                jy = 0 if scheme == "CIC_REF" and (i, j, k) == (0, 1, 1) else j
                wt = f[i][:, 0] * f[jy][:, 1] * f[k][:, 2]
                if w is not None:
                    wt = wt * w
                mesh = mesh.index_add(0, (ix * n + iy) * n + iz, wt) if wt.requires_grad else \
                    mesh.index_add_(0, (ix * n + iy) * n + iz, wt)
    return mesh.view(n, n, n)


def _wavenumbers(n):
    i = torch.arange(n, device=DEVICE)
    return torch.where(i > n // 2, i - n, i)


def _window(n, exponent):
    """(x / sin x)^exponent per axis, x = pi k / n."""
    x = math.pi * _wavenumbers(n).double() / n
    x[0] = 1e-9
    return (x / torch.sin(x)) ** exponent


def _exact_edges(case):
    e = _k_edges(case)
    if e is not None:
        return e * (case["box"] / (2 * math.pi))
    return np.arange(1, math.isqrt(3 * (case["n"] // 2) ** 2) + 2, dtype=np.float64)


def _slots(m, edges):
    """Bin of each squared radius m under numpy's histogram rule (last edge closed); -1 outside."""
    e = torch.as_tensor(edges, device=DEVICE, dtype=torch.float64)
    r = torch.sqrt(m.double())
    b = torch.bucketize(r, e, right=True) - 1
    b[r == e[-1]] = len(edges) - 2
    b[(b < 0) | (b >= len(edges) - 1)] = -1
    return b


def _legendre(k2, m):
    mu2 = k2.double() / m.clamp(min=1).double()
    return 1.0, 1.5 * mu2 - 0.5, (35.0 * mu2 * mu2 - 30.0 * mu2 + 3.0) / 8.0


def _planes(n, bytes_per_plane):
    step = max(1, int(2e8 / bytes_per_plane))
    return [(a, min(n, a + step)) for a in range(0, n, step)]


def _exact_multipoles(delta, case, edges, exponent, shot):
    """(k centres or means, P_l (nb, 3), counts) of a contrast mesh in 64 bits."""
    n, box = case["n"], case["box"]
    spec = torch.fft.rfftn(delta)
    ki = _wavenumbers(n)
    kz2 = torch.arange(n // 2 + 1, device=DEVICE) ** 2
    win = _window(n, 2 * exponent)
    nb = len(edges) - 1
    sums = torch.zeros((3, nb), device=DEVICE, dtype=torch.float64)
    counts = torch.zeros(nb, device=DEVICE, dtype=torch.float64)
    ksum = torch.zeros(nb, device=DEVICE, dtype=torch.float64)
    for a, b in _planes(n, 8 * n * (n // 2 + 1)):
        m = ki[a:b, None, None] ** 2 + ki[None, :, None] ** 2 + kz2[None, None, :]
        slot = _slots(m.reshape(-1), edges)
        keep = slot >= 0
        slot = slot[keep]
        power = spec[a:b].real ** 2 + spec[a:b].imag ** 2
        power = power * win[a:b, None, None] * win[None, :, None] * win[None, None, :n // 2 + 1]
        for l, leg in enumerate(_legendre(kz2[None, None, :], m)):
            if power.requires_grad:
                sums = sums.index_put((torch.full_like(slot, l), slot), (power * leg).reshape(-1)[keep], accumulate=True)
            else:
                sums[l] += torch.bincount(slot, weights=(power * leg).reshape(-1)[keep], minlength=nb)
        counts += torch.bincount(slot, minlength=nb)
        ksum += torch.bincount(slot, weights=torch.sqrt(m.double()).reshape(-1)[keep], minlength=nb)
    scale = torch.tensor([1.0, 5.0, 9.0], device=DEVICE, dtype=torch.float64) * (box / n ** 2) ** 3
    pk = (sums / counts).T * scale - torch.tensor([shot, 0.0, 0.0], device=DEVICE, dtype=torch.float64)
    kf = 2 * math.pi / box
    if _k_edges(case) is None:
        k = ksum / counts * kf
    else:
        k = torch.as_tensor(0.5 * (edges[1:] + edges[:-1]) * kf, device=DEVICE)
    return k, pk, counts


def _exact_estimate(pos, w, case, shot):
    p, _ = _cells(pos, case)
    rho = _exact_mesh(p, None if w is None else w.double(), case["n"], case["scheme"])
    exponent = 3 if case["scheme"] == "TSC" else 2
    return _exact_multipoles(rho / rho.mean() - 1.0, case, _exact_edges(case), exponent, shot)


def _exact_grad(s):
    case = s["case"]
    p, inv = _cells(s["pos"], case)
    p.requires_grad_()
    w = None if s["w"] is None else s["w"].detach().double().requires_grad_()
    rho = _exact_mesh(p, w, case["n"], case["scheme"])
    exponent = 3 if case["scheme"] == "TSC" else 2
    _, pk, _ = _exact_multipoles(rho / rho.mean() - 1.0, case, _exact_edges(case), exponent, 0.0)
    _loss(pk, _target(case, torch.float64)).backward()
    out = (pk.detach(), p.grad * inv)
    return out if w is None else out + (w.grad,)


def _exact_xi(s):
    case = s["case"]
    n, box = case["n"], case["box"]
    win = _window(n, 2 * {"CIC": 2, "NONE": 0}[case["scheme"]])
    spec = torch.fft.rfftn(s["delta"].double())
    power = (spec.real ** 2 + spec.imag ** 2) * win[:, None, None] * win[None, :, None] * win[None, None, :n // 2 + 1]
    del spec
    grid = torch.fft.irfftn(power.to(torch.complex128), s=(n, n, n))
    del power
    edges = s["edges"] * n / box
    nb = len(edges) - 1
    si = _wavenumbers(n)
    sums = torch.zeros((3, nb), device=DEVICE, dtype=torch.float64)
    counts = torch.zeros(nb, device=DEVICE, dtype=torch.float64)
    for a, b in _planes(n, 8 * n * n):
        m = si[a:b, None, None] ** 2 + si[None, :, None] ** 2 + si[None, None, :] ** 2
        slot = _slots(m.reshape(-1), edges)
        keep = slot >= 0
        slot = slot[keep]
        for l, leg in enumerate(_legendre(si[None, None, :] ** 2, m)):
            sums[l] += torch.bincount(slot, weights=(grid[a:b] * leg).reshape(-1)[keep], minlength=nb)
        counts += torch.bincount(slot, minlength=nb)
    scale = torch.tensor([1.0, 5.0, 9.0], device=DEVICE, dtype=torch.float64) / n ** 3
    xi = torch.where(counts > 0, sums / counts, torch.zeros_like(sums)).T * scale
    r = torch.as_tensor(0.5 * (edges[1:] + edges[:-1]) * (box / n), device=DEVICE)
    return r, xi, torch.where(counts > 0, counts, torch.full_like(counts, math.inf))


def _exact_bispec(s):
    case = s["case"]
    n, box = case["n"], case["box"]
    k1, k2 = _legs(case)
    th = s["theta"]
    kf = 2 * math.pi / box
    k_all = np.concatenate([[k1, k2], np.sqrt((k2 * np.sin(th)) ** 2 + (k2 * np.cos(th) + k1) ** 2)])
    win = _window(n, {"CIC": 2, "NONE": 0}[case["scheme"]])
    spec = torch.fft.rfftn(s["delta"].double())
    spec *= win[:, None, None] * win[None, :, None] * win[None, None, :n // 2 + 1]
    ki = _wavenumbers(n)
    r = torch.sqrt((ki[:, None, None] ** 2 + ki[None, :, None] ** 2 +
                    torch.arange(n // 2 + 1, device=DEVICE)[None, None, :] ** 2).double())
    field = []
    pk, bk, qk = [], [], []
    for i, k in enumerate(k_all):
        mask = (r >= (k - kf) / kf) & (r < (k + kf) / kf)
        d = torch.fft.irfftn(spec * mask, s=(n, n, n))
        one = torch.fft.irfftn(mask.to(torch.complex128), s=(n, n, n))
        pk.append(float((d * d).sum() / (one * one).sum()) * (box / n ** 2) ** 3)
        if i < 2:
            field.append((d, one))
            continue
        if i == 2:
            field = [(field[0][0] * field[1][0], field[0][1] * field[1][1])]
        b = float((field[0][0] * d).sum() / (field[0][1] * one).sum()) * (box ** 2 / n ** 3) ** 3
        bk.append(b)
        qk.append(b / (pk[0] * pk[1] + pk[0] * pk[-1] + pk[1] * pk[-1]))
    return tuple(torch.tensor(np.asarray(v), dtype=torch.float64) for v in (k_all, pk, th, bk, qk))


def exact(case, seed):
    kind = case["kind"]
    if kind == "mock":   # random draws of the generator's own streams
        return None
    if kind == "bispec" and case["n"] > 384:
        return None
    if kind == "batch":
        g = _generator(seed)
        out = []
        for i, particles in enumerate(_jobs(case)):
            pos, w = _catalogue(case, particles, g)
            out.append(_exact_estimate(pos, w, _batch_case(case, i), case["box"] ** 3 / particles))
        return out
    if kind in ("estimate", "estimator", "assign"):
        pos, w = _catalogue(case, case["particles"], _generator(seed))
        if kind == "assign":
            p, _ = _cells(pos, case)
            return _exact_mesh(p, None if w is None else w.double(), case["n"], case["scheme"])
        k, pk, counts = _exact_estimate(pos, w, case, case["box"] ** 3 / case["particles"])
        return (k, pk, counts) if kind == "estimate" else (k, pk, counts, None)
    s = prepare(case, seed)
    if kind == "grad":
        return _exact_grad(s)
    if kind == "xi":
        return _exact_xi(s)
    if kind == "bispec":
        return _exact_bispec(s)
    edges = _exact_edges(case)
    return _exact_multipoles(s["delta"].double(), case, edges, {"CIC": 2, "NONE": 0}[case["scheme"]], 0.0)
