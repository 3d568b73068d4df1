"""The work that users of the TreePM step have it do, as cases that can be timed.

A user's program reads GOTPM particle records (or makes positions), uploads them to a box, and then
evolves the box, kicks it once, or measures something on it:

  evolve   records -> box, a number of whole steps (kdk_step), records back: a restart file taken to
           the next snapshot, and a request of the serving loop (36^3 to 192^3, 5 to 50 steps)
  kick     records -> box, one PM kick and one tree kick, velocities back: the two calls that the
           shim puts in the place of pmmain and treecorrection (the reference's own law and theta),
           or a force evaluation to full accuracy (theta -> 0)
  kick64   the same in the plain FP64 arithmetic, on FP64 arrays: the accuracy reference
  batch    an ensemble of independent boxes of several sizes, stepped together (batch_step)
  mesh     density and potential of a snapshot (tsc, psolver)
  pk       power spectrum of a snapshot (power_spectrum)
  prefof   halo candidates of a snapshot (prefof)

Particles are a Zel'dovich-perturbed lattice with a share of them in Plummer halos, as the
repository's benchmark has them (30 % or 40 % in halos of 32 to 1e5 particles), made on the GPU
from the seed. Steps are short against the halos' crossing times (da = 0.002 at a = 1), so that a
state after some steps still follows from the one before.
"""
import math
import weakref

import numpy as np
import torch

from lageunha_amd import lagpm

DEV = "cuda" if torch.cuda.is_available() else "cpu"
A_START, DA = 1.0, 0.002  # scale factor and step of the evolved boxes (amax = 48)
FACT2 = 1.0               # kick factor of single kicks
# mesh sizes with small prime factors, as the benchmark rounds them
SIZES = (32, 36, 40, 42, 48, 50, 54, 60, 64, 70, 72, 80, 84, 90, 96, 100, 108, 112, 120, 126, 128, 140, 144, 150, 160,
         162, 168, 180, 192)

_CTX = None


def context():
    global _CTX
    if _CTX is None:
        _CTX = lagpm.Context(0)
    return _CTX


# ---- the cases ----
def listed():
    return [
        # the smallest box of an ensemble: launches and latency count
        {"name": "evolve 32^3", "kind": "evolve", "n": 32, "np": 32768, "steps": 10, "halos": 0.3, "nleaf": 16, "group": 64, "mode": 0},
        # an ordinary small request of the serving loop
        {"name": "evolve 64^3", "kind": "evolve", "n": 64, "np": 262144, "steps": 20, "halos": 0.3, "nleaf": 16, "group": 64, "mode": 0},
        # a mesh that is no power of two, a particle number that is no cube, packed groups
        {"name": "evolve 100^3 ragged", "kind": "evolve", "n": 100, "np": 700001, "steps": 10, "halos": 0.4, "nleaf": 32, "group": 96, "mode": 2},
        # the default box of a mid-sized run
        {"name": "evolve 128^3", "kind": "evolve", "n": 128, "np": 2097152, "steps": 20, "halos": 0.3, "nleaf": 16, "group": 64, "mode": 0},
        # the benchmark's box with the tuning that its autotuner takes
        {"name": "evolve 256^3", "kind": "evolve", "n": 256, "np": 16777216, "steps": 20, "halos": 0.3, "nleaf": 32, "group": 64, "mode": 0},
        # the shim's two calls with the reference's law, split, cutoff and opening angle
        {"name": "reference kick 128^3", "kind": "kick", "n": 128, "np": 2097152, "law": lagpm.LAW_PMFIT, "theta": 0.3, "halos": 0.3},
        # forces without the tree's approximation, in FP32
        {"name": "kick 32^3 theta 0", "kind": "kick", "n": 32, "np": 32768, "law": lagpm.LAW_ERFC, "theta": 1e-6, "halos": 0.3},
        # the FP64 path at the opening angle of the runs
        {"name": "fp64 kick 64^3", "kind": "kick64", "n": 64, "np": 262144, "law": lagpm.LAW_ERFC, "theta": 0.5, "halos": 0.3},
        # an ensemble of boxes of 32^3 to 96^3
        {"name": "ensemble of 10", "kind": "batch", "nbox": 10, "nmin": 32, "nmax": 96, "steps": 10, "halos": 0.3},
        # density and potential of a snapshot
        {"name": "density, potential 160^3", "kind": "mesh", "n": 160, "np": 4096000, "halos": 0.3},
        # P(k) of a snapshot
        {"name": "power spectrum 192^3", "kind": "pk", "n": 192, "np": 7077888, "halos": 0.3},
        # halo candidates of a snapshot
        {"name": "prefof 128^3", "kind": "prefof", "n": 128, "np": 2097152, "halos": 0.3, "link": 0.2},
    ]


def draw(rng):
    def size(lo, hi):
        x = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        return min(SIZES, key=lambda s: abs(s - x))

    def count(n):  # a particle per cell, or another number (odd ones among them)
        return n ** 3 if rng.random() < 0.5 else rng.randrange(n ** 3 // 2, n ** 3)

    kind = rng.choice(["evolve", "evolve", "evolve", "kick", "kick64", "batch", "mesh", "pk", "prefof"])
    halos = rng.choice([0.0, 0.2, 0.3, 0.4])
    if kind == "evolve":
        n = size(32, 192)
        nleaf, group, mode = rng.choice([(16, 64, 0), (32, 64, 0), (16, 32, 0), (32, 64, 1), (32, 96, 2)])
        return {"kind": kind, "n": n, "np": count(n), "steps": rng.randrange(5, 26), "halos": halos, "nleaf": nleaf, "group": group,
                "mode": mode}
    if kind == "kick":
        if rng.random() < 0.3:
            n, theta = rng.choice([32, 36, 40]), 1e-6
        else:
            n, theta = size(32, 160), rng.choice([0.3, 0.5])
        return {"kind": kind, "n": n, "np": count(n), "law": rng.choice([lagpm.LAW_PMFIT, lagpm.LAW_ERFC, lagpm.LAW_TREEFORCE]),
                "theta": theta, "halos": halos}
    if kind == "kick64":
        n = size(32, 72)
        return {"kind": kind, "n": n, "np": count(n), "law": rng.choice([lagpm.LAW_PMFIT, lagpm.LAW_ERFC]),
                "theta": rng.choice([0.3, 0.5]), "halos": halos}
    if kind == "batch":
        return {"kind": kind, "nbox": rng.randrange(2, 11), "nmin": 32, "nmax": rng.choice([48, 64, 96]), "steps": rng.randrange(5, 16),
                "halos": halos}
    n = size(48, 192)
    if kind == "prefof":
        return {"kind": kind, "n": n, "np": count(n), "halos": halos, "link": rng.choice([0.15, 0.2, 0.25])}
    return {"kind": kind, "n": n, "np": count(n), "halos": halos}


# ---- inputs ----
def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) & 0x7FFFFFFF)


def particles(n, npart, halos, seed):
    """Positions (npart, 3) in [0, n) and velocities: a perturbed lattice and Plummer halos, FP64 on DEV."""
    g = _generator(seed)
    k = torch.fft.fftfreq(n, dtype=torch.float64, device=DEV) * (2 * math.pi)
    kx = torch.fft.rfftfreq(n, dtype=torch.float64, device=DEV) * (2 * math.pi)
    KZ, KY, KX = torch.meshgrid(k, k, kx, indexing="ij")
    k2 = KX ** 2 + KY ** 2 + KZ ** 2
    k2[0, 0, 0] = 1.0
    amp = k2 ** -0.25  # P(k) ~ 1/k
    amp[0, 0, 0] = 0.0
    delta = torch.fft.rfftn(torch.randn((n, n, n), generator=g, dtype=torch.float64, device=DEV)) * amp / k2
    psi = torch.stack([torch.fft.irfftn(1j * K * delta, s=(n, n, n)).reshape(-1) for K in (KX, KY, KZ)], dim=1)
    psi *= 0.3 / torch.sqrt((psi ** 2).sum(dim=1).mean())
    nh = int(round(halos * npart))
    site = torch.randperm(n ** 3, generator=g, device=DEV)[: npart - nh]
    lattice = torch.stack([site % n, (site // n) % n, site // (n * n)], dim=1).double()
    pos, vel = lattice + psi[site], psi[site] * (1.0 / (A_START * n))
    if nh:
        nhalo = max(1, nh // 2500)
        u = torch.rand(nhalo, generator=g, dtype=torch.float64, device=DEV)
        e = 1.0 - 1.9  # dN/dM ~ M^-1.9 from 32 to 1e5 particles
        m = (32.0 ** e + u * (1e5 ** e - 32.0 ** e)) ** (1.0 / e)
        which = torch.searchsorted(torch.cumsum(m / m.sum(), 0),
                                   torch.rand(nh, generator=g, dtype=torch.float64, device=DEV)).clamp_(max=nhalo - 1)
        centre = torch.rand((nhalo, 3), generator=g, dtype=torch.float64, device=DEV) * n
        w = torch.rand(nh, generator=g, dtype=torch.float64, device=DEV).clamp_(min=1e-12) * (1000.0 / 101.0 ** 1.5)
        r = 0.5 / torch.sqrt(w ** (-2.0 / 3.0) - 1.0)  # scale radius 0.5, cut at 10 of them
        d = torch.randn((nh, 3), generator=g, dtype=torch.float64, device=DEV)
        d /= torch.linalg.vector_norm(d, dim=1, keepdim=True)
        pos = torch.cat([pos, centre[which] + d * r[:, None]])
        vel = torch.cat([vel, 0.02 / n * torch.randn((nh, 3), generator=g, dtype=torch.float64, device=DEV)])
    pos = torch.remainder(pos, n)
    pos[pos >= n] = 0.0
    order = torch.randperm(npart, generator=g, device=DEV)
    return pos[order], vel[order], g


def records(n, npart, halos, seed, still=False):
    """The particles as GOTPM records: a lattice site some cells away and the displacement from it."""
    pos, vel, g = particles(n, npart, halos, seed)
    site = torch.round(pos + 2.0 * torch.randn(pos.shape, generator=g, dtype=torch.float64, device=DEV))
    disp = (pos - site).float().cpu().numpy()
    s = torch.remainder(site, n).long()
    rec = np.empty(npart, dtype=lagpm.DM_RECORD)
    rec["u4if"] = (s[:, 0] + n * (s[:, 1] + n * s[:, 2])).cpu().numpy().astype(np.uint64)
    v = (0.0 if still else 1.0) * vel.float().cpu().numpy()
    for a, name in enumerate("xyz"):
        rec[name] = disp[:, a]
        rec["v" + name] = v[:, a]
    return rec


def unpack(rec, n):
    """Positions (FP64) that the records stand for: XofP = fmod(dx + i + nx, nx)."""
    idx = rec["u4if"].astype(np.int64)
    site = (idx % n, (idx // n) % n, idx // (n * n))
    return np.stack([np.fmod(rec[a].astype(np.float64) + site[c] + n, float(n)) for c, a in enumerate("xyz")], axis=1)


def params_of(case, n=None, npart=None, precision=lagpm.PREC_FP32):
    n, npart = n or case["n"], npart or case["np"]
    mass = n ** 3 / npart  # mean density of one per cell
    law = case.get("law", lagpm.LAW_ERFC)
    if law == lagpm.LAW_ERFC:
        return lagpm.make_params(n, mass=mass, theta=case.get("theta", 0.5), precision=precision)
    p = lagpm.reference_params(n, mass=mass, theta=case["theta"], precision=precision)
    p.law = law
    return p


class State:
    """A prepared case: its boxes are closed when it goes."""

    def __init__(self, case, boxes, **data):
        self.case, self.boxes = case, boxes
        self.__dict__.update(data)
        self._end = weakref.finalize(self, _close, list(boxes))


def _close(boxes):
    for b in boxes:
        b.close()


def _ensemble(case, seed):
    """(n, np) of the boxes of an ensemble: sizes evenly in log n."""
    r = np.random.default_rng(seed)
    ns = np.exp(np.linspace(math.log(case["nmin"]), math.log(case["nmax"]), case["nbox"]))
    ns = [min(SIZES, key=lambda s: abs(s - x)) for x in ns]
    r.shuffle(ns)
    return ns


def prepare(case, seed):
    ctx, kind = context(), case["kind"]
    if kind == "batch":
        ns = _ensemble(case, 7)
        recs = [records(n, n ** 3, case["halos"], 64 * seed + i) for i, n in enumerate(ns)]
        boxes = [lagpm.Box(ctx, params_of(case, n, n ** 3), n ** 3) for n in ns]
        return State(case, boxes, rec=recs, out=[r.copy() for r in recs])
    n, npart = case["n"], case["np"]
    precision = lagpm.PREC_FP64 if kind == "kick64" else lagpm.PREC_FP32
    box = lagpm.Box(ctx, params_of(case, precision=precision), npart)
    if kind == "kick64":
        pos, vel, _ = particles(n, npart, case["halos"], seed)
        return State(case, [box], xyz=[np.ascontiguousarray(a) for a in pos.cpu().numpy().T])
    if kind == "evolve":
        box.set_tuning(case["nleaf"], case["group"], case["mode"])
    rec = records(n, npart, case["halos"], seed, still=kind == "kick")
    return State(case, [box], rec=rec, out=rec.copy())


# ---- one pass ----
def _fields(out, names):
    return {k: out[k] for k in names}


def run(state):
    case, kind = state.case, state.case["kind"]
    if kind == "batch":
        for b, r in zip(state.boxes, state.rec):
            b.upload_eunha(r)
        for s in range(case["steps"]):
            lagpm.batch_step(context(), state.boxes, A_START + DA * s, DA)
        for b, o in zip(state.boxes, state.out):
            b.download_eunha(o)
        return [_fields(o, ("x", "y", "z", "vx", "vy", "vz")) for o in state.out]
    box = state.boxes[0]
    if kind == "kick64":
        box.upload(*state.xyz)
        box.pmmain(lagpm.evolfact(FACT2), lagpm.KICK)
        box.treecorrection(lagpm.evolfact(FACT2))
        return box.velocities()
    box.upload_eunha(state.rec)
    if kind == "evolve":
        for s in range(case["steps"]):
            box.kdk_step(A_START + DA * s, DA)
        box.download_eunha(state.out)
        return _fields(state.out, ("x", "y", "z", "vx", "vy", "vz"))
    if kind == "kick":
        box.pmmain(lagpm.evolfact(FACT2), lagpm.KICK)
        box.treecorrection(lagpm.evolfact(FACT2))
        box.download_eunha_vel(state.out)
        return _fields(state.out, ("vx", "vy", "vz"))
    if kind == "mesh":
        den = box.tsc()
        return {"density": den, "potential": box.psolver()}
    if kind == "pk":
        pk, npk, cor, sigma8, slope = box.power_spectrum(256.0)
        return {"pk": pk, "npk": npk, "cor": cor, "sigma8": sigma8, "slope": slope}
    flags, count = box.prefof(case["link"])
    return {"flags": flags, "count": count}


# ---- what a pass cannot do without ----
def work(case):
    """Bytes: the caller's particles in and results out, and each phase's own arrays once (positions and
    velocities read and written per step in FP64, the mesh written and read by the deposit, the two
    transforms, the gradient and the interpolation). Flops: the transforms (2.5 m log2 m each for m
    real values) and the pair terms (21 per pair) of the particles within the cutoff at mean
    density; with the tree about half of them are left."""
    if case["kind"] == "batch":
        one = [work({"kind": "evolve", "n": n, "np": n ** 3, "steps": case["steps"]}) for n in _ensemble(case, 7)]
        return {k: sum(o[k] for o in one) for k in ("bytes", "flops")}
    n, npart, kind = case["n"], case["np"], case["kind"]
    m, real = n ** 3, 8 if kind == "kick64" else 4
    fft = 2.5 * m * math.log2(m)
    rc = 5.625 if case.get("law", lagpm.LAW_ERFC) == lagpm.LAW_ERFC else 4.0
    pairs = 21.0 * 4.19 * rc ** 3 * npart / m * (1.0 if case.get("theta", 0.5) < 0.01 else 0.5)
    pm_bytes = 24 * npart + 8 * real * m + 72 * npart  # deposit, transforms and gradient, kick
    if kind == "evolve":
        return {"bytes": 64 * npart + case["steps"] * (pm_bytes + 96 * npart), "flops": case["steps"] * (2 * fft + pairs * npart)}
    if kind == "kick":
        return {"bytes": 44 * npart + pm_bytes + 72 * npart, "flops": 2 * fft + pairs * npart}
    if kind == "kick64":
        return {"bytes": 48 * npart + pm_bytes + 72 * npart, "flops": 2 * fft + pairs * npart}
    if kind == "mesh":
        return {"bytes": 32 * npart + 24 * npart + 6 * real * m, "flops": 2 * fft + 100 * npart}
    if kind == "pk":
        return {"bytes": 32 * npart + 24 * npart + 4 * real * m, "flops": fft + 100 * npart + 10 * m}
    return {"bytes": 32 * npart + 24 * npart + npart, "flops": 10 * 27 * npart}


# ---- the same in 64 bits, in plain torch ----
def _tsc(x):
    near = torch.round(x)
    d = x - near
    s = torch.where(torch.signbit(d), -1, 1).long()
    a = d.abs()
    w3 = 0.5 * (0.25 + a * (a - 1.0))
    return near.long(), s, (0.75 - a * a, w3 + a, w3)


def _cells(pos, n):
    """The 27 (flat cell, weight) pairs of each particle."""
    ax = [_tsc(pos[:, c]) for c in range(3)]
    for c in range(3):
        for b in range(3):
            for a in range(3):
                i, j, k = (torch.remainder(ax[d][0] + ax[d][1] * (0, 1, -1)[q], n) for d, q in enumerate((a, b, c)))
                yield i + n * (j + n * k), ax[0][2][a] * ax[1][2][b] * ax[2][2][c]


def _density(pos, n, mass):
    den = torch.zeros(n ** 3, dtype=torch.float64, device=pos.device)
    for cell, w in _cells(pos, n):
        den.index_add_(0, cell, w * mass)
    return den - 1.0


def _waves(n, device):
    k = torch.arange(n, dtype=torch.float64, device=device)
    k = torch.where(k > n / 2, k - n, k)
    KZ, KY, KX = torch.meshgrid(k, k, torch.arange(n // 2 + 1, dtype=torch.float64, device=device), indexing="ij")
    return KX, KY, KZ


def _window(k, n):
    h = math.pi * k / n
    return torch.where(k == 0, torch.ones_like(h), torch.sin(h) / torch.where(k == 0, torch.ones_like(h), h)) ** 3


def _potential(den, n, efold, deconvolve):
    KX, KY, KZ = _waves(n, den.device)
    k2 = KX ** 2 + KY ** 2 + KZ ** 2
    k2[0, 0, 0] = 1.0
    f = -1.0 / (math.pi * k2) * torch.exp(-k2 * (math.pi * efold / n) ** 2)
    if deconvolve:
        f = f / (_window(KX, n) * _window(KY, n) * _window(KZ, n)) ** 2
    f[0, 0, 0] = 0.0
    return torch.fft.irfftn(torch.fft.rfftn(den.reshape(n, n, n)) * f, s=(n, n, n))  # 1/n^3 is in the inverse


def _pm(pos, n, p):
    phi = _potential(_density(pos, n, p.mass), n, p.efold, p.deconvolve)
    acc = torch.zeros_like(pos)
    for a, dim in enumerate((2, 1, 0)):
        g = (2.0 / 3.0) * (torch.roll(phi, 1, dim) - torch.roll(phi, -1, dim)) - (torch.roll(phi, 2, dim) - torch.roll(phi, -2, dim)) / 12.0
        g = g.reshape(-1)
        for cell, w in _cells(pos, n):
            acc[:, a] += w * g[cell]
    return acc


def _law(p, s):
    """Short-range force over distance at squared distance s, for n = 1."""
    r = torch.sqrt(s)
    if p.law == lagpm.LAW_ERFC:
        rs = 0.5 * p.efold
        u = r / (2.0 * rs)
        small = (4.0 / (3.0 * math.sqrt(math.pi))) / (8.0 * rs ** 3) * (1.0 - 0.6 * u * u + (3.0 / 14.0) * u ** 4)
        far = (torch.erf(u) - r / (rs * math.sqrt(math.pi)) * torch.exp(-u * u)) / (s * r)
        return (s + p.epsilon ** 2) ** -1.5 - torch.where(u * u < 1e-6, small, far)
    a = (1.0 / 65536.0, 0.78224, 0.37971e-06, -0.60338, -0.34419e-07, -3.9741, -1.0607, -0.38145)
    eps = p.epsilon if p.law == lagpm.LAW_PMFIT else 0.1
    r = r.clamp(min=6.0 / 4096.0)  # the reference's table starts at its first entry
    s = r * r
    fit = (torch.tanh(a[1] * r) / s - a[1] / (torch.cosh(a[1] * r) ** 2 * r) - 2.0 * a[2] / a[0] * r * torch.exp(a[3] * s)
           - 2.0 * a[2] * a[3] / a[0] * r * s * torch.exp(a[3] * s) + a[4] / a[0] * (1.0 + a[5] * s + a[6] * s * s) * torch.exp(a[7] * s))
    return (s + eps * eps) ** -1.5 - fit / r


def _pairs(pos, n, p):
    acc = torch.empty_like(pos)
    for b in range(0, len(pos), 512):
        d = pos[b:b + 512, None, :] - pos[None, :, :]
        d -= n * torch.round(d / n)
        s = (d * d).sum(dim=2)
        f = torch.where((s <= p.rsphere ** 2) & (s > 0), -_law(p, torch.where(s > 0, s, torch.ones_like(s))), torch.zeros_like(s))
        acc[b:b + 512] = (d * f[:, :, None]).sum(dim=1)
    return acc * (p.mass / n ** 2)


def _power(pos, n, mass, boxsize):
    spec = torch.fft.rfftn(_density(pos, n, mass).reshape(n, n, n))[:, :, : n // 2]
    KX, KY, KZ = (k[:, :, : n // 2] for k in _waves(n, pos.device))
    w = _window(KX, n) * _window(KY, n) * _window(KZ, n)
    d = ((spec.real ** 2 + spec.imag ** 2) / float(n) ** 6 / w ** 2).reshape(-1)
    k = torch.sqrt(KX ** 2 + KY ** 2 + KZ ** 2).reshape(-1)
    lo = torch.floor(k)
    t = k - lo
    pk, npk = (torch.zeros(2 * n, dtype=torch.float64, device=pos.device) for _ in range(2))
    for b, x in ((lo.long(), 1.0 - t), (lo.long() + 1, t)):
        pk.index_add_(0, b, x * d)
        npk.index_add_(0, b, x)
    pk, npk = pk[: n + 1].cpu().numpy(), npk[: n + 1].cpu().numpy()
    pk = np.where(npk > 0, pk / np.where(npk > 0, npk, 1.0), 0.0)
    i = np.arange(1, n + 1)
    x = 2 * math.pi * (8.0 / boxsize * n) / n * i
    sigma8 = math.sqrt(36 * math.pi * float(np.sum(pk[1:] * i ** 2.0 * (np.sin(x) - x * np.cos(x)) ** 2 / x ** 6)))
    cor = np.zeros(n + 1)
    cor[1:] = 2.0 * n / i * (np.sin(np.outer(i, i) * (2 * math.pi / n)) @ (i * pk[1:]))
    slope = (math.log(cor[3]) - math.log(cor[2])) / (math.log(4.0) - math.log(3.0)) if cor[2] > 0 and cor[3] > 0 else 0.0
    return {"pk": pk, "npk": npk, "cor": cor, "sigma8": sigma8, "slope": slope}


def exact(case, seed):
    kind = case["kind"]
    if kind not in ("kick", "mesh", "pk") or (kind == "kick" and case["theta"] > 0.01):
        return None
    n, p = case["n"], params_of(case)
    rec = records(n, case["np"], case["halos"], seed, still=True)
    pos = torch.from_numpy(unpack(rec, n)).to(DEV)
    if kind == "kick":
        v = (FACT2 * (_pm(pos, n, p) + _pairs(pos, n, p))).cpu().numpy()
        return {"vx": v[:, 0], "vy": v[:, 1], "vz": v[:, 2]}
    if kind == "mesh":
        den = _density(pos, n, p.mass)
        phi = _potential(den, n, p.efold, p.deconvolve)
        return {"density": den.reshape(n, n, n).cpu().numpy(), "potential": phi.reshape(-1).cpu().numpy()}
    return _power(pos, n, p.mass, 256.0)
