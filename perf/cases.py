"""The work this library is used for, as cases that can be timed and compared.

A case is a dict of plain values; prepare() makes what a program holds before
the call (contexts with their particles in HBM, snapshot records, a net with
its training pairs), run() is one pass through the public entry points of
cola_halo_amd and returns what a program takes from it, work() the bytes and
operations the pass cannot do without, exact() the same outputs in 64 bits
from torch alone.

Kinds of case:
  state     one COLA step and the whole particle state (a checkpoint)
  steps     consecutive COLA steps of one realization (plain, or corrected by
            the committed net), then the density grid of the particles
  ensemble  the steps of several realizations together, then their grids
  ics       2LPT initial conditions of a seed, as the records of the initial
            output file
  snapshot  wrap, PM force and the snapshot records of an output time
  fof       friends-of-friends on the records of a snapshot
  grids     the density grid and the power spectrum of a snapshot
  train     Adam steps of the net on stored coarse/fine force pairs

The sizes are those of the configurations, tests and the benchmark: 32^3 to
512^3 particles, PM grids 1.5 to 3 times finer, mean spacing 1.56 to 1.95
Mpc/h.
"""
import math
import os

import numpy as np
import torch

import cola_halo_amd as ch

OM = 0.273
OMF = float(np.float32(OM))
NET = os.path.join(os.path.dirname(os.path.abspath(ch.__file__)), "nets", "eh98_cell1.30.net")
SPACING = 1.953125  # Mpc/h: 500 Mpc/h over 256 particles, 1000 over 512
LINK = 0.2
LAG = 0.05  # the velocities of a run are half a step behind the positions
NFOF_MIN = 32


def listed():
    return [
        # the smallest call: a step of one small member of an ensemble and the state it leaves, launch bound
        {"name": "state_32", "kind": "state", "nc": 32, "ng": 96, "box": 62.5, "a": 0.5},
        # the 64^3 / 192^3 configuration: the end of its run as replayed graphs, then its density field
        {"name": "steps_64_graph", "kind": "steps", "nc": 64, "ng": 192, "box": 100.0, "a": 0.5, "nsteps": 4,
         "grid": 64, "graph": True, "net": False},
        # a grid that is no power of two times three: factor 2.5, radices 3 and 5
        {"name": "steps_108_270", "kind": "steps", "nc": 108, "ng": 270, "box": 210.9375, "a": 0.4, "nsteps": 3,
         "grid": 54, "graph": False, "net": False},
        # the ordinary call: 256^3 particles on 768^3, mid-run
        {"name": "steps_256_768", "kind": "steps", "nc": 256, "ng": 768, "box": 500.0, "a": 0.4, "nsteps": 3,
         "grid": 128, "graph": False, "net": False},
        # the production comparison's fine run: the largest grid, 512^3 particles on 1536^3
        {"name": "steps_512_1536", "kind": "steps", "nc": 512, "ng": 1536, "box": 1000.0, "a": 0.1, "nsteps": 2,
         "grid": 128, "graph": False, "net": False},
        # the production comparison's corrected run: the headline of the benchmark
        {"name": "corrected_512_768", "kind": "steps", "nc": 512, "ng": 768, "box": 1000.0, "a": 0.1, "nsteps": 3,
         "grid": 128, "graph": False, "net": True},
        # realizations of uneven sizes stepped together, as mock catalogues are made
        {"name": "ensemble_96_128_160", "kind": "ensemble", "sizes": "96:288 128:384 160:480 96:288 128:384 160:480",
         "a": 0.4, "nsteps": 2, "grid": 64},
        # what every run starts with: 2LPT of a seed and the initial output's records
        {"name": "ics_128", "kind": "ics", "nc": 128, "ng": 192, "box": 250.0, "seed": 7},
        # what every run ends with: the force at the output time and the snapshot's records
        {"name": "snapshot_128_384", "kind": "snapshot", "nc": 128, "ng": 384, "box": 250.0, "a": 0.9},
        # the halo catalogue of the 256^3 configuration
        {"name": "fof_256", "kind": "fof", "nc": 256, "box": 500.0},
        # the density grid and the power spectrum of a 256^3 snapshot
        {"name": "grids_256", "kind": "grids", "nc": 256, "box": 500.0, "grid": 256, "pk": 512},
        # backward: Adam steps on force pairs of the training configuration (192^3 / 384^3)
        {"name": "train_192", "kind": "train", "nc": 128, "ng": 192, "box": 250.0, "pairs": 2, "epochs": 2},
    ]


def _smooth(n):
    for p in (2, 3, 5):
        while n % p == 0:
            n //= p
    return n == 1


def _size(rng, lo, hi, ratio, multiple=2):
    """(nc, ng) with even 2^a 3^b 5^c sizes, nc log-uniform in [lo, hi] and ng = ratio nc."""
    while True:
        nc = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / 2)) * 2
        ng = nc * ratio
        if lo <= nc <= hi and ng == int(ng) and int(ng) % multiple == 0 and _smooth(nc) and _smooth(int(ng)):
            return nc, int(ng)


def draw(rng):
    kind = rng.choice(["state", "steps", "steps", "steps", "corrected", "ensemble", "ics", "snapshot", "fof",
                       "grids", "train"])
    ratio = rng.choice([1.5, 2.0, 2.5, 3.0])
    a = rng.choice([0.3, 0.4, 0.5, 0.6, 0.7])
    if kind == "state":
        nc, ng = _size(rng, 24, 64, ratio)
        return {"kind": "state", "nc": nc, "ng": ng, "box": SPACING * nc, "a": a}
    if kind == "steps":
        nc, ng = _size(rng, 32, 256, ratio)
        return {"kind": "steps", "nc": nc, "ng": ng, "box": SPACING * nc, "a": a, "nsteps": rng.randint(1, 3),
                "grid": rng.choice([32, 50, 64, 96, 128]), "graph": rng.random() < 0.3, "net": False}
    if kind == "corrected":
        nc, ng = _size(rng, 64, 256, 1.5, multiple=32)
        return {"kind": "steps", "nc": nc, "ng": ng, "box": SPACING * nc, "a": a, "nsteps": rng.randint(1, 3),
                "grid": rng.choice([32, 50, 64]), "graph": False, "net": True}
    if kind == "ensemble":
        sizes = ["%d:%d" % _size(rng, 32, 128, rng.choice([1.5, 2.0, 3.0])) for _ in range(rng.randint(3, 8))]
        return {"kind": "ensemble", "sizes": " ".join(sizes), "a": a, "nsteps": rng.randint(1, 2), "grid": 32}
    if kind == "ics":
        nc, ng = _size(rng, 32, 160, 1.5)
        return {"kind": "ics", "nc": nc, "ng": ng, "box": SPACING * nc, "seed": rng.randint(1, 1000)}
    if kind == "snapshot":
        nc, ng = _size(rng, 32, 160, ratio)
        return {"kind": "snapshot", "nc": nc, "ng": ng, "box": SPACING * nc, "a": a}
    if kind == "fof":
        nc, _ = _size(rng, 32, 256, 1.0)
        return {"kind": "fof", "nc": nc, "box": SPACING * nc}
    if kind == "grids":
        nc, _ = _size(rng, 32, 256, 1.0)
        return {"kind": "grids", "nc": nc, "box": SPACING * nc, "grid": rng.choice([50, 64, 100, 128, 200, 256]),
                "pk": rng.choice([128, 180, 256, 300, 384, 512])}
    nc, ng = _size(rng, 32, 128, 1.5, multiple=32)
    return {"kind": "train", "nc": nc, "ng": ng, "box": SPACING * nc, "pairs": rng.randint(1, 3), "epochs": 2}


# ---- inputs: a second-order Lagrangian field of a cold-dark-matter spectrum, from the seed alone -------------------

def _wave(n, box, half):
    k = torch.fft.rfftfreq(n, 1.0 / n, device="cuda", dtype=torch.float64) if half else \
        torch.fft.fftfreq(n, 1.0 / n, device="cuda", dtype=torch.float64)
    return k * (2 * math.pi / box)


def _spectrum(k):
    """Bardeen et al. (1986) cold dark matter P(k) with shape 0.19 and sigma8 = 0.8; k in h/Mpc, a numpy array."""
    q = np.maximum(k, 1e-6) / 0.19
    t = np.log(1 + 2.34 * q) / (2.34 * q) * (1 + 3.89 * q + (16.1 * q) ** 2 + (5.46 * q) ** 3
                                             + (6.71 * q) ** 4) ** -0.25
    return k ** 0.96 * t * t


def _sigma8():
    k = np.exp(np.linspace(math.log(1e-4), math.log(30.0), 4000))
    x = 8.0 * k
    w = 3 * (np.sin(x) - x * np.cos(x)) / x ** 3
    f = _spectrum(k) * w * w * k ** 3 / (2 * math.pi ** 2)
    return math.sqrt(float(np.sum((f[1:] + f[:-1]) / 2) * (math.log(30.0) - math.log(1e-4)) / (len(k) - 1)))


def _field(n, box, seed):
    """Displacements (dx1, dx2) at a = 1 on the n^3 lattice, float64 [3, n, n, n] on the GPU."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed) * 7919 + 13)
    white = torch.randn((n, n, n), generator=gen, device="cuda", dtype=torch.float32).double()
    kx, ky, kz = _wave(n, box, False)[:, None, None], _wave(n, box, False)[None, :, None], _wave(n, box, True)
    k2 = kx * kx + ky * ky + kz * kz
    k2[0, 0, 0] = 1.0
    lk = np.linspace(math.log(1e-4), math.log(100.0), 8192)
    table = torch.from_numpy(np.sqrt(_spectrum(np.exp(lk))) * (0.8 / _sigma8())).cuda()
    at = ((0.5 * torch.log(k2) - lk[0]) / (lk[1] - lk[0])).clamp(0, len(lk) - 2)
    i = at.long()
    amp = table[i] + (table[i + 1] - table[i]) * (at - i)
    delta = torch.fft.rfftn(white) * amp * math.sqrt((n / box) ** 3)
    delta[0, 0, 0] = 0.0
    phi = delta / k2  # minus the potential
    ks = (kx, ky, kz)
    dx1 = torch.stack([torch.fft.irfftn(1j * k * phi, s=(n, n, n)) for k in ks])
    second = [[None] * 3 for _ in range(3)]
    for p in range(3):
        for q in range(p, 3):
            second[p][q] = torch.fft.irfftn(ks[p] * ks[q] * phi, s=(n, n, n))
    source = (second[0][0] * (second[1][1] + second[2][2]) + second[1][1] * second[2][2]
              - second[0][1] ** 2 - second[0][2] ** 2 - second[1][2] ** 2)
    phi2 = torch.fft.rfftn(source) / k2
    phi2[0, 0, 0] = 0.0
    dx2 = torch.stack([torch.fft.irfftn(-1j * k * phi2, s=(n, n, n)) for k in ks]) * (-3.0 / 7.0)
    return dx1, dx2


def _growth(a):
    """Linear growth of a flat universe, 1 at a = 1 (H times the integral of (aH)^-3)."""
    x, w = np.polynomial.legendre.leggauss(200)

    def g(b):
        s = 0.5 * b * (x + 1)
        return math.sqrt(OMF / b ** 3 + 1 - OMF) * float(np.sum(0.5 * b * w * (s / (OMF + (1 - OMF) * s ** 3)) ** 1.5))

    return g(a) / g(1.0)


def _growth2(a):
    def d(b):
        return _growth(b) ** 2 * (OMF / (OMF + (1 - OMF) * b ** 3)) ** (-1.0 / 143.0)

    return d(a) / d(1.0)


def _lattice(n, box):
    q = (torch.arange(n, device="cuda", dtype=torch.float64) + 0.5) * (box / n)
    return torch.stack(torch.meshgrid(q, q, q, indexing="ij"))


def _particles(nc, box, a, seed):
    """float32 [3, nc^3] tensors x, dx1, dx2, v of a state at scale factor a, positions inside the box."""
    dx1, dx2 = _field(nc, box, seed)
    x = (_lattice(nc, box) + _growth(a) * dx1 + _growth2(a) * dx2).reshape(3, -1)
    x = torch.remainder(x, box).float()
    x = torch.where(x >= np.float32(box), torch.zeros_like(x), x)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed) * 104729 + 1)
    v = 0.02 * torch.randn(x.shape, generator=gen, device="cuda")  # the residual velocity of the co-moving frame
    return x, dx1.reshape(3, -1).float(), dx2.reshape(3, -1).float(), v


def _context(nc, ng, box, a, seed):
    ctx = ch.Context(nc, ng, box)
    parts = np.zeros(nc ** 3, ch.PARTICLE_DTYPE)
    for name, t in zip(("x", "dx1", "dx2", "v"), _particles(nc, box, a, seed)):
        parts[name] = t.T.contiguous().cpu().numpy()
    parts["id"] = np.arange(1, nc ** 3 + 1)
    ctx.set_particles(parts, a, a - LAG)
    return ctx


def _halo_records(nc, box, seed):
    """float32 x, v [nc^3, 3] of a late snapshot: the displaced lattice, a sixth of it gathered into clumps."""
    dx1, dx2 = _field(nc, box, seed)
    n = nc ** 3
    x = (_lattice(nc, box) + dx1 + dx2).reshape(3, -1).T.contiguous()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed) * 15485863 + 5)
    v = 250.0 * dx1.reshape(3, -1).T / 4.0 + 100.0 * torch.randn((n, 3), generator=gen, device="cuda",
                                                               dtype=torch.float64)
    # clumps: the share of every clump falls with its size, as the halo mass function does
    want = n // 6
    size = (24.0 * torch.rand((max(8, n // 400),), generator=gen, device="cuda", dtype=torch.float64) ** -0.9).long()
    size = size.clamp(max=max(48, n // 200))
    ends = torch.cumsum(size, 0)
    ends = ends[ends <= want]
    if len(ends):
        nm = int(ends[-1])
        member = torch.randperm(n, generator=gen, device="cuda")[:nm]
        clump = torch.searchsorted(ends, torch.arange(nm, device="cuda"), right=True)
        centre = member[torch.cat([torch.zeros(1, device="cuda", dtype=torch.long), ends[:-1]])]
        radius = 0.07 * (box / nc) * size[:len(ends)].double() ** (1.0 / 3.0)
        off = torch.randn((nm, 3), generator=gen, device="cuda", dtype=torch.float64)
        x[member] = x[centre][clump] + radius[clump, None] * off
    x = torch.remainder(x, box).float()
    x = torch.where(x >= np.float32(box), torch.zeros_like(x), x)
    return x, v.float()


def _snapshot_context(nc, box, seed):
    ctx = ch.Context(nc, nc, box)
    x, v = _halo_records(nc, box, seed)
    rec = np.zeros(nc ** 3, ch.PARTICLE_MIN_DTYPE)
    rec["x"], rec["v"], rec["id"] = x.cpu().numpy(), v.cpu().numpy(), np.arange(1, nc ** 3 + 1)
    ctx.set_snapshot_records(rec)
    return ctx


def _sizes(case):
    return [tuple(int(v) for v in s.split(":")) for s in case["sizes"].split()]


def _kmax(case):
    """Just under the particles' Nyquist wave number, so that no mode lies on the edge of a shell."""
    return 0.9713579 * math.pi * case["nc"] / case["box"]


def _power(ctx):
    k, p = ch.eh98_table()
    ctx.power_init_table(k, p, 0.1, 0.8, OM, 1.0 - OM)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("state", "steps", "snapshot"):
        if case["nc"] > 256:  # the production sizes start from the library's own initial conditions
            ctx = ch.Context(case["nc"], case["ng"], case["box"])
            _power(ctx)
            ctx.lpt_set_displacement(case["a"], OM, 1 + seed % 100000)
            ctx.set_times(case["a"], case["a"])
        else:
            ctx = _context(case["nc"], case["ng"], case["box"], case["a"], seed)
        ctx.state_save()
        net = None
        if case.get("net"):
            net = ch.ResidualNet.from_file(case["ng"], NET)
            ctx.set_residual_net(net)
        if case.get("graph"):
            ctx.set_step_graph(True)
        ctx.synchronize()
        return {"case": case, "ctx": ctx, "net": net}
    if kind == "ensemble":
        ctxs = [_context(nc, ng, SPACING * nc, case["a"], seed * 16 + i) for i, (nc, ng) in enumerate(_sizes(case))]
        for c in ctxs:
            c.state_save()
            c.synchronize()
        return {"case": case, "ctxs": ctxs, "ens": ch.Ensemble(ctxs, graph=True)}
    if kind == "ics":
        ctx = ch.Context(case["nc"], case["ng"], case["box"])
        _power(ctx)
        return {"case": case, "ctx": ctx, "seed": case["seed"] + seed % 100000}
    if kind in ("fof", "grids"):
        state = {"case": case, "ctx": _snapshot_context(case["nc"], case["box"], seed)}
        if kind == "fof":  # the program's table of halos, as long as any catalogue can be
            state["halos"] = np.zeros(case["nc"] ** 3 // NFOF_MIN, ch.HALO_DTYPE)
        return state
    # train: pairs of the coarse and the fine force on the same particles, late and early
    nc, ng, box = case["nc"], case["ng"], case["box"]
    net = ch.ResidualNet.from_file(ng, NET)
    for i in range(case["pairs"]):
        a = (0.9, 0.5, 0.3)[i]
        with _context(nc, ng, box, a, seed * 4 + i) as coarse, ch.Context(nc, 2 * ng, box) as fine:
            fine.copy_particles_from(coarse)
            net.add_pair(coarse, fine)
    return {"case": case, "net": net}


def _schedule(case):
    """(a_vel, a_pos) of each step: tenths of the expansion, as every configuration steps."""
    a = case["a"]
    return [(a + (i + 0.5) * 0.1, a + (i + 1) * 0.1) for i in range(case["nsteps"])]


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "state":
        ctx = state["ctx"]
        ctx.state_restore()
        ctx.step(OMF, case["a"] + 0.05, case["a"] + 0.1)
        p = ctx.get_particles()
        return {"x": p["x"], "v": p["v"], "id": p["id"]}
    if kind == "steps":
        ctx = state["ctx"]
        ctx.state_restore()
        for a_vel, a_pos in _schedule(case):
            ctx.step(OMF, a_vel, a_pos)
        return ctx.coarse_grid(case["grid"], "particles")[0]
    if kind == "ensemble":
        for c in state["ctxs"]:
            c.state_restore()
        for a_vel, a_pos in _schedule(case):
            state["ens"].step(OMF, a_vel, a_pos)
        return [c.coarse_grid(case["grid"], "particles")[0] for c in state["ctxs"]]
    if kind == "ics":
        ctx = state["ctx"]
        ctx.lpt_set_displacement(0.1, OM, state["seed"])
        r = ctx.set_noncola_initial(OMF)
        return {"x": r["x"], "v": r["v"], "id": r["id"]}
    if kind == "snapshot":
        ctx = state["ctx"]
        ctx.state_restore()
        ctx.move_particles()
        ctx.pm_calculate_forces()
        r = ctx.set_snapshot(case["a"], OMF)
        return {"x": r["x"], "v": r["v"], "id": r["id"]}
    if kind == "fof":
        ctx = state["ctx"]
        h = ctx.fof_find_halos(float(np.float32(LINK * case["box"] / case["nc"])), NFOF_MIN)
        table = state["halos"]
        table[:len(h)] = h
        table[len(h):] = 0
        return {"nfof": table["nfof"], "x": table["x"], "v": table["v"], "labels": ctx.fof_labels()}
    if kind == "grids":
        ctx = state["ctx"]
        delta = ctx.coarse_grid(case["grid"])[0]
        k, p, modes = ctx.power_spectrum(case["pk"], 0.0, _kmax(case), 32, deconvolve=True, source="snapshot")
        return {"delta": delta, "k": k.astype(np.float32), "p": p.astype(np.float32), "modes": modes.astype(np.int64)}
    net = state["net"]
    losses = net.train(case["pairs"], case["epochs"], 2e-4, 1)
    return {"params": net.params(), "loss": losses.astype(np.float32)}


# ---- what a pass cannot do without ----------------------------------------------------------------------------------

def _step_work(nc, ng, net):
    """One PM step: x and v read and written, dx1 and dx2 read; the density and three force grids written once and
    read once; a real forward and three real inverse transforms; the net's products per cell."""
    return (72 * nc ** 3 + 32 * ng ** 3,
            4 * 2.5 * ng ** 3 * 3 * math.log2(ng) + (31968 * ng ** 3 if net else 0))


def work(case):
    kind = case["kind"]
    if kind == "state":
        b, f = _step_work(case["nc"], case["ng"], False)
        return {"bytes": b + 56 * case["nc"] ** 3, "flops": f}
    if kind == "steps":
        b, f = _step_work(case["nc"], case["ng"], case["net"])
        return {"bytes": case["nsteps"] * b + 12 * case["nc"] ** 3 + 4 * case["grid"] ** 3, "flops": case["nsteps"] * f}
    if kind == "ensemble":
        each = [_step_work(nc, ng, False) for nc, ng in _sizes(case)]
        out = sum(12 * nc ** 3 + 4 * case["grid"] ** 3 for nc, _ in _sizes(case))
        return {"bytes": case["nsteps"] * sum(b for b, _ in each) + out, "flops": case["nsteps"] * sum(f for _, f in each)}
    n = case["nc"] ** 3
    if kind == "ics":
        # three spectra of white noise, ten transforms of the lattice, the records
        return {"bytes": 12 * n * 2 + 48 * n + 32 * n, "flops": 13 * 2.5 * n * 3 * math.log2(case["nc"])}
    if kind == "snapshot":
        return {"bytes": 48 * n + 32 * case["ng"] ** 3 + 32 * n,
                "flops": 4 * 2.5 * case["ng"] ** 3 * 3 * math.log2(case["ng"])}
    if kind == "fof":
        return {"bytes": 32 * n + 4 * n, "flops": 27 * 8 * n}
    if kind == "grids":
        pk = case["pk"] ** 3
        return {"bytes": 2 * 12 * n + 4 * case["grid"] ** 3 + 2 * 4 * pk,
                "flops": 2.5 * pk * 3 * math.log2(case["pk"]) + 2 * 40 * n}
    # forward, data gradient and weight gradient: three times the forward's products; the pair's feature and target
    cells = case["ng"] ** 3 * case["pairs"] * case["epochs"]
    return {"bytes": 8 * cells, "flops": 3 * 31968 * cells}


# ---- the same outputs in 64 bits ------------------------------------------------------------------------------------

def _cic(x, n, box):
    """Cells (flat) and weights of the eight corners of positions x [3, np], periodic."""
    g = x * (n / box)
    i = torch.floor(g)
    d = g - i
    i = i.long()
    for c in range(8):
        bits = ((c >> 2) & 1, (c >> 1) & 1, c & 1)
        w = 1.0
        flat = 0
        for a in range(3):
            w = w * (d[a] if bits[a] else 1.0 - d[a])
            flat = flat * n + torch.remainder(i[a] + bits[a], n)
        yield flat, w


def _density(x, n, box):
    rho = torch.zeros(n ** 3, device="cuda", dtype=torch.float64)
    for flat, w in _cic(x, n, box):
        rho.index_add_(0, flat, w)
    return rho.reshape(n, n, n) * (n ** 3 / x.shape[1]) - 1.0


def _pm_force(x, n, box):
    dk = torch.fft.fftn(torch.fft.rfft(_density(x, n, box)), dim=(0, 1))
    full = torch.arange(n, device="cuda", dtype=torch.float64)
    full = torch.where(full > n // 2, full - n, full)
    ks = (full[:, None, None], full[None, :, None], torch.arange(n // 2 + 1, device="cuda", dtype=torch.float64))
    k2 = ks[0] ** 2 + ks[1] ** 2 + ks[2] ** 2
    k2[0, 0, 0] = 1.0
    dk = dk * (-1.0 / (2 * math.pi / box)) / k2
    dk[0, 0, 0] = 0.0
    out = torch.zeros_like(x)
    for a in range(3):
        f = torch.fft.ifftn(1j * ks[a] * dk, dim=(0, 1))
        f[:, :, 0] = f[:, :, 0].real.clone().to(f.dtype)
        f[:, :, n // 2] = f[:, :, n // 2].real.clone().to(f.dtype)
        grid = torch.fft.irfft(f, n=n).reshape(-1)
        for flat, w in _cic(x, n, box):
            out[a] += grid[flat] * w
    return out


def _q(a):
    return math.sqrt(OMF / a ** 3 + 1 - OMF) * a ** 3


N_LPT = -2.5


def _s_phi(ai, af, ref):
    return (af ** N_LPT - ai ** N_LPT) * ref / _q(ref) / (N_LPT * ref ** (N_LPT - 1))


def _s_q(ai, af, ref):
    x, w = np.polynomial.legendre.leggauss(64)
    s = 0.5 * (af - ai) * x + 0.5 * (af + ai)
    f = s ** N_LPT / np.sqrt(OMF / s ** 3 + 1 - OMF) / s ** 3
    return 0.5 * (af - ai) * float(np.sum(w * f)) / ref ** N_LPT


def _accel(f, dx1, dx2, a):
    g = _growth(a)
    om143 = (OMF / (OMF + (1 - OMF) * a ** 3)) ** (1.0 / 143.0)
    return -1.5 * OMF * (f + dx1 * g + dx2 * (g * g * (1.0 + 7.0 / 3.0 * om143)))


def _wrap(x, box):
    return torch.where(x < 0, x + box, torch.where(x >= box, x - box, x))


def _f32(v):
    return float(np.float32(v))


def _exact_steps(nc, ng, box, a, seed, schedule):
    x, dx1, dx2, v = (t.double() for t in _particles(nc, box, a, seed))
    a_x, a_v = _f32(a), _f32(a - LAG)
    for a_vel, a_pos in schedule:
        a_vel, a_pos = _f32(a_vel), _f32(a_pos)
        x = _wrap(x, box)
        v = v + _accel(_pm_force(x, ng, box), dx1, dx2, a_x) * _s_phi(a_v, a_vel, a_x)
        a_v = a_vel
        x = x + v * _s_q(a_x, a_pos, a_v) + dx1 * (_growth(a_pos) - _growth(a_x)) + dx2 * (_growth2(a_pos)
                                                                                       - _growth2(a_x))
        a_x = a_pos
    return x, v


def _exact_snapshot(case, seed):
    box = case["box"]
    x, dx1, dx2, v = (t.double() for t in _particles(case["nc"], box, case["a"], seed))
    x = _wrap(x, box)
    a = _f32(case["a"])
    # the output time is that of the positions: a kick to it, no drift, and the velocity's 2LPT part
    v = v + _accel(_pm_force(x, case["ng"], box), dx1, dx2, a) * _s_phi(_f32(case["a"] - LAG), a, a)
    nn = 6.0 * (1.0 - OMF) ** 1.5 / _growth_norm()
    dv = math.sqrt(OMF / a ** 3 + 1 - OMF) ** -1 * (nn - 3.0 * OMF * _growth(a) / (2.0 * a))
    dv2 = _q(a) * _growth2(a) / a * 2.0 * (OMF / (OMF + (1 - OMF) * a ** 3)) ** (6.0 / 11.0)
    return x.T, (100.0 / a * (v + dx1 * dv + dx2 * dv2)).T


def _growth_norm():
    """The growing mode at a = 1, normalised as 6 (1 - Om)^(3/2) H times the integral of (a / (Om + (1 - Om) a^3))^(3/2)."""
    x, w = np.polynomial.legendre.leggauss(200)
    s = 0.5 * (x + 1)
    integral = float(np.sum(0.5 * w * (s / (OMF + (1 - OMF) * s ** 3)) ** 1.5))
    return 6.0 * (1.0 - OMF) ** 1.5 * integral


def _exact_power(x, n, box, kmax, nbins):
    dk = torch.fft.rfftn(_density(x, n, box))
    full = torch.fft.fftfreq(n, 1.0 / n, device="cuda", dtype=torch.float64)
    ks = (full[:, None, None], full[None, :, None], torch.arange(n // 2 + 1, device="cuda", dtype=torch.float64))
    k = (2 * math.pi / box) * torch.sqrt(ks[0] ** 2 + ks[1] ** 2 + ks[2] ** 2)
    win = 1.0
    for a in range(3):
        win = win * torch.sinc(ks[a] / n) ** 2
    p = (dk.real ** 2 + dk.imag ** 2) * (box ** 3 / float(n) ** 6) / win ** 2
    wt = torch.full_like(k, 2.0)
    wt[:, :, 0] = 1.0
    wt[:, :, n // 2] = 1.0
    b = torch.floor(k / (kmax / nbins)).long()
    wt[0, 0, 0] = 0.0
    ok = (b < nbins) & (wt > 0)
    sums = [torch.zeros(nbins, device="cuda", dtype=torch.float64).index_add_(0, b[ok], q[ok])
            for q in (wt, wt * k, wt * p)]
    n_ = sums[0].clamp(min=1.0)
    return sums[1] / n_, sums[2] / n_


def exact(case, seed):
    kind = case["kind"]
    if kind == "state":
        x, v = _exact_steps(case["nc"], case["ng"], case["box"], case["a"], seed,
                            [(case["a"] + 0.05, case["a"] + 0.1)])
        return {"x": x.T, "v": v.T, "id": None}
    if kind == "steps":
        if case["net"] or case["nc"] > 256:  # bfloat16 layers; initial conditions of the library's own
            return None
        x, _ = _exact_steps(case["nc"], case["ng"], case["box"], case["a"], seed, _schedule(case))
        return _density(x, case["grid"], case["box"])
    if kind == "ensemble":
        out = []
        for i, (nc, ng) in enumerate(_sizes(case)):
            x, _ = _exact_steps(nc, ng, SPACING * nc, case["a"], seed * 16 + i, _schedule(case))
            out.append(_density(x, case["grid"], SPACING * nc))
        return out
    if kind == "snapshot":
        x, v = _exact_snapshot(case, seed)
        return {"x": x, "v": v, "id": None}
    if kind == "grids":
        x = _halo_records(case["nc"], case["box"], seed)[0].double().T.contiguous()
        delta = _density(x, case["grid"], case["box"])
        k, p = _exact_power(x, case["pk"], case["box"], _kmax(case), 32)
        return {"delta": delta, "k": k, "p": p, "modes": None}
    return None
