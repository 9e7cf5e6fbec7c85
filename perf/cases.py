"""Workloads by which the engine's speed is followed, each one pass through the public
entry points as a user's program makes it.

A case is a dict of plain values; its "kind" says which pass it is:

  steps     a small box stepped by hgpm_step from a state kept in a second context (a
            checkpoint on the device), its particles read back: parameter scans, tests;
  host      a box whose particles the caller keeps on the host: handed over, one step in
            the reference's single calls (UpdatePositions, CIC, SolveGradient,
            UpdateVelocities, UpdatePositions), taken back;
  run       a run from a parameter file: initial conditions, steps, P(k);
  late      the last steps of a run, resumed from a clustered checkpoint, and P(k);
  pk        P(k) of an evolved box at every fold, as a P(k) dump writes it;
  force     the force grid of a particle set, for a caller with an integrator of its own;
  fft       the 3-D transform of a grid the caller keeps on the device;
  f64       steps of the FP64 path, the accuracy reference of a run;
  ensemble  boxes of several sizes with seeds of their own: initial conditions, the
            steps as one graph run, P(k) of each.

`exact` restates each pass in 64 bits with plain torch.  Particles are placed and moved
with closed forms of a flat universe, so that both sides of a comparison start from the
same numbers.
"""
import ctypes
import functools
import math

import numpy as np
import torch

import hacc_gpm_amd as hg

SIZES = (32, 64, 96, 128, 192, 256, 384, 512, 768, 1024)  # transform lengths of the engine
CELL = 2.0     # Mpc/h per grid cell
OM = 0.31      # matter density of hg.make_params' defaults
Z0 = 50.0      # first redshift of a run ...
NSTEPS = 50    # ... and its steps to z = 0


def listed():
    return [
        # the smallest boxes: a step is a few dozen launches over almost no data
        {"name": "steps_32", "kind": "steps", "np": 32, "ng": 32, "steps": 6, "disp": 0.08},
        # a radix-3 length, and particles of mass 8 on a finer grid
        {"name": "steps_96_on_192", "kind": "steps", "np": 96, "ng": 192, "steps": 4, "disp": 0.05},
        # a host program that owns the particles and calls the reference's functions
        {"name": "host_128", "kind": "host", "np": 128, "ng": 128, "disp": 0.08},
        # an ordinary run of the driver: NG 256, P(k) with the parameter file's default bins
        {"name": "run_256", "kind": "run", "np": 256, "ng": 256, "steps": 10, "bins": 221},
        # fewer particles than cells, the large class of the memory-pressure workload
        {"name": "run_384_on_768", "kind": "run", "np": 384, "ng": 768, "steps": 4, "bins": 64},
        # the benchmark's box
        {"name": "run_1024", "kind": "run", "np": 1024, "ng": 1024, "steps": 8, "bins": 32},
        # clustered tiles: the end of a run, where the particle kernels are slowest
        {"name": "late_512", "kind": "late", "np": 512, "ng": 512, "steps": 4, "bins": 32},
        # a P(k) dump with folds
        {"name": "pk_256", "kind": "pk", "np": 256, "ng": 256, "bins": 221, "folds": 2, "disp": 3.0},
        {"name": "force_96", "kind": "force", "np": 96, "ng": 96, "disp": 0.5},
        {"name": "fft_384", "kind": "fft", "ng": 384, "dir": -1, "f64": False},
        {"name": "f64_128", "kind": "f64", "np": 128, "ng": 128, "steps": 2, "disp": 0.08},
        # the ensemble workload's classes, fewer boxes of each
        {"name": "ensemble_24", "kind": "ensemble", "small": 64, "large": 192, "per": 8, "steps": 8, "bins": 32},
    ]


def draw(rng):
    kind = rng.choice(("steps", "steps", "host", "run", "run", "late", "pk", "force", "fft", "f64", "ensemble"))
    pick = lambda lo, hi: rng.choice([n for n in SIZES if lo <= n <= hi])  # noqa: E731
    if kind in ("steps", "host", "force"):
        ng = pick(32, 192)
        c = {"kind": kind, "np": pick(max(32, ng // 3), ng), "ng": ng, "disp": round(rng.uniform(0.02, 0.1), 4)}
        return dict(c, steps=rng.randint(1, 16)) if kind == "steps" else c
    if kind == "run":
        ng = pick(96, 768)
        return {"kind": kind, "np": rng.choice([n for n in SIZES if n in (ng, ng // 2)]), "ng": ng,
                "steps": rng.randint(2, 12), "bins": rng.randint(16, 221)}
    if kind == "late":
        n = pick(128, 512)
        return {"kind": kind, "np": n, "ng": n, "steps": rng.randint(2, 5), "bins": rng.randint(16, 221)}
    if kind == "pk":
        ng = pick(64, 384)
        return {"kind": kind, "np": rng.choice([n for n in SIZES if n in (ng, ng // 2)]), "ng": ng,
                "bins": rng.randint(16, 221), "folds": rng.randint(0, 3), "disp": round(rng.uniform(0.5, 4.0), 3)}
    if kind == "fft":
        f64 = rng.random() < 0.4
        return {"kind": kind, "ng": pick(32, 384 if f64 else 768), "dir": rng.choice((-1, 1)), "f64": f64}
    if kind == "f64":
        n = pick(32, 256)
        return {"kind": kind, "np": n, "ng": n, "steps": rng.randint(1, 4), "disp": round(rng.uniform(0.02, 0.1), 4)}
    small = rng.choice((32, 64, 96))
    return {"kind": kind, "small": small, "large": rng.choice((96, 128, 192)) if small < 96 else 128,
            "per": rng.randint(2, 10), "steps": rng.randint(2, 12), "bins": rng.randint(16, 64)}


# ------------------------------------------------------- closed forms of a run ----
def adot(a):
    return math.sqrt(OM / a + (1.0 - OM) * a * a)


def schedule(first, n):
    """(drift0, kick_dt, kick_fscal, drift1, skip_drift0) of steps first .. first + n - 1 of
    a run from Z0 to 0 in NSTEPS steps of equal length in a, the half drifts between
    steps merged (prefactors rounded to float, as UpdatePositions takes them)."""
    a0 = 1.0 / (1.0 + Z0)
    da = (1.0 - a0) / NSTEPS
    half = lambda a: float(np.float32(0.5 * da / (a * a * adot(a))))  # noqa: E731
    out = []
    for s in range(first, first + n):
        a = a0 + s * da
        m = a + 0.5 * da
        last = s == first + n - 1
        out.append((half(a) if s == first else 0.0, da, 1.5 * OM / (m * adot(m)),
                    half(a + da) * (1.0 if last else 2.0), s != first))
    return out


def coeffs(first, n):
    out = []
    for d0, dt, fs, d1, skip in schedule(first, n):
        c = hg.StepCoeffs()
        c.drift0, c.kick_dt, c.kick_fscal, c.drift1, c.skip_drift0 = d0, dt, fs, d1, 1 if skip else 0
        out.append(c)
    return out


def shape(k):
    """A cold-dark-matter spectrum (Bardeen et al. 1986, eq. G3; Gamma 0.21), unnormalised;
    k in h/Mpc."""
    q = k / 0.21
    t = np.log1p(2.34 * q) / (2.34 * q) / (1 + 3.89 * q + (16.1 * q) ** 2 + (5.46 * q) ** 3 + (6.71 * q) ** 4) ** 0.25
    return k * t * t


@functools.lru_cache(maxsize=None)
def table():
    """The .ipk numbers of a run: header (k_max and the bin width where the reader puts
    them) and P(k) at Z0, sigma_8 = 0.81 today and growth proportional to a."""
    dk, n = 0.0005, 20001
    k = dk * np.arange(n)
    p = np.zeros(n)
    p[1:] = shape(k[1:])
    x = 8.0 * k[1:]
    w = 3.0 * (np.sin(x) - x * np.cos(x)) / x ** 3
    p *= 0.81 ** 2 / float(np.sum(p[1:] * w * w * k[1:] ** 2) * dk / (2 * math.pi ** 2)) / (1.0 + Z0) ** 2
    hdr = np.zeros(20)
    hdr[1], hdr[3] = k[-1], dk
    return hdr, p


def ic_numbers():
    """(delta, dot_delta, fscal, deltaT) of the initial conditions: growth D = a, the
    velocities half a step before the positions."""
    a0 = 1.0 / (1.0 + Z0)
    da = (1.0 - a0) / NSTEPS
    h = a0 - 0.5 * da
    return a0, 1.0, 1.5 * OM / (h * adot(h)), da


def placed(case, seed):
    """Positions (grid units) and velocities of a cell-centred lattice of np^3 points
    displaced by a Gaussian field with the spectrum above to an RMS of `disp` cells per
    axis, moving in the growing mode: float32 host arrays in the reference's order."""
    n, ng = case["np"], case["ng"]
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    d = torch.fft.rfftn(torch.randn((n, n, n), generator=g, device="cuda", dtype=torch.float64))
    m = torch.fft.fftfreq(n, 1.0 / n, device="cuda", dtype=torch.float64)
    mz = torch.arange(n // 2 + 1, device="cuda", dtype=torch.float64)
    k2 = m[:, None, None] ** 2 + m[None, :, None] ** 2 + mz[None, None, :] ** 2
    k2[0, 0, 0] = 1.0
    kk = 2 * math.pi / (CELL * ng) * torch.sqrt(k2)
    q = kk / 0.21
    t = torch.log1p(2.34 * q) / (2.34 * q) / (1 + 3.89 * q + (16.1 * q) ** 2 + (5.46 * q) ** 3 + (6.71 * q) ** 4) ** 0.25
    d *= torch.sqrt(kk) * t / k2
    d[0, 0, 0] = 0.0
    psi = []
    for a, ka in enumerate((m[:, None, None], m[None, :, None], mz[None, None, :])):
        ka = torch.where(ka.abs() == n // 2, torch.zeros_like(ka), ka)
        psi.append(torch.fft.irfftn(1j * ka * d, s=(n, n, n)))
    psi = torch.stack(psi, dim=-1)
    psi *= case["disp"] / torch.sqrt((psi ** 2).mean())
    i = (torch.arange(n, device="cuda", dtype=torch.float64) + 0.5) * (ng / n)
    x = torch.stack(torch.meshgrid(i, i, i, indexing="ij"), dim=-1) + psi
    a0 = 1.0 / (1.0 + Z0)
    h = a0 - 0.5 * (1.0 - a0) / NSTEPS
    v = psi / a0 * (h * h * adot(h))
    return (torch.remainder(x, float(ng)).reshape(-1, 3).float().cpu().numpy(), v.reshape(-1, 3).float().cpu().numpy())


def params(case, seed, prec=hg.FP32, n=None):
    np_, ng = n or case["np"], n or case["ng"]
    return hg.make_params(ng, np_, CELL * ng, Z0, 0.0, NSTEPS, seed=int(seed) % 2147483647, precision=prec,
                          pk_bins=case.get("bins", 32), pk_folds=case.get("folds", 0))


def box_seeds(case, seed):
    return [(int(seed) * 131 + b) % 2147483647 for b in range(len(box_sizes(case)))]


def box_sizes(case):
    return [n for n in (case["small"], 128 if case["large"] != 128 else 96, case["large"]) for _ in range(case["per"])]


# ------------------------------------------------------------ prepare and run ----
def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind in ("steps", "f64"):
        p = params(case, seed, hg.FP64 if kind == "f64" else hg.FP32)
        s["ck"], s["m"], s["co"] = hg.MemoryManager(p), hg.MemoryManager(p), coeffs(0, case["steps"])
        pos, vel = placed(case, seed)
        if kind == "f64":
            s["ck"].set_particles_f64(pos % np.float32(case["ng"]), vel)
        else:
            s["ck"].set_particles(pos, vel)
    elif kind == "host":
        s["m"], s["co"] = hg.MemoryManager(params(case, seed)), schedule(0, 1)[0]
        s["pos"], s["vel"] = placed(case, seed)
    elif kind == "run":
        s["m"], s["co"], s["ic"] = hg.MemoryManager(params(case, seed)), coeffs(0, case["steps"]), (*table(), *ic_numbers())
    elif kind == "late":
        p = params(case, seed)
        s["ck"], s["m"], s["co"] = hg.MemoryManager(p), hg.MemoryManager(p), coeffs(NSTEPS - case["steps"], case["steps"])
        s["ck"].generate_ic(*table(), *ic_numbers())
        for c in coeffs(0, NSTEPS - case["steps"]):
            s["ck"].step(c)
    elif kind in ("pk", "force"):
        s["m"] = hg.MemoryManager(params(case, seed))
        s["m"].set_particles(*placed(case, seed))
    elif kind == "fft":
        p = hg.make_params(case["ng"], 32, CELL * case["ng"], Z0, 0.0, NSTEPS, precision=hg.FP64 if case["f64"] else hg.FP32)
        s["m"] = hg.MemoryManager(p)
        s["x"] = grid(case, seed)
        s["y"] = torch.empty_like(s["x"])
    else:
        ps = [params(case, sd, n=n) for n, sd in zip(box_sizes(case), box_seeds(case, seed))]
        s["e"], s["ic"] = hg.Ensemble(ps), (*table(), *ic_numbers())
        s["co"] = [[c] * len(ps) for c in coeffs(0, case["steps"])]
    return s


def grid(case, seed):
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    n = case["ng"]
    return torch.randn((n, n, n), generator=g, device="cuda", dtype=torch.complex128 if case["f64"] else torch.complex64)


def spectrum(kpc):
    """P(k) of the FP32 engine: its modes come from complex64 transforms (and its files
    carry six digits), so the means are handed on in single precision."""
    k, pk, count = kpc
    return {"k": k, "pk": pk.astype(np.float32), "count": count}


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind in ("steps", "f64"):
        m = s["m"]
        m.copy_particles_from(s["ck"])
        for c in s["co"]:
            m.step(c)
        pos, vel = m.get_particles_f64() if kind == "f64" else m.get_particles()
        return {"pos": pos, "vel": vel}
    if kind == "host":
        m = s["m"]
        d0, dt, fs, d1, _ = s["co"]
        m.set_particles(s["pos"], s["vel"])
        m.update_positions(d0)
        m.cic()
        m.solve_gradient()
        m.update_velocities(dt, fs)
        m.update_positions(d1)
        pos, vel = m.get_particles()
        return {"pos": pos, "vel": vel}
    if kind == "run":
        s["m"].generate_ic(*s["ic"])
        for c in s["co"]:
            s["m"].step(c)
        return spectrum(s["m"].power_spectrum())
    if kind == "late":
        s["m"].copy_particles_from(s["ck"])
        for c in s["co"]:
            s["m"].step(c)
        return spectrum(s["m"].power_spectrum())
    if kind == "pk":
        return [spectrum(s["m"].power_spectrum(f)) for f in range(case["folds"] + 1)]
    if kind == "force":
        s["m"].cic()
        s["m"].solve_gradient()
        return s["m"].get_force()
    if kind == "fft":
        s["y"].copy_(s["x"])  # the transform is in place and the caller keeps its grid
        torch.cuda.current_stream().synchronize()  # ... and runs on the context's own stream
        s["m"]._c(hg.lib().hgpm_fft_device(s["m"].h, ctypes.c_void_p(s["y"].data_ptr()), case["dir"]))
        s["m"].synchronize()
        return s["y"]
    e = s["e"]
    for b in range(len(s["co"][0])):
        e.generate_ic(b, *s["ic"])
    e.run(s["co"])
    return stacked([spectrum(e.power_spectrum(b)) for b in range(len(s["co"][0]))])


def stacked(boxes):
    """The boxes' results as one array each."""
    return {name: None if boxes[0][name] is None else np.stack([b[name] for b in boxes]) for name in boxes[0]}


# --------------------------------------------------------------------- work ----
def step_work(np_, ng, b=4):
    """One step of a box: positions and velocities read and written, the positions read
    once more by the deposit; the density, two transforms of a real field (three passes
    over half the modes in all, the middle one both ways) and the potential's reading."""
    n, g = np_ ** 3, ng ** 3
    return (12 * b + 3 * b) * n + 8 * b * g, 200 * n + 5 * g * math.log2(g)


def pk_work(np_, ng, bins):
    """Positions read, the density written, one real transform in two passes over half
    the modes, the modes read."""
    n, g = np_ ** 3, ng ** 3
    return 12 * n + 4 * g + 5 * 4 * g + 24 * bins, 60 * n + 2.5 * g * math.log2(g) + 15 * g


def ic_work(np_):
    """Noise to modes, three displacement components back, particles written."""
    n = np_ ** 3
    return 24 * n + 4 * 4 * 4 * n, 4 * 2.5 * n * math.log2(n) + 200 * n


def work(case):
    kind = case["kind"]
    add = lambda *w: {"bytes": sum(x[0] for x in w), "flops": sum(x[1] for x in w)}  # noqa: E731
    times = lambda w, n: (w[0] * n, w[1] * n)  # noqa: E731
    if kind == "fft":
        g, b = case["ng"] ** 3, 16 if case["f64"] else 8
        return add((4 * b * g, 5 * g * math.log2(g)))  # two passes: no side of the grid stays on the chip
    if kind == "ensemble":
        w = [times(step_work(n, n), case["steps"]) for n in box_sizes(case)]
        return add(*w, *(ic_work(n) for n in box_sizes(case)), *(pk_work(n, n, case["bins"]) for n in box_sizes(case)))
    n, ng = case["np"], case["ng"]
    if kind in ("steps", "late"):
        w = add(times(step_work(n, ng), case["steps"]), (48 * n ** 3, 0))
    elif kind == "f64":
        w = add(times(step_work(n, ng, 8), case["steps"]), (96 * n ** 3, 0))
    elif kind == "host":
        w = add(step_work(n, ng), (48 * n ** 3, 0))
    elif kind == "run":
        w = add(ic_work(n), times(step_work(n, ng), case["steps"]))
    elif kind == "force":
        w = add((12 * n ** 3 + 8 * 4 * ng ** 3 + 12 * ng ** 3, 60 * n ** 3 + 5 * ng ** 3 * math.log2(ng ** 3)))
    else:
        return add(*(pk_work(n, ng, case["bins"]) for _ in range(case["folds"] + 1)))
    return add((w["bytes"], w["flops"]), pk_work(n, ng, case["bins"])) if kind in ("run", "late") else w


# -------------------------------------------------------------- in 64 bits ----
def corners(x, ng):
    """Cells and CIC weights of positions x (n, 3): eight (flat index, weight) pairs."""
    c = torch.floor(x)
    f = x - c
    c = c.long() % ng
    for i in range(8):
        o = ((i >> 2) & 1, (i >> 1) & 1, i & 1)
        w = torch.ones_like(f[:, 0])
        at = torch.zeros_like(c[:, 0])
        for d in range(3):
            w = w * (f[:, d] if o[d] else 1.0 - f[:, d])
            at = at * ng + (c[:, d] + o[d]) % ng
        yield at, w


def density(x, np_, ng):
    rho = torch.zeros(ng ** 3, dtype=torch.float64, device="cuda")
    for at, w in corners(x, ng):
        rho.index_add_(0, at, w * (ng / np_) ** 3)
    return rho.reshape(ng, ng, ng)


def forces(rho):
    ng = rho.shape[0]
    r = torch.fft.fftn(rho)
    k = 2 * math.pi / ng * torch.arange(ng, dtype=torch.float64, device="cuda")
    cs = torch.cos(k)
    den = cs[:, None, None] + cs[None, :, None] + cs[None, None, :] - 3.0
    den[0, 0, 0] = 1.0
    r *= 0.5 / den
    r[0, 0, 0] = 0.0
    sn = torch.sin(k)
    return torch.stack([torch.fft.ifftn(-1j * w * r).real for w in (sn[:, None, None], sn[None, :, None], sn[None, None, :])],
                       dim=-1).reshape(-1, 3)


def stepped(x, v, np_, ng, first, n):
    for d0, dt, fs, d1, _ in schedule(first, n):
        x = torch.remainder(x + v * d0, float(ng))
        f = forces(density(x, np_, ng))
        for at, w in corners(x, ng):
            v = v + (dt * fs) * w[:, None] * f[at]
        x = torch.remainder(x + v * float(np.float32(d1)), float(ng))
    return x, v


def binned(x, case, n, ng, fold):
    folds, bins = case.get("folds", 0), case.get("bins", 32)
    rl = float(np.float32(CELL * ng))
    for _ in range(fold):
        x = 2.0 * torch.remainder(x, ng / 2)
    p = torch.fft.fftn(density(x, n, ng)).abs() ** 2 * (rl / float(ng) ** 4)
    m = torch.arange(ng, device="cuda")
    m = torch.where(m > ng // 2 - 1, m - ng, m)
    t = math.pi * m.double() / ng
    win = torch.where(m == 0, torch.ones_like(t), t / torch.where(m == 0, torch.ones_like(t), torch.sin(t))) ** 4
    p *= win[:, None, None] * win[None, :, None] * win[None, None, :]
    d = 2 * math.pi / (rl / 2 ** fold)
    k1 = (m.double() * d).float()  # the reference's bin index is formed in FP32
    k = torch.sqrt((k1 * k1)[:, None, None] + (k1 * k1)[None, :, None] + (k1 * k1)[None, None, :])
    dk = 2 * math.pi / (rl / 2 ** folds)
    top = math.sqrt(3 * ((ng // 2) ** 2 * dk * dk))
    width = (top - dk) / bins
    b = ((k.double() - dk).float().double() / width).trunc().long()
    ok = (b >= 0) & (b < bins)
    ok[0, 0, 0] = False
    ok[ng // 2, ng // 2, ng // 2] = False
    b, p = b[ok], p[ok]
    count = torch.zeros(bins, dtype=torch.int64, device="cuda").index_add_(0, b, torch.ones_like(b))
    total = torch.zeros(bins, dtype=torch.float64, device="cuda").index_add_(0, b, p)
    mean = torch.where(count > 0, total / count.clamp(min=1), torch.zeros_like(total))
    return {"k": dk + width * (np.arange(bins, dtype=np.float32) + np.float32(0.5)).astype(np.float64), "pk": mean.cpu().numpy(),
            "count": None}


def normals(n, seed):
    """The white noise of cells 0 .. n - 1: Philox4x32-10 (Salmon et al. 2011) on counter
    (cell, 0, 0, 0), key (seed, 0), and Box-Muller on two 53-bit uniforms."""
    m32 = 0xFFFFFFFF
    i = torch.arange(n, dtype=torch.int64, device="cuda")
    c = [i & m32, i >> 32, torch.zeros_like(i), torch.zeros_like(i)]
    k0, k1 = int(seed) & m32, 0
    for _ in range(10):
        a, b = c[0] * 0xD2511F53, c[2] * 0xCD9E8D57  # low 64 bits
        c = [((b >> 32) & m32) ^ c[1] ^ k0, b & m32, ((a >> 32) & m32) ^ c[3] ^ k1, a & m32]
        k0, k1 = (k0 + 0x9E3779B9) & m32, (k1 + 0xBB67AE85) & m32
    u = [((h >> 5).double() * 67108864.0 + (lo >> 6).double()) / 9007199254740992.0 for h, lo in ((c[0], c[1]), (c[2], c[3]))]
    return torch.sqrt(-2.0 * torch.log1p(-u[0])) * torch.cos(2 * math.pi * u[1])


def initial(np_, ng, seed):
    hdr, p = table()
    delta, dot, fscal, da = ic_numbers()
    rl = float(np.float32(CELL * ng))
    m = torch.arange(np_, device="cuda")
    m = torch.where(m > np_ // 2 - 1, m - np_, m).double() * (2 * math.pi / rl)
    k2 = m[:, None, None] ** 2 + m[None, :, None] ** 2 + m[None, None, :] ** 2
    k2[0, 0, 0] = 1.0
    k = torch.sqrt(k2)
    left = (k / hdr[3]).long()
    t = torch.tensor(p, device="cuda")
    y1, y2, x1, x2 = torch.log(t[left]), torch.log(t[left + 1]), torch.log(hdr[3] * left), torch.log(hdr[3] * (left + 1))
    y = torch.where(left == 0, t[left + 1], torch.exp(y1 + (y2 - y1) / (x2 - x1) * (torch.log(k) - x1)))
    y *= np_ ** 3 / rl ** 3
    y[0, 0, 0] = 0.0
    amp = torch.fft.fftn(normals(np_ ** 3, seed).reshape(np_, np_, np_)) * torch.sqrt(y) / (delta * k2)
    psi = torch.stack([torch.fft.ifftn(-1j * ka * amp).real for ka in (m[:, None, None], m[None, :, None], m[None, None, :])], dim=-1)
    i = torch.arange(np_, dtype=torch.float64, device="cuda") * (ng / np_)
    x = torch.stack(torch.meshgrid(i, i, i, indexing="ij"), dim=-1) + delta * psi
    h = (1.0 / (1.0 + Z0)) - 0.5 * da
    return torch.remainder(x, float(ng)).reshape(-1, 3), (h * h * dot * fscal * psi).reshape(-1, 3)


def exact(case, seed):
    kind = case["kind"]
    if kind == "fft":
        x = grid(case, seed).to(torch.complex128)
        return torch.fft.fftn(x) if case["dir"] < 0 else torch.fft.ifftn(x, norm="forward")
    if kind == "ensemble":
        got = []
        for n, sd in zip(box_sizes(case), box_seeds(case, seed)):
            x, _ = stepped(*initial(n, n, sd), n, n, 0, case["steps"])
            got.append(binned(x, case, n, n, 0))
        return stacked(got)
    n, ng = case["np"], case["ng"]
    if kind == "late" or ng > 512:  # thousands of tiles long past crossing, or minutes of work
        return None
    if kind == "run":
        x, _ = stepped(*initial(n, ng, int(seed) % 2147483647), n, ng, 0, case["steps"])
        return binned(x, case, n, ng, 0)
    pos, vel = placed(case, seed)
    x, v = torch.tensor(pos, device="cuda").double() % ng, torch.tensor(vel, device="cuda").double()
    if kind == "pk":
        return [binned(x, case, n, ng, f) for f in range(case["folds"] + 1)]
    if kind == "force":
        return forces(density(x, n, ng))
    x, v = stepped(x, v, n, ng, 0, 1 if kind == "host" else case["steps"])
    return {"pos": x.cpu().numpy(), "vel": v.cpu().numpy()}
