"""Measured cases: the force evaluations and steps a StePS user has this engine do.

A case goes through the Python binding of the C ABI, as a host program does:

  oneshot  steps_force_eval from host arrays, the call the drop-in shim makes
           for every force routine call of the reference's own main loop;
  sim      a resident simulation that takes new positions, evaluates every
           row and gives its forces back (the host keeps the integrator);
  kdk      a resident simulation set up, evaluated and stepped on the device.

Particles come from the package's generators (compactified R3, perturbed T3
lattice, S1R2 cylinder) with the seed; tables are those the engine builds.
Forces of a mixed-precision evaluation are FP32 pair sums, and the caller keeps
them as float32.
"""
import math

import numpy as np
import torch

import steps_amd
from steps_amd import workloads as wl

KDK_STEPS = 4
KDK_H = 1e-4

# FLOP of one unordered pair, both of its forces: displacement and r^2 8,
# r^-3 4, two masses, twelve for the sums; plus the wrap and the tabulated
# correction (tricubic 3 x 84 FMA and its weights; bilinear; 3 x 3)
FLOP_PAIR = {"r3": 26, "t3_nearest": 32, "t3_ewald": 600, "s1r2_cic": 70, "s1r2_tsc": 112, "octree_r3": 26}


def listed():
    return [
        # a glass or test run of the drop-in: launches, copies and latency count
        dict(name="r3_oneshot_1500", path="r3", call="oneshot", n=1500, precision="fp64"),
        # the 16384-particle leapfrog run, particles resident
        dict(name="r3_kdk_16384", path="r3", call="kdk", n=16384, precision="fp64"),
        # an ordinary drop-in call, a size that fills no block evenly
        dict(name="r3_oneshot_100003", path="r3", call="oneshot", n=100003, precision="fp64"),
        # a production zoom-free run in full precision
        dict(name="r3_sim_1000000", path="r3", call="sim", n=1000000, precision="fp64"),
        # the same kind of run in mixed precision, larger
        dict(name="r3_mixed_1500000", path="r3", call="sim", n=1500000, precision="mixed"),
        # periodic box with the Ewald table: a small box, the common one, and mixed
        dict(name="t3_ewald_24", path="t3_ewald", call="oneshot", side=24, precision="fp64"),
        dict(name="t3_ewald_56", path="t3_ewald", call="sim", side=56, precision="fp64"),
        dict(name="t3_ewald_mixed_40", path="t3_ewald", call="sim", side=40, precision="mixed"),
        # periodic box, nearest image only (IS_PERIODIC = 1)
        dict(name="t3_nearest_64", path="t3_nearest", call="sim", side=64, precision="fp64"),
        # cylinder with the tabulated correction, bilinear and 3 x 3
        dict(name="s1r2_cic_262144", path="s1r2_cic", call="sim", shells=64, ring=64, planes=64, precision="fp64"),
        dict(name="s1r2_tsc_mixed_38220", path="s1r2_tsc", call="sim", shells=39, ring=28, planes=35, precision="mixed"),
        # the octree build (USE_BH) on the largest glass
        dict(name="octree_r3_2097152", path="octree_r3", call="sim", n=2097152, precision="fp64"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["r3", "r3", "t3_ewald", "t3_nearest", "s1r2_cic", "s1r2_tsc", "octree_r3"])
    if path == "octree_r3":
        return dict(path=path, call="sim", n=_log(rng, 20000, 2097152), precision="fp64")
    precision = rng.choice(["fp64", "fp64", "mixed"])
    mixed = precision == "mixed"
    if path == "r3":
        call = rng.choice(["oneshot", "sim", "kdk"])
        top = {"oneshot": 300000, "sim": 1500000 if mixed else 1000000, "kdk": 120000}[call]
        return dict(path=path, call=call, n=_log(rng, 1500, top), precision=precision)
    call = rng.choice(["oneshot", "sim"])
    if path.startswith("t3"):
        return dict(path=path, call=call, side=_log(rng, 16, 56 if path == "t3_ewald" else 64), precision=precision)
    q = _log(rng, 12, 64)
    return dict(path=path, call=call, shells=_log(rng, 24, 72), ring=q, planes=max(8, q + rng.randint(-4, 4)),
                precision=precision)


def _count(case):
    if "n" in case:
        return case["n"]
    return case["side"] ** 3 if "side" in case else case["shells"] * case["ring"] * case["planes"]


def _particles(case, seed):
    path = case["path"]
    if path in ("r3", "octree_r3"):
        return wl.r3_compactified(N=case["n"], seed=seed)
    if path.startswith("t3"):
        return wl.t3_lattice(n_side=case["side"], seed=seed, is_periodic=2 if path == "t3_ewald" else 1)
    return wl.s1r2_cylinder(n_omega=case["shells"], n_phi=case["ring"], n_z=case["planes"], seed=seed)


def _descriptor(case, w):
    prec = steps_amd.PREC_MIXED if case["precision"] == "mixed" else steps_amd.PREC_FP64
    path = case["path"]
    if path in ("r3", "octree_r3"):
        octree = dict(bh_theta=0.5, bh_particle_radius=w.particle_radius) if path == "octree_r3" else {}
        return steps_amd.make_desc(steps_amd.TOPO_R3, cosmology=1, comoving=1, precision=prec,
                                   mass_in_unit_sphere=w.mass_in_unit_sphere, **octree)
    if path == "t3_nearest":
        return steps_amd.make_desc(steps_amd.TOPO_T3, is_periodic=1, L=w.L, cosmology=1, comoving=1, precision=prec)
    if path == "t3_ewald":
        return steps_amd.make_desc(steps_amd.TOPO_T3, is_periodic=2, L=w.L, cosmology=1, comoving=1, precision=prec,
                                   t3_table=steps_amd.t3_table(2, w.L))
    table, shape = steps_amd.s1r2_table(2, w.L, w.Rsim)
    return steps_amd.make_desc(steps_amd.TOPO_S1R2, is_periodic=2, L=w.L, Rsim=w.Rsim, cosmology=1, comoving=1,
                               mass_in_unit_sphere=w.mass_in_unit_sphere, s1r2_lookup=1, precision=prec,
                               interp_order=2 if path == "s1r2_cic" else 4, s1r2_table=table, s1r2_shape=shape)


def _scale(w, k):
    """Scale factor and Hubble rate before step k."""
    a = w.a_start * (1.0 + 1e-3 * k)
    return a, wl.H0 * math.sqrt(wl.OMEGA_M * a ** -3 + wl.OMEGA_L)


def prepare(case, seed):
    w = _particles(case, seed)
    desc, keep = _descriptor(case, w)
    state = dict(case=case, w=w, desc=desc, keep=keep)
    if case["call"] != "oneshot":
        sim = steps_amd.Sim(desc, w.N)
        sim.set_state(w.x, w.M, w.soft, w.v)
        sim.synchronize()
        state["sim"] = sim
    return state


def run(state):
    case, w = state["case"], state["w"]
    keep_as = np.float32 if case["precision"] == "mixed" else np.float64
    if case["call"] == "oneshot":
        return steps_amd.force_eval(state["desc"], w.x, w.M, w.soft).astype(keep_as, copy=False)
    sim = state["sim"]
    if case["call"] == "sim":
        sim.set_positions(w.x)
        sim.forces()
        return sim.get_forces().astype(keep_as, copy=False)
    sim.set_state(w.x, w.M, w.soft, w.v)
    sim.forces()
    errmax = 0.0
    for k in range(KDK_STEPS):
        (a1, h1), (a2, h2) = _scale(w, k), _scale(w, k + 1)
        errmax = sim.step(KDK_H, a1, h1, a2, h2, w.rho_part)
    x, v = sim.get_state()
    return dict(x=x, v=v.astype(keep_as, copy=False), F=sim.get_forces().astype(keep_as, copy=False),
                errmax=keep_as(errmax))


def work(case):
    n = _count(case)
    passes = 1 + KDK_STEPS if case["call"] == "kdk" else 1
    # x, M, softening in and forces out; a kdk run also velocities in and x, v out
    nbytes = n * (64 + (72 if case["call"] == "kdk" else 0))
    if case["path"] == "octree_r3":
        pairs = n * 140.0 * math.log2(n)
    else:
        pairs = 0.5 * n * (n - 1.0)
    return dict(bytes=nbytes, flops=passes * pairs * FLOP_PAIR[case["path"]])


# ---------------------------------------------------------------------------
# the same outputs in plain torch, 64 bits
# ---------------------------------------------------------------------------

def _spline(r, beta):
    """The softened r^-3 inside beta (Gadget-2 spline)."""
    u = r / beta
    inner = 32.0 * u ** 3 - 38.4 * u ** 2 + 32.0 / 3.0
    outer = -32.0 / 3.0 * u ** 3 + 38.4 * u ** 2 - 48.0 * u + 64.0 / 3.0 - 1.0 / (15.0 * u.clamp(min=0.25) ** 3)
    return torch.where(u > 0.5, outer, inner) / beta ** 3


def _t3_exact_table(L):
    """63^3 Ewald corrections at the cell centres (real images to 2.6 L, |n| < 10 in k space)."""
    ng, alpha = 63, 2.0 / L
    dev = _device()
    g = (torch.arange(ng, dtype=torch.float64, device=dev) - (ng - 1) / 2) * (L / ng)
    r = torch.stack(torch.meshgrid(g, g, g, indexing="ij"), dim=-1)
    D = torch.zeros_like(r)

    def images(R):
        m = range(-int(R) - 1, int(R) + 2)
        return [(i, j, k) for i in m for j in m for k in m if i * i + j * j + k * k < R * R]

    for n in images(3.6):
        d = r + torch.tensor(n, dtype=torch.float64, device=dev) * L
        q = (d * d).sum(-1)
        s = q.clamp(min=1e-300).sqrt()
        c = torch.special.erfc(alpha * s) + 2.0 * alpha / math.sqrt(math.pi) * s * torch.exp(-alpha ** 2 * q)
        c = torch.where((q == 0) | (q > (2.6 * L) ** 2), torch.zeros_like(q), c / s ** 3)
        D -= d * c[..., None]
    for n in images(10.0):
        k = torch.tensor(n, dtype=torch.float64, device=dev) * (2.0 * math.pi / L)
        k2 = float((k * k).sum())
        if k2 == 0.0:
            continue
        s = torch.sin(r @ k) * (4.0 * math.pi / L ** 3 * math.exp(-k2 / (4.0 * alpha ** 2)) / k2)
        D -= s[..., None] * k
    q = (r * r).sum(-1, keepdim=True)
    D = torch.where(q > 0, D + r / q.clamp(min=1e-300) ** 1.5, torch.zeros_like(D))
    return D.reshape(-1, 3)


def _s1r2_exact_table(L, Rsim):
    """1440 x 128 corrections of the other z images, summed directly with an Euler-Maclaurin tail."""
    dev = _device()
    nrho, nz, M = 1440, 128, 400
    rho = torch.arange(nrho, dtype=torch.float64, device=dev)[:, None] * (2.25 * Rsim / (nrho - 1))
    z = ((torch.arange(nz, dtype=torch.float64, device=dev) + 0.5) * (L / nz) - 0.5 * L)[None, :]
    Dr, Dz = torch.zeros(nrho, nz, dtype=torch.float64, device=dev), torch.zeros(nrho, nz, dtype=torch.float64, device=dev)
    q = rho * rho
    for m in range(1, M + 1):
        for sgn in (-1.0, 1.0):
            d = z + sgn * m * L
            w = (q + d * d) ** -1.5
            if m == M:
                w = 0.5 * w
            Dr -= rho * w
            Dz -= d * w
    for sgn in (-1.0, 1.0):  # integral from M on and the derivative term of the end point
        d = z * sgn + M * L
        s = (q + d * d).sqrt()
        Dr -= rho / (s * (s + d) * L)
        Dz -= sgn / (s * L)
        Dr -= rho * (3.0 * d * L) * s ** -5 / 12.0
        Dz -= sgn * (3.0 * d * d * s ** -5 - s ** -3) * L / 12.0
    return torch.stack([Dr, Dz], dim=-1).reshape(-1, 2), nrho, nz


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _tricubic(T, ng, L, d):
    u = (d + 0.5 * L) * (ng / L) - 0.5
    f = u.floor()
    t = u - f
    w = torch.stack([-0.5 * t ** 3 + t ** 2 - 0.5 * t, 1.5 * t ** 3 - 2.5 * t ** 2 + 1.0,
                     -1.5 * t ** 3 + 2.0 * t ** 2 + 0.5 * t, 0.5 * t ** 3 - 0.5 * t ** 2])
    out = torch.zeros_like(d)
    for a in range(4):
        ix = (f[..., 0].long() + a - 1) % ng
        for b in range(4):
            iy = (f[..., 1].long() + b - 1) % ng
            for c in range(4):
                iz = (f[..., 2].long() + c - 1) % ng
                out += (w[a, ..., 0] * w[b, ..., 1] * w[c, ..., 2])[..., None] * T[(ix * ng + iy) * ng + iz]
    return out


def _cylinder(T, nrho, nz, L, Rsim, order, d):
    rho = (d[..., 0] ** 2 + d[..., 1] ** 2).sqrt()
    ur = (rho * ((nrho - 1) / (2.25 * Rsim))).clamp(max=nrho - 1.0)
    uz = (d[..., 2] + 0.5 * L) * (nz / L) - 0.5
    if order == 2:
        fr, fz = ur.floor(), uz.floor()
        wr, wz, first = [1.0 - (ur - fr), ur - fr], [1.0 - (uz - fz), uz - fz], 0
    else:
        fr, fz = (ur + 0.5).floor(), (uz + 0.5).floor()
        wr, wz = ([0.5 * (0.5 - s) ** 2, 0.75 - s * s, 0.5 * (0.5 + s) ** 2] for s in (ur - fr, uz - fz))
        first = -1
    D = torch.zeros(*rho.shape, 2, dtype=torch.float64, device=d.device)
    for a, p in enumerate(wr):
        ir = (fr.long() + a + first).clamp(0, nrho - 1)
        for b, q in enumerate(wz):
            D += (p * q)[..., None] * T[ir * nz + (fz.long() + b + first) % nz]
    over = torch.where(rho > 0, D[..., 0] / rho.clamp(min=1e-300), torch.zeros_like(rho))
    return torch.stack([over * d[..., 0], over * d[..., 1], D[..., 1]], dim=-1)


def _forces(case, w, x, table):
    dev, path = x.device, case["path"]
    M, h = torch.from_numpy(w.M).to(dev), torch.from_numpy(w.soft).to(dev)
    F = torch.empty_like(x)
    rows = max(1, (1 << 21 if path == "t3_ewald" else 1 << 24) // w.N)
    for i in range(0, w.N, rows):
        d = x[None, :, :] - x[i:i + rows, None, :]
        for axis in {"r3": (), "t3": (0, 1, 2), "s1": (2,)}[path[:2]]:
            c = d[..., axis]
            d[..., axis] = torch.where(c.abs() > 0.5 * w.L, c - torch.copysign(torch.full_like(c, w.L), c), c)
        r = (d * d).sum(-1).sqrt()
        beta = h[i:i + rows, None] + h[None, :]
        p = M * torch.where(r < beta, _spline(r, beta), r.clamp(min=1e-300) ** -3)
        f = (p[..., None] * d).sum(1)
        if path == "t3_ewald":
            f -= (M[:, None] * _tricubic(table, 63, w.L, d)).sum(1)
        elif path.startswith("s1r2"):
            T, nrho, nz = table
            f -= (M[:, None] * _cylinder(T, nrho, nz, w.L, w.Rsim, 2 if path == "s1r2_cic" else 4, d)).sum(1)
        F[i:i + rows] = f
    if path == "r3":
        F += w.mass_in_unit_sphere * x
    elif path.startswith("s1r2"):
        F[:, :2] += w.mass_in_unit_sphere * x[:, :2]
    return F


def exact(case, seed):
    path, n = case["path"], _count(case)
    most = {"r3": 1.2e10, "t3_nearest": 1.0e10, "t3_ewald": 3.0e8, "s1r2_cic": 4.0e9, "s1r2_tsc": 2.5e9, "octree_r3": 0.0}
    passes = 1 + KDK_STEPS if case["call"] == "kdk" else 1
    if passes * float(n) * n > most[path]:
        return None
    w = _particles(case, seed)
    x = torch.from_numpy(w.x).to(_device())
    table = None
    if path == "t3_ewald":
        table = _t3_exact_table(w.L)
    elif path.startswith("s1r2"):
        table = _s1r2_exact_table(w.L, w.Rsim)
    F = _forces(case, w, x, table)
    if case["call"] != "kdk":
        return F
    v = torch.from_numpy(w.v).to(x.device)
    size = torch.from_numpy(w.soft).to(x.device)
    for k in range(KDK_STEPS):
        (a1, h1), (a2, h2) = _scale(w, k), _scale(w, k + 1)
        v = v + 0.5 * KDK_H * (F * a1 ** -3 - 2.0 * h1 * v)
        x = x + KDK_H * v
        F = _forces(case, w, x, table)
        A = F * a2 ** -3 - 2.0 * h2 * v
        v = v + 0.5 * KDK_H * A
    return dict(x=x, v=v, F=F, errmax=float(((A * A).sum(-1).sqrt() / size).max()))
