"""What users of this framework have it do, as measurable cases.

Four kinds of pass, each through the public entry points of lb3d_amd.gpu:

  step     one timestep over device buffers that the caller owns
           (lb3d_gpu_step_noalloc), as a program does that couples the lattice
           update to its own GPU code and alternates two buffers;
  run      a stretch of a simulation between two dumps: Lattice.time_loop, then
           the observables that are dumped.  FP32 lattices dump 32-bit values
           (the dump files hold float32), FP64 lattices 64-bit ones;
  segment  a restart segment as the Fortran host runs it: upload of the site
           records, some steps, download of the site records;
  batch    a parameter sweep: Batch.time_loop over lattices of uneven sizes,
           then every lattice's populations.

`exact` is the same timestep in plain torch, in 64 bits.
"""
import ctypes
import math

import numpy as np
import torch

from lb3d_amd import gpu
from lb3d_amd.gpu import (LB3D_BC_LEES_EDWARDS, LB3D_BC_PERIODIC, LB3D_FP32_DEV, LB3D_FP64, Batch, Lattice,
                          make_params)

RHO = 0.7          # mean density of every component
G_SURF = dict(g_bs=-0.006, g_ss=-0.003)
WALL = dict(g_wr=-0.1, rock_colour_r=1.0, rock_colour_b=0.0)

# D3Q19: vectors, degeneracies, opposite directions
CX = (1, -1, 0, 0, 0, 0, 1, 1, 1, 1, -1, -1, -1, -1, 0, 0, 0, 0, 0)
CY = (0, 0, 1, -1, 0, 0, 1, -1, 0, 0, 1, -1, 0, 0, 1, 1, -1, -1, 0)
CZ = (0, 0, 0, 0, 1, -1, 0, 0, 1, -1, 0, 0, 1, -1, 1, -1, 1, -1, 0)
GD = (2, 2, 2, 2, 2, 2) + (1,) * 13
BOUNCE = (1, 0, 3, 2, 5, 4, 11, 10, 13, 12, 7, 6, 9, 8, 17, 16, 15, 14, 18)
W = (1.0 / 36.0,) * 18 + (1.0 / 3.0,)
CLAMP_RHO = 9.99999993922529e-09
CLAMP_SURF = 9.999999747378752e-05


def case(kind, nx, ny, nz, ncomp, precision, **more):
    return dict(kind=kind, nx=nx, ny=ny, nz=nz, ncomp=ncomp, precision=precision, **more)


def listed():
    return [
        # the smallest call: one step of a lattice of the reference's test size
        # in a caller's own loop, where launches and latency count
        dict(name="step_ternary_fp32_16", **case("step", 16, 16, 16, 3, "fp32")),
        # an ordinary binary lattice with odd edges, reference precision
        dict(name="step_binary_fp64_61x47x53", **case("step", 61, 47, 53, 2, "fp64")),
        # about the largest lattices that the caller-buffer step takes
        dict(name="step_ternary_fp32_120x116x112", **case("step", 120, 116, 112, 3, "fp32")),
        dict(name="step_ternary_fp64_80x96x88", **case("step", 80, 96, 88, 3, "fp64")),
        # the reference's own test runs: 16^3 with surfactant, 10 steps, dumps
        dict(name="segment_ternary_fp64_16", **case("segment", 16, 16, 16, 3, "fp64", steps=10)),
        # a channel with wetting walls, restarted and dumped
        dict(name="segment_walls_fp64_48x40x56", **case("segment", 48, 40, 56, 2, "fp64", steps=50, walls=True)),
        # the parity configuration: 32^3 in reference precision for 100 steps
        dict(name="run_binary_fp64_32", **case("run", 32, 32, 32, 2, "fp64", steps=100, pops=True)),
        # an ordinary spinodal decomposition run, ragged edges, many steps a dump
        dict(name="run_binary_fp32_90x100x77", **case("run", 90, 100, 77, 2, "fp32", steps=300)),
        # the largest binary lattice
        dict(name="run_binary_fp32_256", **case("run", 256, 256, 256, 2, "fp32", steps=100)),
        # sheared flow
        dict(name="run_lees_edwards_fp32_256x64x64", **case("run", 256, 64, 64, 2, "fp32", steps=300, shear=0.05)),
        # a large microemulsion
        dict(name="run_ternary_fp32_128", **case("run", 128, 128, 128, 3, "fp32", steps=100)),
        # a sweep over the coupling on lattices of uneven sizes
        dict(name="batch_ternary_fp32_8", **case("batch", 0, 0, 0, 3, "fp32", steps=100,
                                                  edges="64 24 48 16 56 40 32 48")),
    ]


def edges_of(rng, sites, least=8):
    """Three edges, odd ones among them, whose product is about `sites`."""
    e = round(sites ** (1.0 / 3.0))
    a, b = (max(least, round(e * math.exp(rng.uniform(-0.4, 0.4)))) for _ in range(2))
    return a, b, max(least, round(sites / (a * b)))


def log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(("step", "step", "run", "run", "segment", "batch"))
    ncomp, precision = rng.choice((2, 3)), rng.choice(("fp32", "fp64"))
    if kind == "step":
        # the caller-buffer step holds the moments of so many sites
        most = 60e6 / ((40 if ncomp == 3 else 16) * (2 if precision == "fp64" else 1))
        return case(kind, *edges_of(rng, log_uniform(rng, 10 ** 3, 0.9 * most)), ncomp, precision)
    if kind == "run":
        sites = log_uniform(rng, 12 ** 3, 1.5e6 if ncomp == 3 or precision == "fp64" else 4e6)
        more = dict(shear=round(rng.uniform(0.02, 0.06), 3)) if ncomp == 2 and rng.random() < 0.4 else {}
        return case(kind, *edges_of(rng, sites), ncomp, precision, steps=rng.randrange(20, 121), **more)
    if kind == "segment":
        more = dict(walls=True) if ncomp == 2 and rng.random() < 0.5 else {}
        return case(kind, *edges_of(rng, log_uniform(rng, 12 ** 3, 60 ** 3)), ncomp, "fp64",
                    steps=rng.randrange(10, 81), **more)
    edges = [rng.randrange(13, 57) for _ in range(rng.randrange(4, 9))]
    return case(kind, 0, 0, 0, ncomp, precision, steps=rng.randrange(20, 81), edges=" ".join(map(str, edges)))


def dims_of(c):
    if c["kind"] == "batch":
        return [(int(e),) * 3 for e in c["edges"].split()]
    return [(c["nx"], c["ny"], c["nz"])]


def g_br_of(k):
    return 0.06 + 0.01 * (k % 7)


def keywords(c):
    kw = dict(ncomp=c["ncomp"], bdist=2, precision=LB3D_FP64 if c["precision"] == "fp64" else LB3D_FP32_DEV,
              boundary=LB3D_BC_PERIODIC, **G_SURF)
    if c["kind"] != "batch":
        kw["g_br"] = 0.08
    if c.get("shear"):
        kw.update(boundary=LB3D_BC_LEES_EDWARDS, shear_u=c["shear"])
    if c.get("walls"):
        kw.update(WALL)
    return kw


def amp_of(c):
    return (0.01, 0.01, 0.0)


# --------------------------------------------------------------------------
# inputs


def step_inputs(c, seed):
    """Populations near a rest equilibrium (deviations from it for FP32) and
    dipoles of up to unit length, in the device layout."""
    dt = torch.float64 if c["precision"] == "fp64" else torch.float32
    shape = (c["nz"], c["ny"], c["nx"])
    g = torch.Generator(device="cuda").manual_seed(seed)

    def noise(*lead):
        return torch.rand(*lead, *shape, generator=g, device="cuda", dtype=torch.float64) * 2 - 1

    w = torch.tensor(W, device="cuda", dtype=torch.float64)[None, :, None, None, None]
    f = w * (0.01 * noise(c["ncomp"], 1) + 0.002 * noise(c["ncomp"], 19))
    if c["precision"] == "fp64":
        f = f + w * RHO
    db = 0.5 * noise(3) if c["ncomp"] == 3 else None
    return f.to(dt).contiguous(), None if db is None else db.to(dt).contiguous()


def wall_sites(c):
    """Two walls across x and a post between them."""
    rock = np.zeros((c["nz"], c["ny"], c["nx"]), bool)
    rock[:, :, 0] = rock[:, :, -1] = True
    rock[c["nz"] // 3:c["nz"] // 2, c["ny"] // 4:c["ny"] // 2, c["nx"] // 2] = True
    return rock


def site_records(c, seed):
    """Site records with a one-site halo, as the Fortran host hands them over."""
    C, nx, ny, nz = c["ncomp"], c["nx"], c["ny"], c["nz"]
    sd = 79 if C == 3 else 49
    r = np.random.default_rng(seed)
    N = np.zeros((nz + 2, ny + 2, nx + 2, sd))
    I = N[1:-1, 1:-1, 1:-1]
    for k in range(C):
        rho = RHO + (0.01 if k < 2 else 0.0) * (2 * r.random((nz, ny, nx)) - 1)
        I[..., 24 * k:24 * k + 19] = rho[..., None] * np.array(W)
    if C == 3:
        z, ph = 2 * r.random((nz, ny, nx)) - 1, 2 * np.pi * r.random((nz, ny, nx))
        s = np.sqrt(1 - z * z)
        I[..., 75], I[..., 76], I[..., 77] = s * np.cos(ph), s * np.sin(ph), z
    if c.get("walls"):
        rock = wall_sites(c)
        I[rock] = 0.0
        I[rock, sd - 1] = 1.0
        I[rock, 23] = WALL["rock_colour_r"]
    return N


def prepare(c, seed):
    kw = keywords(c)
    s = dict(case=c)
    if c["kind"] == "step":
        f, db = step_inputs(c, seed)
        s.update(params=make_params(c["nx"], c["ny"], c["nz"], **kw), f=[f, torch.empty_like(f)],
                 db=[db, None if db is None else torch.empty_like(db)], cur=0)
        return s
    if c["kind"] == "batch":
        dims = dims_of(c)
        b = Batch(dims, per_lattice=[dict(g_br=g_br_of(k)) for k in range(len(dims))], **kw)
        for k in range(len(dims)):
            b.init_noise(k, 1000 * seed + k, rho_mean=(RHO,) * 3, amp=amp_of(c), dipoles=True)
        s["batch"] = b
        return s
    g = s["lattice"] = Lattice(c["nx"], c["ny"], c["nz"], **kw)
    if c["kind"] == "segment":
        s["sites"] = site_records(c, seed)
    else:
        g.init_noise(seed, rho_mean=(RHO,) * 3, amp=amp_of(c), dipoles=True)
        g.bc_init()
    return s


def dumped(c, a):
    """A dump's values: 32-bit ones of FP32 lattices."""
    return a if c["precision"] == "fp64" else a.astype(np.float32)


def run(s):
    c = s["case"]
    if c["kind"] == "step":
        a, b = s["cur"], 1 - s["cur"]

        def ptr(t):
            return None if t is None else ctypes.c_void_p(t.data_ptr())

        gpu.check(gpu.lib().lb3d_gpu_step_noalloc(ctypes.byref(s["params"]), ptr(s["f"][a]), ptr(s["f"][b]),
                                                  ptr(s["db"][a]), ptr(s["db"][b]),
                                                  ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)),
                  "step_noalloc")
        s["cur"] = b
        return dict(f=s["f"][b], db=s["db"][b])
    if c["kind"] == "batch":
        b = s["batch"]
        b.time_loop(c["steps"])
        return [dumped(c, b.populations(k)) for k in range(len(b.dims))]
    g = s["lattice"]
    if c["kind"] == "segment":
        g.upload_sites(s["sites"])
        g.bc_init()
        g.time_loop(c["steps"])
        return dict(sites=g.download_sites())
    g.time_loop(c["steps"])
    out = dict(density=dumped(c, g.density()))
    if c.get("pops"):
        out["populations"] = dumped(c, g.populations())
    return out


# --------------------------------------------------------------------------
# work


def work(c):
    """Every step reads and writes each population (and dipole) once; then the
    outputs, once."""
    r = 8 if c["precision"] == "fp64" else 4
    C, steps = c["ncomp"], c.get("steps", 1)
    sites = sum(x * y * z for x, y, z in dims_of(c))
    state = (19 * C + (3 if C == 3 else 0)) * r
    # densities, forces, relaxation (and dipoles): about so many operations a site
    flops = 1400 if C == 3 else 500
    out = 0
    if c["kind"] == "run":
        out = C * r * (20 if c.get("pops") else 1)
    elif c["kind"] == "segment":
        out = 2 * 8 * (79 if C == 3 else 49)
    elif c["kind"] == "batch":
        out = 19 * C * r
    return dict(bytes=sites * (2 * state * steps + out), flops=sites * flops * steps)


# --------------------------------------------------------------------------
# the same in plain torch, in 64 bits


def shift(a, dx, dy, dz):
    """a at (x + dx, y + dy, z + dz), periodic; a[..., z, y, x]."""
    sh, dims = [], []
    for d, axis in ((dx, -1), (dy, -2), (dz, -3)):
        if d:
            sh.append(-d)
            dims.append(axis)
    return torch.roll(a, sh, dims) if sh else a


class Plain:
    """One lattice's timestep in torch, 64 bits; tau = amass = 1, bdist 2."""

    def __init__(self, c, n, db=None, g_br=0.08, rock=None):
        self.C, self.n, self.db, self.g_br, self.rock = c["ncomp"], n, db, g_br, rock
        self.beta, self.da = 10.0, None
        nx, self.nz = n.shape[-1], n.shape[-3]
        self.shear = nx / (nx - 1.0) * c["shear"] if c.get("shear") else None
        self.shear_sum = self.shear

    def halo(self, n):
        """The Lees-Edwards x-halo planes of populations n, (C, 19, nz, ny) each."""
        off = 2.0 * self.shear_sum
        lelo = int(math.fmod(int(off), self.nz))
        f, b = abs(off - math.trunc(off)), 0 if lelo >= 0 else -1
        hi, lo = n[..., -1], n[..., 0]

        def at(p, dz):
            return torch.roll(p, -dz, -2)

        low = (1 - f) * at(hi, lelo + b) + f * at(hi, lelo + 1 + b)
        high = f * at(lo, -lelo - 1 - b) + (1 - f) * at(lo, -lelo - b)
        out = []
        for p, sign in ((low, -1.0), (high, 1.0)):
            rho = torch.stack([self.rho(p[k]) for k in range(2)])
            u = sum(self.mom(p[k]) for k in range(2)) / rho.sum(0)
            v = u.clone()
            v[2] = v[2] + 2.0 * sign * self.shear
            out.append(p + rho[:, None] * (self.feq(v) - self.feq(u))[None])
        return out

    @staticmethod
    def rho(n):
        r = n[0] * float(GD[0])
        for i in range(1, 19):
            r = r + n[i] * float(GD[i])
        return r

    @staticmethod
    def mom(n):
        m = [torch.zeros_like(n[0]) for _ in range(3)]
        for i in range(18):
            for a, cv in enumerate((CX, CY, CZ)):
                if cv[i]:
                    m[a] = m[a] + n[i] * float(GD[i] * cv[i])
        return torch.stack(m)

    @staticmethod
    def feq(u):
        """Third-order equilibrium weights of velocity u."""
        t = 3.0 * u
        uke = (t * t).sum(0) / 6.0
        out = []
        for i in range(18):
            cu = sum(float(cv[i]) * t[a] for a, cv in enumerate((CX, CY, CZ)) if cv[i])
            out.append((1 - uke) * (1 + cu) / 36.0 + cu * cu / 72.0 + cu ** 3 / 216.0)
        out.append((1 - uke) / 3.0)
        return torch.stack(out)

    def stream(self):
        if self.shear is not None:
            low, high = self.halo(self.n)
            e = torch.cat((low[..., None], self.n, high[..., None]), -1)
            return torch.stack([shift(e[:, i], -CX[i], -CY[i], -CZ[i])[..., 1:-1] for i in range(19)], 1)
        s = torch.stack([shift(self.n[:, i], -CX[i], -CY[i], -CZ[i]) for i in range(19)], 1)
        if self.rock is not None:
            for i in range(19):
                src = shift(self.rock, -CX[i], -CY[i], -CZ[i])
                s[:, i] = torch.where(self.rock, self.n[:, i], torch.where(src, self.n[:, BOUNCE[i]], s[:, i]))
        return s

    def dipoles(self, s, rho):
        """Advected dipole, then the relaxed dipole field."""
        da = torch.zeros_like(self.db)
        for i in range(19):
            da = da + GD[i] * s[2, i][None] * shift(self.db, -CX[i], -CY[i], -CZ[i])
        drb = rho[1] - rho[0]  # g_bs < 0
        h = da.clone()
        hc = torch.zeros_like(da)
        for i in range(18):
            cv = (CX[i], CY[i], CZ[i])
            p = shift(da, *cv)
            m = shift(drb, *cv) * GD[i]
            pc = sum(cv[a] * p[a] for a in range(3) if cv[a])
            h = h + GD[i] * p
            for a in range(3):
                if cv[a]:
                    hc[a] = hc[a] + m * cv[a]
                    h[a] = h[a] - 2.0 * GD[i] * cv[a] * pc
        h = h + hc
        mag = self.beta * torch.sqrt((h * h).sum(0))
        big = mag > 10.0e-3
        safe = torch.where(big, mag, torch.ones_like(mag))
        e = torch.where(big[None], (1.0 / torch.tanh(safe) - 1.0 / safe)[None] * (self.beta * h) / safe[None],
                        self.beta / 3.0 * h)
        self.da, self.db = da, e  # tau_d = 1, d_0 = 1: only the relaxed part stays

    def forces(self, psi, rho, halo):
        C = self.C
        F = torch.zeros(C, 3, *psi.shape[1:], dtype=psi.dtype, device=psi.device)
        frb, fbr = torch.zeros_like(F[0]), torch.zeros_like(F[0])
        wall = None
        if self.rock is not None:
            wall = torch.stack([1 - torch.exp(-(rho[0] + WALL["rock_colour_r"])),
                                1 - torch.exp(-(rho[1] + WALL["rock_colour_b"]))])
            fwr = torch.zeros_like(frb)
            psi_f, psi_w = psi * ~self.rock, wall[0] * self.rock
        else:
            psi_f = psi
        if halo is not None:
            psi_f = torch.cat((halo[0][..., None], psi, halo[1][..., None]), -1)
        if C == 3:
            fcs, fsc, fss = (torch.zeros_like(frb) for _ in range(3))
            d_all, x = self.db * psi[2][None], self.db
        for i in range(18):
            cv = (CX[i], CY[i], CZ[i])
            q = shift(psi_f, *cv)
            q = q[..., 1:-1] if halo is not None else q
            for a in range(3):
                if cv[a]:
                    frb[a] = frb[a] + (GD[i] * cv[a]) * q[1]
                    fbr[a] = fbr[a] + (GD[i] * cv[a]) * q[0]
            if wall is not None:
                w = shift(psi_w, *cv)
                for a in range(3):
                    if cv[a]:
                        fwr[a] = fwr[a] + (GD[i] * cv[a]) * w
            if C == 3:
                d = shift(d_all, *cv)
                dc = sum(cv[a] * d[a] for a in range(3) if cv[a])
                xc = sum(cv[a] * x[a] for a in range(3) if cv[a])
                dx = (d * x).sum(0)
                br = (q[1] - q[0]) * GD[i]
                for a in range(3):
                    t = d[a] * xc + dc * x[a]
                    fc, fs = d[a], x[a]
                    if cv[a]:
                        t = t + cv[a] * (dx - 2.0 * xc * dc)
                        fc, fs = fc - 2.0 * cv[a] * dc, fs - 2.0 * cv[a] * xc
                    fcs[a] = fcs[a] + GD[i] * fc
                    fsc[a] = fsc[a] + br * fs
                    fss[a] = fss[a] + 8.0 * GD[i] * t
        F[0] = -self.g_br * frb * psi[0]
        F[1] = -self.g_br * fbr * psi[1]
        if wall is not None:
            F[0] = F[0] - WALL["g_wr"] * fwr * psi[0]
            F[:, :, self.rock] = 0.0
        if C == 3:
            two_bs = 2.0 * G_SURF["g_bs"]
            F[0] = F[0] + two_bs * fcs * psi[0]
            F[1] = F[1] - two_bs * fcs * psi[1]
            F[2] = (two_bs * fsc - G_SURF["g_ss"] * fss) * psi[2]
        return F

    def step(self):
        if self.shear is not None:
            self.shear_sum = self.shear_sum + self.shear
        s = self.stream()
        rho = torch.stack([self.rho(s[k]) for k in range(self.C)])
        halo = None
        if self.shear is not None:
            halo = [torch.stack([1 - torch.exp(-self.rho(p[k])) for k in range(2)]) for p in self.halo(s)]
        if self.C == 3:
            self.dipoles(s, rho)
        F = self.forces(1 - torch.exp(-rho), rho, halo)
        u = sum(self.mom(s[k]) for k in range(self.C)) / rho.sum(0).clamp(min=CLAMP_RHO)
        for k in range(self.C):
            # tau = 1: relaxation to the equilibrium itself
            s[k] = rho[k] * self.feq(u + F[k] / rho[k].clamp(min=CLAMP_RHO))
        self.n, self.last_rho = s, rho


def mix64(z):
    """The finaliser of splitmix64 on int64 tensors (wrapping arithmetic)."""
    def right(v, k):
        return (v >> k) & ((1 << (64 - k)) - 1)

    def signed(k):
        return k - (1 << 64) if k >> 63 else k

    z = z + signed(0x9E3779B97F4A7C15)
    z = (z ^ right(z, 30)) * signed(0xBF58476D1CE4E5B9)
    z = (z ^ right(z, 27)) * signed(0x94D049BB133111EB)
    return z ^ right(z, 31)


def noise_state(c, seed, dims):
    """The seeded state of init_noise."""
    nx, ny, nz = dims
    site = torch.arange(nx * ny * nz, dtype=torch.int64, device="cuda")

    def uniform(stream):
        key = mix64(torch.tensor(seed ^ (stream << 48), dtype=torch.int64, device="cuda"))
        h = mix64(key ^ site)
        return (((h >> 11) & ((1 << 53) - 1)).to(torch.float64) * 2.0 ** -53).reshape(nz, ny, nx)

    w = torch.tensor(W, dtype=torch.float64, device="cuda")[:, None, None, None]
    n = torch.stack([w * (RHO + amp_of(c)[k] * (2.0 * uniform(k) - 1.0)) for k in range(c["ncomp"])])
    if c["ncomp"] == 2:
        return n, None
    z, ph = 2.0 * uniform(3) - 1.0, 2.0 * math.pi * uniform(4)
    r = torch.sqrt(1.0 - z * z)
    return n, torch.stack((r * torch.cos(ph), r * torch.sin(ph), z))


def exact(c, seed):
    if c["kind"] == "step":
        f, db = step_inputs(c, seed)
        base = RHO * torch.tensor(W, dtype=torch.float64, device="cuda")[None, :, None, None, None]
        base = 0.0 if c["precision"] == "fp64" else base
        p = Plain(c, f.double() + base, None if db is None else db.double())
        p.step()
        return dict(f=p.n - base, db=p.db)
    if c["kind"] == "segment":
        N = site_records(c, seed)
        C, I = c["ncomp"], N[1:-1, 1:-1, 1:-1]

        def field(cols):
            return torch.from_numpy(np.ascontiguousarray(np.moveaxis(I[..., cols], -1, 0))).cuda()

        n = torch.stack([field(slice(24 * k, 24 * k + 19)) for k in range(C)])
        rock = torch.from_numpy(wall_sites(c)).cuda() if c.get("walls") else None
        p = Plain(c, n, field(slice(75, 78)) if C == 3 else None, rock=rock)
        for _ in range(c["steps"]):
            p.step()
        for k in range(C):
            I[..., 24 * k:24 * k + 19] = p.n[k].movedim(0, -1).cpu().numpy()
            I[..., 24 * k + 19] = p.last_rho[k].cpu().numpy()
            I[..., 24 * k + 20:24 * k + 23] = p.mom(p.n[k]).movedim(0, -1).cpu().numpy()
        if C == 3:
            I[..., 72:75] = p.da.movedim(0, -1).cpu().numpy()
            I[..., 75:78] = p.db.movedim(0, -1).cpu().numpy()
        return dict(sites=np.pad(I, ((1, 1), (1, 1), (1, 1), (0, 0)), mode="wrap"))
    if c["kind"] == "batch":
        out = []
        for k, dims in enumerate(dims_of(c)):
            p = Plain(c, *noise_state(c, 1000 * seed + k, dims), g_br=g_br_of(k))
            for _ in range(c["steps"]):
                p.step()
            out.append(p.n.cpu().numpy())
        return out
    p = Plain(c, *noise_state(c, seed, (c["nx"], c["ny"], c["nz"])))
    for _ in range(c["steps"]):
        p.step()
    out = dict(density=torch.stack([p.rho(p.n[k]) for k in range(c["ncomp"])]).cpu().numpy())
    if c.get("pops"):
        out["populations"] = p.n.cpu().numpy()
    return out
