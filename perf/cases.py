"""The work that users of this package have it do, as cases that can be timed.

A pass is what a simulation program does between two of its output times:
step a run that is under way, then read the particles and the fluid back (or,
for the served workload, submit runs and wait for their trajectories). Every
run continues from a moving state: a random solenoidal flow with particles
moving in it, as a program that resumes a simulation has it, so the advection
term, the particle forces and the AB2 history all count.

    listed()            the cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) the run (or the server and its requests) on the GPU
    run(state)          one pass through the public entry points
    work(case)          bytes and floating-point operations of a pass
    exact(case, seed)   the pass in 64 bits, in plain torch and numpy
"""
import math

import numpy as np
import torch

import kapsel3_amd
from kapsel3_amd import serving, workloads
from kapsel3_amd._abi import FP64, JAX_Z, JP_MOTOR, JP_NONE, JP_SLIP, MIXED, CTime, Params, make_species

DT, ETA, RHO, GRAVITY, XI = 0.05, 1.0, 1.0, 1e-3, 2.0
TS0 = 100          # steps the run has made before the pass
U_RMS = 0.05       # flow speed, grid units per time unit (particle Reynolds number about 0.25)
SHEAR_RATE = 1e-3
SERVED_A = 4.0


def _case(name, kind, n, particles, steps, precision="fp64", a=5.0, kbt=0.0):
    c = {"kind": kind, "nx": n[0], "ny": n[1], "nz": n[2], "particles": particles, "steps": steps,
         "precision": precision, "a": a, "kbt": kbt}
    return dict(c, name=name) if name else c


def listed():
    return [
        # a program that couples to the run after every step: one sphere, one
        # step, everything read back (launches, latency and small copies)
        _case("motor 32 one step", "motor", (32, 32, 32), 1, 1, a=4.0),
        # a small box between two outputs: launch-bound steps
        _case("suspension 64", "suspension", (64, 64, 64), 30, 100, a=4.0),
        # the mid-size sedimentation deck
        _case("suspension 128", "suspension", (128, 128, 128), 200, 50),
        # a flat channel, sizes that are no power of two along y and z
        _case("suspension 64x96x192", "suspension", (64, 96, 192), 120, 50),
        # the benchmark's grid and colloid count with thermal noise, 64 bits
        _case("suspension 256", "suspension", (256, 256, 256), 2000, 48, kbt=1e-3),
        # the same in mixed precision
        _case("suspension 256 mixed", "suspension", (256, 256, 256), 2000, 96, "mixed", kbt=1e-3),
        # mixed precision on a grid that is no power of two
        _case("suspension 192 mixed", "suspension", (192, 192, 192), 800, 48, "mixed"),
        # the largest grid, at the benchmark's volume fraction
        _case("suspension 512 mixed", "suspension", (512, 512, 512), 16000, 24, "mixed"),
        # squirmers: the slip iteration inside each step
        _case("squirmers 256", "squirmers", (256, 256, 256), 1000, 16),
        # Lees-Edwards shear with its stress record
        _case("sheared 256", "sheared", (256, 256, 256), 2000, 24, kbt=1e-3),
        # rigid composite bodies (trimers)
        _case("rigid 128", "rigid", (128, 128, 128), 192, 50, a=4.0),
        # the serving workload: runs of 32^3 to 96^3, all submitted at once
        _case("served 32 runs", "served", (96, 96, 96), 32, 50, "mixed", a=SERVED_A),
    ]


def draw(rng):
    kind = rng.choices(["suspension", "motor", "squirmers", "sheared", "rigid", "served"], [12, 1, 2, 2, 1, 2])[0]
    if kind == "served":
        return _case(None, kind, (96, 96, 96), rng.randint(4, 48), rng.randint(8, 64), "mixed", SERVED_A)
    a = rng.choice([4.0, 5.0])
    mixed = kind == "suspension" and rng.random() < 0.5
    # axes over the supported lengths; mixed precision is for large suspensions
    lengths = [128, 192, 256, 384] if mixed else [24, 32, 48, 64, 96, 128, 192, 256]
    while True:
        n = [rng.choice(lengths) for _ in range(3)]
        vol = n[0] * n[1] * n[2]
        if vol <= 256 ** 3 and vol >= (2 << 20 if mixed else 1 << 14):
            break
    top = max(1, int(2000 / 256 ** 3 * vol * (5.0 / a) ** 3))
    low = min(top, 400 if mixed else 1)
    if kind == "squirmers":
        top = max(1, top // 2)
        low = 1
    particles = max(1, round(math.exp(rng.uniform(math.log(low), math.log(top)))))
    if kind == "motor":
        particles = min(particles, 8)
    if kind == "rigid":
        particles = 3 * max(1, particles // 9)
    most = min(128, max(8, int(24 * 512 ** 3 / vol / (8 if kind in ("squirmers", "sheared") else 3))))
    steps = round(math.exp(rng.uniform(0.0, math.log(most))))
    kbt = 1e-3 if kind in ("suspension", "sheared") and rng.random() < 0.5 else 0.0
    return _case(None, kind, n, particles, steps, "mixed" if mixed else "fp64", a, kbt)


# ------------------------------------------------------------------ inputs
def _place(n, count, clear, rng):
    """`count` places at least `clear` apart in the periodic box: sites of a
    lattice with a third more sites than that, shifted at random."""
    m = [max(1, int(x / clear)) for x in n]
    while True:  # thin the lattice while enough sites are left
        d = max(range(3), key=lambda d: m[d] / n[d])
        if m[d] == 1 or math.prod(m) // m[d] * (m[d] - 1) < 1.35 * count + 1:
            break
        m[d] -= 1
    if math.prod(m) < count:
        raise ValueError("%d particles do not fit" % count)
    site = rng.choice(math.prod(m), count, replace=False)
    ijk = np.stack(np.unravel_index(site, m), 1)
    cell = np.array(n, float) / m
    x = ijk * cell + (0.5 + rng.uniform(-0.5, 0.5, (count, 3))) * np.maximum(cell - clear, 0.0) + rng.uniform(0, 1, 3) * cell
    return np.mod(x, np.array(n, float))


def _flow(c, rng):
    """zeta (two fields in the reference's spectral layout) of a random
    solenoidal flow of the wave numbers up to 4, and the mean velocity."""
    nx, ny, nz = c["nx"], c["ny"], c["nz"]
    z = [np.zeros((nx, ny, 2 * (nz // 2 + 1))) for _ in range(2)]
    kx, ky, kz = np.meshgrid(np.arange(-4, 5), np.arange(-4, 5), np.arange(1, 5), indexing="ij")
    k = 2 * np.pi * np.sqrt((kx / nx) ** 2 + (ky / ny) ** 2 + (kz / nz) ** 2)
    amp = U_RMS * nx * ny * nz * k / math.sqrt(4.0 * k.size)
    for f in z:
        for part in (0, 1):
            # (values that 32 bits hold, so that both precisions start alike)
            f[kx % nx, ky % ny, 2 * kz + part] = (amp * rng.standard_normal(k.shape)).astype(np.float32)
    return z[0], z[1], 0.01 * rng.standard_normal(3)


def _inputs(c, seed):
    """Parameters, particles and fluid of a run under way (one that serves no requests)."""
    rng = np.random.default_rng(seed)
    n, count, a, kind = (c["nx"], c["ny"], c["nz"]), c["particles"], c["a"], c["kind"]
    precision = MIXED if c["precision"] == "mixed" else FP64
    g = GRAVITY
    if kind == "motor":
        species, g = [make_species(propulsion=JP_MOTOR, janus_axis=JAX_Z, janus_force=(0.0, 0.0, 1e-3),
                                   janus_torque=(1e-3, 0.0, 0.0))], 0.0
    elif kind == "squirmers":
        species, g = [make_species(propulsion=JP_SLIP, janus_axis=JAX_Z, slip_vel=0.01, slip_mode=b)
                      for b in rng.uniform(-2.0, 2.0, count)], 0.0
    else:
        species = [make_species(mass_ratio=2.0, propulsion=JP_NONE)]
    P = Params(n, a=a, a_xi=XI, dt=DT, eta=ETA, rho=RHO, species=species, g=g, g_dir=2, kbt=c["kbt"],
               precision=precision, seed=int(rng.integers(1 << 30)))
    if kind == "rigid":  # bent trimers: a centre bead and two at 7.2 from it, turned at random
        arm = np.array([[0.0, 0.0, 0.0], [7.2, 0.0, 0.0], [-2.4, 6.6, 1.5]])
        centre = _place(n, count // 3, 2 * (7.3 + a) + 1.0, rng)
        q = workloads.random_quaternions(count // 3, int(rng.integers(1 << 30)))
        pos = np.concatenate([ctr + _rotate(qq, arm) for ctr, qq in zip(centre, q)])
        p = workloads.particles_at(np.mod(pos, np.array(n, float)))
        p["x_nopbc"] = pos
        return P, p, _flow(c, rng)
    p = workloads.particles_at(_place(n, count, 2 * a + 1.0, rng))
    p["q"] = p["q_old"] = workloads.random_quaternions(count, int(rng.integers(1 << 30)))
    if kind == "squirmers":
        p["spec"] = np.arange(count)
    p["v"] = 0.3 * U_RMS * rng.standard_normal((count, 3))
    p["omega"] = 0.005 * rng.standard_normal((count, 3))
    p["v_old"] = 0.99 * p["v"]
    p["omega_old"] = 0.99 * p["omega"]
    if kind == "suspension" or kind == "sheared":
        p["fr_previous"][:, 2] = -GRAVITY * RHO * 4.0 / 3.0 * math.pi * a ** 3
    return P, p, _flow(c, rng)


def _rotate(q, v):
    s, u = q[0], q[1:]
    return v + 2 * s * np.cross(u, v) + 2 * np.cross(u, np.cross(u, v))


def _requests(count, seed):
    """Parameters and particles of `count` served runs, mixed precision: the
    grids and colloid counts are the serving workload's, the places the seed's."""
    rng, place = np.random.default_rng(2024), np.random.default_rng(seed)
    out = []
    for _ in range(count):
        n = int(rng.choice(serving.SIZES))
        npart = min(int(rng.integers(1, 65)), serving.max_colloids(n, SERVED_A))
        out.append(workloads.sedimentation(n, npart, a=SERVED_A, precision=MIXED, seed=int(place.integers(1 << 30))))
    return out


def prepare(case, seed):
    c = dict(case, seed=seed)
    if c["kind"] == "served":
        srv = kapsel3_amd.Server(max_active=32, chunk_steps=8)
        return {"case": c, "server": srv, "requests": _requests(c["particles"], seed)}
    P, p, (z0, z1, uk) = _inputs(c, seed)
    r = kapsel3_amd.Run(P, c["particles"])
    r.set_particles(p)
    if c["kind"] == "rigid":
        rng = np.random.default_rng(seed + 1)
        nb = c["particles"] // 3
        r.set_rigid(3 * np.arange(nb + 1), v0=0.3 * U_RMS * rng.standard_normal((nb, 3)),
                    w0=0.002 * rng.standard_normal((nb, 3)))
        r.init_fluid()
    else:
        r.set_time(CTime(TS0, TS0 * DT, DT, DT / 2, DT, DT / 2))
    if c["kind"] == "sheared":
        r.set_shear(SHEAR_RATE)
        r.set_shear_state(0.1, SHEAR_RATE)
    r.set_fluid(z0, z1, uk)
    return {"case": c, "run": r}


# -------------------------------------------------------------------- pass
def run(state):
    c = state["case"]
    if c["kind"] == "served":
        srv = state["server"]
        ids = [srv.submit(P, p, c["steps"]) for P, p in state["requests"]]
        for rid, _ in ids:
            srv.wait(rid)
        return [traj for _, traj in ids]
    r = state["run"]
    r.step(c["steps"])
    z0, z1, uk = r.get_fluid()
    out = {"zeta0": z0, "zeta1": z1}
    if c["precision"] == "fp64":
        # (in mixed precision the mean velocity is the small difference of
        # large 32-bit sums: three numbers of rounding noise)
        out["uk_dc"] = uk
    if c["kind"] == "rigid":
        b = r.get_rigid()
        out.update({k: b[k] for k in ("xG_nopbc", "vG", "omegaG", "q", "f_hydro", "torque_hydro")})
        return out
    p = r.get_particles()
    out.update({"x": p["x_nopbc"], "v": p["v"], "omega": p["omega"], "q": p["q"],
                "f_hydro": p["f_hydro_previous"], "torque_hydro": p["torque_hydro_previous"]})
    if c["kind"] == "squirmers":
        out["f_slip"] = p["f_slip_previous"]
    if c["kind"] == "sheared":
        out["record"] = np.array(list(r.shear_record().values()))
    return out


# -------------------------------------------------------------------- work
def _sekibun(a):
    nh = int(a) + int(XI) + 2
    o = np.arange(-nh, nh + 1)
    c = np.stack(np.meshgrid(o, o, o, indexing="ij"), -1).reshape(-1, 3)
    return c[np.sqrt((c ** 2).sum(1)) < a + 0.5 * XI + 1.7321]


def _step_work(n, word, points):
    """Bytes and operations of one step of one run: the kept modes of zeta
    read and written once, u* and the force read or written once at the
    particles' points; the transforms of three velocities, five products,
    three velocities again and three forces."""
    t = [(x + 2) // 3 for x in n]
    kept = (2 * t[0] - 1) * (2 * t[1] - 1) * t[2]
    vol = n[0] * n[1] * n[2]
    fft = 2.5 * vol * math.log2(vol)
    return 2 * 2 * 2 * word * kept + 7 * word * points, 14 * fft + 200 * kept + 100 * points


def work(case):
    c = case
    if c["kind"] == "served":
        b = f = 0.0
        for P, p in _requests(c["particles"], 1):
            sb, sf = _step_work(P.shape, 4, len(p) * len(_sekibun(c["a"])))
            b, f = b + sb * c["steps"] + 48 * len(p) * c["steps"], f + sf * c["steps"]
        return {"bytes": b, "flops": f}
    n, word = (c["nx"], c["ny"], c["nz"]), 4 if c["precision"] == "mixed" else 8
    points = c["particles"] * len(_sekibun(c["a"]))
    b, f = _step_work(n, word, points)
    more = {"squirmers": 4 * 6 / 14, "sheared": 1 / 14}.get(c["kind"], 0.0)  # slip iterations; 15 transforms
    out = 2 * n[0] * n[1] * (n[2] + 2) * word + 1048 * c["particles"]        # the state read back
    return {"bytes": c["steps"] * b + out, "flops": c["steps"] * f * (1 + more)}


# ------------------------------------------------------------------- exact
class _Exact:
    """One run of spheres in 64 bits: the step of the smoothed profile method
    in the order of Time_evolution_hydro, in plain torch."""

    def __init__(self, P, p, zeta, uk, ts):
        self.dev = dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        self.c, self.n, self.ts = P.c, P.shape, ts
        t = lambda v: torch.tensor(np.ascontiguousarray(v), dtype=torch.float64, device=dev)  # noqa: E731
        self.p = {k: t(p[k]) for k in ("x", "x_nopbc", "v", "v_old", "omega", "omega_old", "q", "q_old")}
        self.p["fr"] = t(p["fr_previous"])
        s = P._species[0]  # every particle of these runs is of one species
        m = s.mass_ratio * self.c.rho * 4.0 / 3.0 * math.pi * self.c.a ** 3
        self.mass, self.moi, self.ratio = m, 0.4 * m * self.c.a ** 2, s.mass_ratio
        self.motor = (t(list(s.janus_force)), t(list(s.janus_torque))) if s.propulsion == JP_MOTOR else None
        self.cells = torch.tensor(_sekibun(self.c.a), device=dev)
        self.box = t([float(x) for x in self.n])
        # wave numbers and the 2/3 rule
        i = [torch.arange(x, device=dev) for x in (self.n[0], self.n[1], self.n[2] // 2 + 1)]
        kint = [torch.where(i[d] > self.n[d] // 2, i[d] - self.n[d], i[d]) for d in range(2)] + [i[2]]
        shape = [(-1, 1, 1), (1, -1, 1), (1, 1, -1)]
        self.k = [(kint[d].double() * (2 * math.pi / self.n[d])).view(shape[d]) for d in range(3)]
        keep = [(kint[d].abs() < (self.n[d] + 2) // 3).view(shape[d]) for d in range(3)]
        self.keep = keep[0] & keep[1] & keep[2]
        k2 = self.k[0] ** 2 + self.k[1] ** 2 + self.k[2] ** 2
        self.ik2 = torch.where(k2 > 0, 1.0 / torch.where(k2 > 0, k2, torch.ones_like(k2)), torch.zeros_like(k2))
        self.decay = torch.expm1(-self.c.eta / self.c.rho * self.c.dt * k2)
        # zeta holds (w1, w2) where kx != 0, (w2, w0) where only kx = 0, else (w0, w1)
        self.zeta = [torch.view_as_complex(t(z).view(*z.shape[:2], -1, 2)) * self.keep for z in zeta]
        self.uk = t(uk)

    def fwd(self, a):
        return torch.fft.rfftn(a) * self.keep

    def inv(self, a):
        return torch.fft.irfftn(a, s=self.n)

    def u_hat(self):
        (a, b), (kx, ky, kz) = self.zeta, self.k
        w0, w1, w2 = torch.empty_like(a), a.clone(), b.clone()
        w0[1:] = -(ky * a[1:] + kz * b[1:]) / kx[1:]
        w0[0, 1:], w1[0, 1:], w2[0, 1:] = b[0, 1:], -(kz[0] / ky[0, 1:]) * a[0, 1:], a[0, 1:]
        w0[0, 0], w1[0, 0], w2[0, 0] = a[0, 0], b[0, 0], 0.0
        u = self.curl([w0, w1, w2])
        for d in range(3):
            u[d] *= self.ik2
            u[d][0, 0, 0] = self.uk[d]
        return u

    def curl(self, f):
        kx, ky, kz = self.k
        return [1j * (ky * f[2] - kz * f[1]), 1j * (kz * f[0] - kx * f[2]), 1j * (kx * f[1] - ky * f[0])]

    @staticmethod
    def reduced(w):
        a, b = w[1].clone(), w[2].clone()
        a[0, 1:], b[0, 1:] = w[2][0, 1:], w[0][0, 1:]
        a[0, 0], b[0, 0] = w[0][0, 0], w[1][0, 0]
        return a, b

    def solve_fluid(self):
        """Advection (u . grad u, truncated) and slaved Euler, then u*."""
        u = [self.inv(x) for x in self.u_hat()]
        kx, ky, kz = self.k
        k = self.k
        conv = [torch.zeros_like(self.zeta[0]) for _ in range(3)]  # div(u u), a row at a time
        for d in range(3):
            for e in range(d, 3):
                f = self.fwd(u[d] * u[e])
                conv[d] += 1j * k[e] * f
                if e != d:
                    conv[e] += 1j * k[d] * f
        del u
        w = self.reduced(self.curl(conv))  # curl of div(u u): minus the advection of the vorticity
        del conv
        nu = self.c.eta / self.c.rho
        for d in range(2):
            z = self.zeta[d]
            z += self.decay * (z + self.ik2 / nu * w[d])
        for d in range(3):
            if self.c.fix_cell[d]:
                self.uk[d] = 0.0
        self.us_hat = self.u_hat()
        self.us = [self.inv(x) for x in self.us_hat]

    def move(self):
        p, h = self.p, self.c.dt / 2
        dx = h * (3 * p["v"] - p["v_old"]) if self.ts else self.c.dt * p["v"]
        p["x_nopbc"] = p["x_nopbc"] + dx
        p["x"] = torch.remainder(p["x"] + dx, self.box)

        def qdot(q, w):
            s, v = q[:, :1], q[:, 1:]
            return 0.5 * torch.cat([-(w * v).sum(1, keepdim=True), s * w + torch.linalg.cross(w, v)], 1)

        dq = qdot(p["q"], p["omega"])
        q = p["q"] + (h * (3 * dq - qdot(p["q_old"], p["omega_old"])) if self.ts else self.c.dt * dq)
        p["q_old"], p["q"] = p["q"], q / q.norm(dim=1, keepdim=True)

    def points(self, lo, hi):
        """Grid index, offset from the centre and profile at the points of particles lo .. hi - 1."""
        x = self.p["x"][lo:hi]
        base = x.floor()
        r = self.cells - (x - base)[:, None, :]
        g = torch.remainder(base.long()[:, None, :] + self.cells, self.box.long())
        dist = g - x[:, None, :]
        dist = (dist - torch.round(dist / self.box) * self.box).norm(dim=2)
        H = lambda y: torch.where(y > 0, torch.exp(-1.0 / torch.where(y > 0, y, torch.ones_like(y)) ** 2),  # noqa: E731
                                  torch.zeros_like(y))
        h = H(self.c.a + 0.5 * self.c.a_xi - dist)
        phi = h / (h + H(dist - self.c.a + 0.5 * self.c.a_xi))
        return (g[..., 0] * self.n[1] + g[..., 1]) * self.n[2] + g[..., 2], r, phi

    def pair_forces(self):
        """Truncated Lennard-Jones 12:6 with the multiplicity of the reference's link cells."""
        x, sigma = self.p["x"], 2.0 * self.c.a
        f = torch.zeros_like(x)
        for lo in range(0, len(x), 1024):
            d = x[lo:lo + 1024, None, :] - x
            d = d - torch.round(d / self.box) * self.box
            r2 = (d * d).sum(2)
            i, j = torch.nonzero((r2 < (2 ** (1 / 6) * sigma) ** 2) & (r2 > 0), as_tuple=True)
            r2, d = r2[i, j], d[i, j]
            s6 = (sigma ** 2 / r2) ** 3
            mag = 24.0 * self.c.epsilon / r2 * (2.0 * s6 * s6 - s6)
            for axis in range(3):
                cells = self.n[axis] // 16
                ci, cj = (x[lo + i, axis] / 16).floor(), (x[j, axis] / 16).floor()
                if cells <= 1:
                    mag = mag * 3
                elif cells == 2:
                    mag = mag * torch.where(ci == cj, 1.0, 2.0)
            f.index_add_(0, lo + i, mag[:, None] * d)
        return f

    def noise(self):
        """Philox4x32-10 normals of (particle, step, block): six per particle."""
        n, c = len(self.p["x"]), self.c
        out = np.zeros((n, 6))
        mask, u32 = np.uint64(0xFFFFFFFF), np.uint64(32)
        for b in range(3):
            w = [np.arange(n, dtype=np.uint64), np.full(n, self.ts, np.uint64), np.full(n, b, np.uint64),
                 np.full(n, c.stream_id, np.uint64)]
            k0, k1 = c.seed & 0xFFFFFFFF, c.seed >> 32
            for _ in range(10):
                m0, m1 = w[0] * np.uint64(0xD2511F53), w[2] * np.uint64(0xCD9E8D57)
                w = [(m1 >> u32) ^ w[1] ^ np.uint64(k0), m1 & mask, (m0 >> u32) ^ w[3] ^ np.uint64(k1), m0 & mask]
                k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
            u = [((w[2 * i] >> np.uint64(5)).astype(float) * 67108864.0 + (w[2 * i + 1] >> np.uint64(6)).astype(float)
                  + 0.5) / 9007199254740992.0 for i in (0, 1)]
            rad = np.sqrt(-2.0 * np.log(u[0]))
            out[:, 2 * b], out[:, 2 * b + 1] = rad * np.cos(2 * np.pi * u[1]), rad * np.sin(2 * np.pi * u[1])
        return torch.tensor(out, device=self.dev)

    def step(self):
        c, p = self.c, self.p
        self.solve_fluid()
        self.move()
        count, per = len(p["x"]), 512
        vol = self.n[0] * self.n[1] * self.n[2]
        phis = torch.zeros(vol, dtype=torch.float64, device=self.dev)
        for lo in range(0, count, per):
            g, r, phi = self.points(lo, lo + per)
            phis.index_add_(0, g.reshape(-1), phi.reshape(-1))
        us = [x.reshape(-1) for x in self.us]
        fh, th = torch.empty_like(p["v"]), torch.empty_like(p["v"])
        for lo in range(0, count, per):
            g, r, phi = self.points(lo, lo + per)
            rigid = p["v"][lo:lo + per, None] + torch.linalg.cross(p["omega"][lo:lo + per, None].expand_as(r), r)
            f = (rigid - torch.stack([x[g] for x in us], 2)) * (phi / phis[g].clamp(min=1.0))[..., None]
            fh[lo:lo + per] = -c.rho / c.dt * f.sum(1)
            th[lo:lo + per] = -c.rho / c.dt * torch.linalg.cross(r, f).sum(1)
        fr = self.pair_forces()
        fr[:, c.g_dir] -= c.g * c.rho * 4.0 / 3.0 * math.pi * c.a ** 3 * (self.ratio - 1.0)
        fm = tm = 0.0
        if self.motor is not None:
            s, v = p["q"][:, :1], p["q"][:, 1:]
            turn = lambda b: b + 2 * s * torch.linalg.cross(v, b) + 2 * torch.linalg.cross(v, torch.linalg.cross(v, b))  # noqa: E731
            fm, tm = (turn(b.expand_as(v)) for b in self.motor)
        h = c.dt / 2
        dv = h * (2 * (fh + fm) + fr + p["fr"]) if self.ts else c.dt * (fh + fm + fr)
        p["v_old"], p["omega_old"] = p["v"], p["omega"]
        p["v"] = p["v"] + dv / self.mass
        p["omega"] = p["omega"] + c.dt * (th + tm) / self.moi
        p["fr"], p["fh"], p["th"] = fr, fh, th
        if c.kbt > 0:
            z = self.noise()
            p["v"] = p["v"] + z[:, :3] * 1.439 * math.sqrt(6 * math.pi * c.eta * c.a * c.dt * c.kbt) / self.mass
            p["omega"] = p["omega"] + z[:, 3:] * 1.22 * math.sqrt(8 * math.pi * c.eta * c.a ** 3 * c.dt * c.kbt) / self.moi
        up = [torch.zeros(vol, dtype=torch.float64, device=self.dev) for _ in range(3)]
        for lo in range(0, count, per):
            g, r, phi = self.points(lo, lo + per)
            rigid = p["v"][lo:lo + per, None] + torch.linalg.cross(p["omega"][lo:lo + per, None].expand_as(r), r)
            f = rigid * (phi / phis[g].clamp(min=1.0))[..., None]
            for d in range(3):
                up[d].index_add_(0, g.reshape(-1), f[..., d].reshape(-1))
        phis.clamp_(max=1.0)
        fhat = [self.fwd((up[d] - phis * us[d]).view(*self.n)) for d in range(3)]
        kf = (self.k[0] * fhat[0] + self.k[1] * fhat[1] + self.k[2] * fhat[2]) * self.ik2
        u = [self.us_hat[d] + fhat[d] - self.k[d] * kf for d in range(3)]
        self.uk = torch.stack([x[0, 0, 0].real for x in u])
        self.zeta = list(self.reduced(self.curl(u)))
        self.ts += 1


def exact(case, seed):
    c = case
    if c["kind"] == "served":
        if c["particles"] * c["steps"] > 2000:
            return None
        out = []
        for P, p in _requests(c["particles"], seed):  # from rest: the fluid starts at rest too
            shape = (P.c.nx, P.c.ny, P.nz_)
            e = _Exact(P, p, [np.zeros(shape), np.zeros(shape)], np.zeros(3), 0)
            traj = torch.zeros((c["steps"], len(p), 6), dtype=torch.float64, device=e.dev)
            for k in range(c["steps"]):
                e.step()
                traj[k, :, :3], traj[k, :, 3:] = e.p["x"], e.p["v"]
            out.append(traj)
        return out
    if c["kind"] not in ("suspension", "motor"):
        return None  # the slip loop, the oblique grid and the bodies have no short form
    P, p, (z0, z1, uk) = _inputs(c, seed)
    e = _Exact(P, p, [z0, z1], uk, TS0)
    del z0, z1
    for _ in range(c["steps"]):
        e.step()
    out = {"zeta%d" % d: torch.view_as_real(e.zeta[d]).reshape(c["nx"], c["ny"], -1) for d in range(2)}
    if c["precision"] == "fp64":
        out["uk_dc"] = e.uk
    out.update({"x": e.p["x_nopbc"], "v": e.p["v"], "omega": e.p["omega"], "q": e.p["q"], "f_hydro": e.p["fh"],
                "torque_hydro": e.p["th"]})
    return out
