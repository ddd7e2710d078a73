"""Performance cases: the calls a program makes of this framework, over the range of sizes it serves.

kinds
  steps  a simulation's n time steps (`Sim.steps`), fused engine or the mode that replays the reference's
         call sequence; returns m
  batch  n trials of a batch of simulations of mixed sizes (`Batch`), as the sweep runs them; returns every m
  conv   the convolution of a drop-in caller: three padded forward FFTs, the k-space multiply, three inverse
         FFTs through the C entry points; returns the field
  table  what a table row costs: the total energy and the average magnetisation of the current state
  new    a simulation of a shape no live simulation has: construction, first step, m back on the host

Adaptive solvers run with their step bounded by MaxDt below what the error would allow, as a program does that
wants evenly sampled dynamics, so the trajectory is the same sequence of steps in any arithmetic.
"""
import importlib
import math

import numpy as np
import torch

mm = importlib.import_module("1_amd")

MU0 = 4e-7 * math.pi
GAMMA0 = 2.211e5


def _case(name, kind, X, Y, Z, **kw):
    c = dict(name=name, kind=kind, X=X, Y=Y, Z=Z)
    c.update(kw)
    return c


def listed():
    return [
        # the thin film of the standard problem 4 geometry: the smallest simulation a script runs, bound by launches
        _case("film_128x32_rk4", "steps", 1, 32, 128, solver="rk4", dt=2e-13, n=20, field=True),
        # an ordinary film with sizes that are no powers of two, default adaptive solver, in a static field
        _case("film_301x180_rkdp", "steps", 1, 180, 301, solver="rkdp", dt=5e-14, n=8, field=True),
        # the vortex film of the reference's larger runs
        _case("film_1024x1024_rkdp", "steps", 1, 1024, 1024, solver="rkdp", dt=3e-14, n=3, field=True),
        # a film a few cells thick, odd sizes: the shape of most members of a parameter sweep
        _case("slab_150x91x3_rkdp", "steps", 3, 91, 150, solver="rkdp", dt=3e-14, n=8, field=True),
        # the headline workload: a cuboid with uniaxial anisotropy, fixed-step RK4
        _case("cuboid_256x256x16_rk4", "steps", 16, 256, 256, solver="rk4", dt=1e-14, n=10, aniso=True),
        # a bulky grid of odd sizes, Bogacki-Shampine
        _case("block_70x60x51_rk23", "steps", 51, 60, 70, solver="rk23", dt=2e-14, n=8, aniso=True),
        # the batched sweep: simulations of mixed sizes advanced together
        _case("sweep_40_rkdp", "batch", 4, 256, 256, members=40, sweep=4, dt=2e-14, n=4),
        # the reference's own call sequence with a current through the film (spin-transfer torque)
        _case("callseq_stt_film_256x64_rk4", "steps", 1, 64, 256, mode="abi", solver="rk4", dt=1e-13, n=4, field=True,
              stt=True),
        # the drop-in convolution at powers of two, as the reference's Go driver calls it
        _case("dropin_conv_128x128x16", "conv", 16, 128, 128),
        # the same for sizes with odd and prime factors
        _case("dropin_conv_106x75x10", "conv", 10, 75, 106),
        # a table row of a running simulation
        _case("table_512x512", "table", 1, 512, 512, field=True),
        # a new simulation of a new shape: what every script pays before its first step
        _case("new_sim_128x128x8", "new", 8, 128, 128, solver="rk4", dt=1e-14, n=1, aniso=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _shape(rng, xmax, ymax, zmax, cells):
    while True:
        X = 1 if xmax == 1 else _log(rng, 2, xmax)
        Y, Z = _log(rng, 12, ymax), _log(rng, 12, zmax)
        if rng.random() < 0.3:  # people do like powers of two
            Y, Z = 1 << max(4, Y.bit_length() - 1), 1 << max(4, Z.bit_length() - 1)
        if X * Y * Z <= cells:
            return X, Y, Z


def draw(rng):
    kind = rng.choice(["film", "film", "slab", "bulk", "bulk", "batch", "abi", "conv", "conv", "table", "new"])
    solver = rng.choice(["rk4", "rkdp", "rk23"])
    dt = round(rng.uniform(1e-14, 2.5e-14), 17)
    if kind == "film":
        X, Y, Z = _shape(rng, 1, 1024, 1024, 1 << 20)
        return dict(kind="steps", X=X, Y=Y, Z=Z, solver=solver, dt=dt, n=rng.randint(2, 3), field=True)
    if kind == "slab":
        X, Y, Z = _shape(rng, 6, 400, 400, 1 << 18)
        return dict(kind="steps", X=X, Y=Y, Z=Z, solver=solver, dt=dt, n=rng.randint(2, 4), field=True)
    if kind == "bulk":
        X, Y, Z = _shape(rng, 80, 256, 256, 1 << 20)
        return dict(kind="steps", X=X, Y=Y, Z=Z, solver=solver, dt=dt, n=rng.randint(2, 4), aniso=True)
    if kind == "batch":
        return dict(kind="batch", X=4, Y=256, Z=256, members=rng.randint(8, 40), sweep=rng.randint(1, 10 ** 6), dt=dt,
                    n=rng.randint(2, 4))
    if kind == "abi":
        X, Y, Z = _shape(rng, rng.choice([1, 8]), 160, 256, 1 << 16)
        stt = rng.random() < 0.5
        return dict(kind="steps", X=X, Y=Y, Z=Z, mode="abi", solver="rk4", dt=dt, n=rng.randint(1, 3), field=True, stt=stt)
    if kind == "conv":
        X, Y, Z = _shape(rng, rng.choice([1, 24, 24]), 200, 256, 1 << 18)
        return dict(kind="conv", X=X, Y=Y, Z=Z)
    if kind == "table":
        X, Y, Z = _shape(rng, rng.choice([1, 16]), 1024, 1024, 1 << 19)
        return dict(kind="table", X=X, Y=Y, Z=Z, field=True)
    X, Y, Z = _shape(rng, rng.choice([1, 12]), 200, 200, 1 << 17)
    return dict(kind="new", X=X, Y=Y, Z=Z, solver="rk4", dt=dt, n=1, aniso=True)


# ---------------------------------------------------------------- inputs
def _m0(shape, seed, key=0):
    """A magnetised state with disorder: unit vectors about a common direction, and a slow twist."""
    rs = np.random.RandomState((seed * 7919 + key * 104729 + 17) % (1 << 31))
    X, Y, Z = shape
    d = rs.normal(size=3)
    d /= np.linalg.norm(d)
    m = 0.2 * rs.standard_normal((3, X, Y, Z)).astype(np.float32) + d.astype(np.float32)[:, None, None, None]
    ph = (2 * np.pi * (np.arange(Z) / Z + rs.uniform())).astype(np.float32)
    m[2] += 0.5 * np.sin(ph)
    m[1] += 0.5 * np.cos(ph)
    return (m / np.sqrt((m * m).sum(0, keepdims=True))).astype(np.float32)


def _config(c, seed, key=0):
    X, Y, Z = c["X"], c["Y"], c["Z"]
    film = X == 1
    cfg = dict(size=(X, Y, Z), cellsize=(3e-9, 4e-9, 4e-9) if film else (4e-9, 4e-9, 4e-9),
               msat=8e5 if film else 1e6, aexch=1.3e-11, alpha=0.1, solver=c.get("solver", "rkdp"),
               maxerror=1e-4, dt=c.get("dt", 1e-14), max_dt=c.get("dt", 1e-14), m0=_m0((X, Y, Z), seed, key))
    if cfg["solver"] == "rk4":
        cfg["max_dt"] = 0.0
    if c.get("field"):
        cfg["field"] = ("static", (1e-3, 4.3e-3, -24.6e-3))
    if c.get("aniso"):
        cfg.update(k1=5e5, anis_axis=(1.0, 0.0, 0.0))
    if c.get("stt"):
        rs = np.random.RandomState(seed % (1 << 31))
        cfg["stt"] = dict(j=(2e11, 3e11, 1e12), pol=0.6, xi=0.05,
                          mask=(0.5 + rs.uniform(size=(3, X, Y, Z))).astype(np.float32))
    return cfg


def _members(c, seed):
    out = []
    for j, cfg in enumerate(mm.workloads.sweep(c["members"], seed=c["sweep"])):
        cfg.update(dt=c["dt"], max_dt=c["dt"], maxerror=1e-4, m0=_m0(cfg["size"], seed, j + 1))
        out.append(cfg)
    return out


def _sim(cfg, mode="fused"):
    s = mm.workloads.make_sim(cfg, mode)
    stt = cfg.get("stt")
    if stt:
        s.currentmask_array(stt["mask"])
        s.spinpolarization(stt["pol"])
        s.xi(stt["xi"])
        jx, jy, jz = stt["j"]
        s.currentdensity(jz, jy, jx)
    return s


class _View:
    """m in device memory, as a tensor that shares it."""

    def __init__(self, sim, shape):
        ptr = sim._lib.mm_sim_device_m(sim._ptr)
        self.__cuda_array_interface__ = dict(shape=(3,) + tuple(shape), typestr="<f4", data=(int(ptr), False), version=3,
                                             strides=None)


def _tensor(sim, shape):
    return torch.as_tensor(_View(sim, shape), device="cuda")


def _conv_kernel(c, seed):
    """Kernel spectra of random values (6 components, 4 for a film), real and the same at (kx, ky) and (-kx, -ky)
    as a real kernel's are, divided by the size."""
    X, Y, Z = c["X"], c["Y"], c["Z"]
    P = (2 * X if X > 1 else 1, 2 * Y, 2 * Z)
    g = torch.Generator().manual_seed(seed + 12345)
    k = torch.rand((6 if X > 1 else 4, P[0], P[1], Z + 1), generator=g) - 0.3
    k = 0.5 * (k + k.flip(1, 2).roll((1, 1), (1, 2)))
    return P, (k / (P[0] * P[1] * P[2])).float()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "steps":
        cfg = _config(case, seed)
        s = _sim(cfg, case.get("mode", "fused"))
        s.state()  # construction
        return dict(kind=kind, sim=s, n=case["n"], m=_tensor(s, cfg["size"]))
    if kind == "batch":
        cfgs = _members(case, seed)
        sims = [_sim(cfg) for cfg in cfgs]
        b = mm.Batch(sims)
        return dict(kind=kind, batch=b, n=case["n"], m=[_tensor(s, cfg["size"]) for s, cfg in zip(sims, cfgs)])
    if kind == "conv":
        P, k = _conv_kernel(case, seed)
        size = (case["X"], case["Y"], case["Z"])
        lib = mm.load()
        isz, ip = np.array(size, np.int32), np.array(P, np.int32)
        plan = _Plan(lib, lib.new_gpuFFT3dPlan_padded(isz.ctypes.data, ip.ctypes.data))
        m = torch.from_numpy(_m0(size, seed)).cuda()
        phys = P[0] * P[1] * (P[2] + 2)
        st = dict(kind=kind, lib=lib, plan=plan, m=m, h=torch.empty_like(m), k=k.cuda(), n=size[0] * size[1] * size[2],
                  phys=phys, buf=[torch.empty(phys, device="cuda") for _ in range(3)])
        torch.cuda.synchronize()
        return st
    if kind == "table":
        s = _sim(_config(dict(case, solver="rk4"), seed))
        s.state()
        return dict(kind=kind, sim=s)
    return dict(kind=kind, cfg=_config(case, seed), n=case["n"])


class _Plan:
    def __init__(self, lib, p):
        self.lib, self.p = lib, p

    def __del__(self):
        self.lib.delete_gpuFFT3dPlan(self.p)


def run(st):
    kind = st["kind"]
    if kind == "steps":
        st["sim"].steps(st["n"])
        return st["m"]
    if kind == "batch":
        st["batch"].start(steps=st["n"])
        st["batch"].trials(st["n"])
        return st["m"]
    if kind == "conv":
        lib, plan, n = st["lib"], st["plan"].p, st["n"]
        m, h, buf = st["m"].data_ptr(), st["h"].data_ptr(), [b.data_ptr() for b in st["buf"]]
        for c in range(3):
            lib.gpuFFT3dPlan_forward(plan, m + 4 * c * n, buf[c])
        k = [st["k"][i].data_ptr() for i in range(len(st["k"]))]
        if len(k) == 6:
            lib.gpu_kernelmul6(*buf, *k, st["phys"])
        else:
            lib.gpu_kernelmul4(*buf, *k, st["phys"])
        for c in range(3):
            lib.gpuFFT3dPlan_inverse(plan, buf[c], h + 4 * c * n)
        return st["h"]
    if kind == "table":
        return {"energy": st["sim"].energy(), "m": st["sim"].average_m()}
    s = _sim(st["cfg"])
    s.steps(st["n"])
    m = s.m
    s.free()
    return m


# ---------------------------------------------------------------- work
STAGES = {"rk4": 4, "rkdp": 6, "rk23": 3}


def _pad(size):
    return tuple(1 if n == 1 else 2 * n for n in size)


def _eval_work(size):
    """One field evaluation: m in, h out and the kernel spectrum read once; the transforms of the padded grid's
    nonzero lines, the multiply and the torque."""
    X, Y, Z = size
    P = _pad(size)
    Q = Z + 1
    nk = 6 if X > 1 else 4
    n = X * Y * Z
    byts = 24 * n + 4 * nk * (P[0] // 2 + 1) * (P[1] // 2 + 1) * Q
    fz = 2 * 3 * X * Y * 2.5 * P[2] * math.log2(P[2])
    fy = 2 * 3 * X * Q * 5 * P[1] * math.log2(P[1])
    fx = 0 if X == 1 else 2 * 3 * Q * P[1] * 5 * P[0] * math.log2(P[0])
    return byts, fz + fy + fx + 30 * P[0] * P[1] * Q + 40 * n


def _steps_work(size, solver, n):
    b, f = _eval_work(size)
    s = STAGES[solver] * n
    return {"bytes": float(s * b), "flops": float(s * f)}


def work(case):
    size = (case["X"], case["Y"], case["Z"])
    kind = case["kind"]
    if kind == "steps":
        return _steps_work(size, case["solver"], case["n"])
    if kind == "batch":
        w = [_steps_work(cfg["size"], "rkdp", case["n"]) for cfg in _members_sizes(case)]
        return {k: float(sum(x[k] for x in w)) for k in ("bytes", "flops")}
    if kind == "conv":
        P = _pad(size)
        full = (6 if size[0] > 1 else 4) * P[0] * P[1] * (P[2] // 2 + 1) * 4
        return {"bytes": float(24 * size[0] * size[1] * size[2] + full), "flops": float(_eval_work(size)[1])}
    if kind == "table":
        b, f = _eval_work(size)
        return {"bytes": float(b), "flops": float(f)}
    # the kernel's 6 components from 8 x 8 charges on two faces of each axis, one octant; then the step
    w = _steps_work(size, case["solver"], case["n"])
    n = size[0] * size[1] * size[2]
    return {"bytes": w["bytes"] + 24.0 * n, "flops": w["flops"] + 3 * 128 * 20.0 * n}


def _members_sizes(case):
    out = []
    W = mm.workloads
    for j in range(case["members"]):
        u = W.uniform01((case["sweep"] * 1000003 + j) & W.MASK64, 10)
        nx = W.SWEEP_SIZES[int(u[0] * len(W.SWEEP_SIZES)) % len(W.SWEEP_SIZES)]
        ny = W.SWEEP_SIZES[int(u[1] * len(W.SWEEP_SIZES)) % len(W.SWEEP_SIZES)]
        nz = W.SWEEP_THICK[int(u[2] * len(W.SWEEP_THICK)) % len(W.SWEEP_THICK)]
        out.append(dict(size=(nz, ny, nx)))
    return out


# ---------------------------------------------------------------- 64-bit values
def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _demag_spectrum(size, cell, acc=8):
    """rfftn over the padded grid of the kernel: the field at displacement R of a cell magnetised along each axis,
    from acc x acc point charges on its two faces, plus the 6-neighbour exchange (a film's centre value is
    overwritten by its out-of-plane neighbours). Order xx yy zz yz xz xy."""
    dev = _dev()
    f8 = torch.float64
    X, Y, Z = size
    ax = [torch.arange(n, dtype=f8, device=dev) * c for n, c in zip(size, cell)]
    R = torch.stack(torch.meshgrid(*ax, indexing="ij")).reshape(3, -1)
    npt = R.shape[1]
    oct_ = torch.zeros(6, npt, dtype=f8, device=dev)
    slot = [[0, 5, 4], [5, 1, 3], [4, 3, 2]]
    chunk = 1 << 15
    for s in range(3):
        u, v, w = s, (s + 1) % 3, (s + 2) % 3
        off = (torch.arange(acc, dtype=f8, device=dev) + 0.5) / acc - 0.5
        pv, pw = torch.meshgrid(off * cell[v], off * cell[w], indexing="ij")
        pos = torch.zeros(3, 2, acc * acc, dtype=f8, device=dev)
        pos[u, 0], pos[u, 1] = 0.5 * cell[u], -0.5 * cell[u]
        pos[v], pos[w] = pv.reshape(-1), pw.reshape(-1)
        pos = pos.reshape(3, -1)
        q = torch.cat([torch.ones(acc * acc), -torch.ones(acc * acc)]).to(device=dev, dtype=f8)
        q *= cell[v] * cell[w] / (4 * math.pi * acc * acc)
        for a in range(0, npt, chunk):
            d = R[:, a:a + chunk, None] - pos[:, None, :]
            r2 = (d * d).sum(0)
            f = q / (r2 * r2.sqrt())
            for e in range(s, 3):
                oct_[slot[s][e], a:a + chunk] = (d[e] * f).sum(1)
    oct_ = oct_.reshape(6, X, Y, Z)
    P = _pad(size)
    sgn = [(1, 1, 1), (1, 1, 1), (1, 1, 1), (1, -1, -1), (-1, 1, -1), (-1, -1, 1)]
    spec = []
    hx, hy, hz = (c * c for c in cell)
    for k in range(6):
        K = torch.zeros(P, dtype=f8, device=dev)
        K[:X, :Y, :Z] = oct_[k]
        if Z > 1:
            K[:X, :Y, P[2] - Z + 1:] = sgn[k][2] * oct_[k][:, :, 1:].flip(2)
        if Y > 1:
            K[:X, P[1] - Y + 1:, :] = sgn[k][1] * K[:X, 1:Y, :].flip(1)
        if X > 1:
            K[P[0] - X + 1:, :, :] = sgn[k][0] * K[1:X, :, :].flip(0)
        if k < 3:
            K[0, 0, 0] += 1 / hx if X == 1 else -2 / hx - 2 / hy - 2 / hz
            if X > 1:
                K[1, 0, 0] += 1 / hx
                K[-1, 0, 0] += 1 / hx
            K[0, 1, 0] += 1 / hy
            K[0, -1, 0] += 1 / hy
            K[0, 0, 1] += 1 / hz
            K[0, 0, -1] += 1 / hz
        spec.append(torch.fft.rfftn(K).real.contiguous())
    return spec


def _convolve(m, spec, P):
    X, Y, Z = m.shape[1:]
    M = [torch.fft.rfftn(m[c], s=P) for c in range(3)]
    xx, yy, zz, yz, xz, xy = spec
    H = (xx * M[0] + xy * M[1] + xz * M[2], xy * M[0] + yy * M[1] + yz * M[2], xz * M[0] + yz * M[1] + zz * M[2])
    return torch.stack([torch.fft.irfftn(h, s=P)[:X, :Y, :Z] for h in H])


TABLEAU = {
    "rk4": ([[], [.5], [0, .5], [0, 0, 1]], [1 / 6, 1 / 3, 1 / 3, 1 / 6]),
    "rk23": ([[], [.5], [0, .75]], [2 / 9, 1 / 3, 4 / 9]),
    "rkdp": ([[], [1 / 5], [3 / 40, 9 / 40], [44 / 45, -56 / 15, 32 / 9],
              [19372 / 6561, -25360 / 2187, 64448 / 6561, -212 / 729],
              [9017 / 3168, -355 / 33, 46732 / 5247, 49 / 176, -5103 / 18656]],
             [35 / 384, 0, 500 / 1113, 125 / 192, -2187 / 6784, 11 / 84]),
}


class _Exact:
    def __init__(self, cfg, spec=None):
        self.size = cfg["size"]
        ms, A = cfg["msat"], cfg["aexch"]
        self.L = math.sqrt(2 * A / (MU0 * ms * ms))
        self.T = 1 / (GAMMA0 * ms)
        self.cell = [c / self.L for c in cfg["cellsize"]]
        self.alpha = cfg["alpha"]
        dev = _dev()
        b = cfg["field"][1] if cfg.get("field") else (0, 0, 0)
        self.hext = (torch.tensor(b, dtype=torch.float64, device=dev) / (MU0 * ms))[:, None, None, None]
        self.u = None
        if cfg.get("anis_axis") is not None:
            self.u = torch.tensor(cfg["anis_axis"], dtype=torch.float64, device=dev)[:, None, None, None]
            self.k = cfg["k1"] / (A / (self.L * self.L))
        self.m = torch.from_numpy(cfg["m0"]).to(dev).double()
        self.P = _pad(self.size)
        self.spec = spec or _demag_spectrum(self.size, self.cell)
        self.stt = cfg.get("stt")
        if self.stt:
            P, xi, a = self.stt["pol"], self.stt["xi"], self.alpha
            muB, e = 9.2740091523e-24 / (ms * self.L ** 3), 1.60217646e-19 / (ms * self.L * self.T)
            bb = P * muB / (e * (1 + xi * xi))
            self.beta, self.eps = bb * (1 + a * xi), bb * (xi - a)
            mask = torch.from_numpy(self.stt["mask"]).to(dev).double()
            self.uj = [mask[i] * 0.5 * (self.stt["j"][i] / (ms / self.L)) / self.cell[i] for i in range(3)]

    def torque(self, m):
        h = _convolve(m, self.spec, self.P) + self.hext
        if self.u is not None:
            h = h + self.k * (m * self.u).sum(0, keepdim=True) * self.u
        a = self.alpha
        if not self.stt:
            c = torch.linalg.cross(m, h, dim=0)
            return (c - a * torch.linalg.cross(m, c, dim=0)) / (1 + a * a)
        hs = torch.zeros_like(m)
        for i in range(3):
            n = self.size[i]
            idx = torch.arange(n, device=m.device)
            hi, lo = (idx + 1).clamp(max=n - 1), (idx - 1).clamp(min=0)
            hs += self.uj[i] * (m.index_select(i + 1, hi) - m.index_select(i + 1, lo))
        p = torch.linalg.cross(m, h + self.eps * hs, dim=0)
        q = torch.linalg.cross(m, a * h + self.beta * hs, dim=0)
        return (p - torch.linalg.cross(m, q, dim=0)) / (1 + a * a)

    def steps(self, solver, dt, n):
        a, b = TABLEAU[solver]
        dt = dt / self.T
        m = self.m
        for _ in range(n):
            ks = []
            for row in a:
                mi = m
                for w, k in zip(row, ks):
                    if w:
                        mi = mi + dt * w * k
                ks.append(self.torque(mi))
            for w, k in zip(b, ks):
                if w:
                    m = m + dt * w * k
            m = m / (m * m).sum(0, keepdim=True).sqrt()
        self.m = m
        return m.cpu().numpy()

    def energy(self):
        m = self.m
        phi = -0.5 * (m * _convolve(m, self.spec, self.P)).sum() - (m * self.hext).sum()
        if self.u is not None:
            phi = phi - 0.5 * self.k * ((m * self.u).sum(0) ** 2).sum()
        return float(phi) * self.cell[0] * self.cell[1] * self.cell[2]


def exact(case, seed):
    kind = case["kind"]
    if kind == "conv":
        P, k = _conv_kernel(case, seed)
        m = torch.from_numpy(_m0((case["X"], case["Y"], case["Z"]), seed)).to(_dev()).double()
        k = [x.to(m.device).double() * (P[0] * P[1] * P[2]) for x in k]
        if len(k) == 4:
            k += [torch.zeros_like(k[0])] * 2
        return _convolve(m, k, P).cpu().numpy()
    if kind == "batch":
        return [_Exact(cfg).steps("rkdp", cfg["dt"], case["n"]) for cfg in _members(case, seed)]
    if kind == "table":
        e = _Exact(_config(dict(case, solver="rk4"), seed))
        return {"energy": np.float64(e.energy()), "m": e.m.mean(dim=(1, 2, 3)).cpu().numpy()}
    return _Exact(_config(case, seed)).steps(case["solver"], case["dt"], case["n"])
