"""The work that users of this framework have it do, as measurable cases.

A case is a program's inner loop on a context that it keeps: a few time steps
(RK2 or RK4, with scalars, particles or the learned closure), a set of
statistics, a training snapshot, or some training steps, followed by the read
of what it computed into a host buffer that the program also keeps (pinned, so
that the copy runs at the rate of the link).

Physical space is ux[v][y][z][x]; a cylinder state is u[v][a][y] with a over
the (kx, kz) columns, kx slowest.  The 64-bit results of exact() come from
plain torch transforms of dense arrays uhat[y][z][kx].
"""
import ctypes
import importlib.util
import math
import pathlib
import random
import sys

import numpy as np
import torch

PKG_DIR = pathlib.Path(__file__).resolve().parents[1] / "nasa-bluewater-psdns-benchmark-minsky_amd"
CFL = math.pi  # Courant number 0.5 in the reference's convention
SYM = ((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2))
CW = (1.0, 2.0, 2.0, 1.0, 2.0, 1.0)  # Frobenius weights of the 6 components
# the closure's parameter blocks (include/psdns_sgs.h)
THETA = (("W0", (16, 135)), ("b0", (16,)), ("W1", (64, 21)), ("b1", (64,)), ("W2", (64, 64)), ("b2", (64,)),
         ("W3", (64, 64)), ("b3", (64,)), ("W4", (4, 64)), ("b4", (4,)))


def package():
    if "psdns_amd" in sys.modules:
        return sys.modules["psdns_amd"]
    spec = importlib.util.spec_from_file_location("psdns_amd", PKG_DIR / "__init__.py",
                                                  submodule_search_locations=[str(PKG_DIR)])
    mod = importlib.util.module_from_spec(spec)
    sys.modules["psdns_amd"] = mod
    spec.loader.exec_module(mod)
    return mod


def device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest grid the library takes, one forced FP32 step between two
        # reads of the state: a coarse LES or a coupled program that looks at
        # every step; launches and waits count
        {"name": "rk2_32_f32", "kind": "rk2", "n": 32, "prec": 4, "nc": 0, "kf": 3, "steps": 1},
        # a plain 64^3 FP64 DNS with shells k <= 2 held, as a student or a
        # validation run has it: several steps, then the state
        {"name": "rk2_64_f64", "kind": "rk2", "n": 64, "prec": 8, "nc": 0, "kf": 3, "steps": 10},
        # the fourth-order scheme at a size that is run for hours on one GPU
        {"name": "rk4_128_f32", "kind": "rk4", "n": 128, "prec": 4, "nc": 0, "kf": 2, "steps": 4},
        # forced isotropic turbulence in the reference's shipped precision
        {"name": "rk2_256_f64", "kind": "rk2", "n": 256, "prec": 8, "nc": 0, "kf": 3, "steps": 10},
        # the same turbulence in FP32, one size up
        {"name": "rk2_512_f32", "kind": "rk2", "n": 512, "prec": 4, "nc": 0, "kf": 3, "steps": 10},
        # the largest grid: production DNS on one GPU
        {"name": "rk2_1024_f32", "kind": "rk2", "n": 1024, "prec": 4, "nc": 0, "kf": 3, "steps": 8},
        # two passive scalars with a mean gradient carried along
        {"name": "scalars_512_f32", "kind": "rk2", "n": 512, "prec": 4, "nc": 2, "kf": 3, "steps": 5},
        # 2^20 fluid particles followed through the FP32 DNS
        {"name": "particles_512_f32", "kind": "particles", "n": 512, "prec": 4, "np": 1 << 20, "kf": 3, "steps": 5},
        # the output step of a DNS: spectrum, dissipation and the moments of
        # the velocity gradient
        {"name": "stats_512_f32", "kind": "stats", "n": 512, "prec": 4},
        # one training snapshot: the DNS field filtered onto a coarse grid with
        # its subgrid stress, and the closure's features there
        {"name": "snapshot_512_64_f32", "kind": "snapshot", "nf": 512, "n": 64, "prec": 4},
        # training of the closure on stored snapshots
        {"name": "train_64_b16384", "kind": "train", "n": 64, "snaps": 8, "batch": 16384, "steps": 20},
        # a coarse LES with the learned closure, bf16 inference
        {"name": "les_128_f32", "kind": "les", "n": 128, "prec": 4, "bf16": True, "kf": 3, "steps": 4},
    ]


def draw(rng: random.Random):
    kind = rng.choice(["rk2", "rk2", "rk2", "scalars", "rk4", "particles", "stats", "snapshot", "train", "les"])
    n = rng.choice([32, 64, 128, 256, 512])
    prec = rng.choice([4, 8])
    kf = rng.choice([2, 3, 4])  # always forced: a decaying field would die out over the passes of a measurement
    few = rng.randint(1, 8 if n > 256 else 12)
    if kind == "rk2":
        return {"kind": "rk2", "n": n, "prec": prec, "nc": 0, "kf": kf, "steps": few}
    if kind == "scalars":
        return {"kind": "rk2", "n": min(n, 256), "prec": prec, "nc": rng.randint(1, 3), "kf": kf, "steps": few}
    if kind == "rk4":
        return {"kind": "rk4", "n": min(n, 256), "prec": prec, "nc": rng.randint(0, 1), "kf": kf,
                "steps": rng.randint(1, 5)}
    if kind == "particles":
        return {"kind": "particles", "n": min(n, 256), "prec": prec, "np": round(math.exp(rng.uniform(math.log(1000),
                math.log(1 << 20)))), "kf": kf, "steps": rng.randint(2, 6)}
    if kind == "stats":
        return {"kind": "stats", "n": n, "prec": prec, "kpeak": rng.randint(3, 9)}
    if kind == "snapshot":
        nc = rng.choice([32, 64, 128])
        r = rng.choice([2, 4, 8])
        return {"kind": "snapshot", "nf": min(nc * r, 512), "n": nc, "prec": prec, "kpeak": rng.randint(3, 9)}
    if kind == "train":
        return {"kind": "train", "n": rng.choice([32, 64]), "snaps": rng.randint(1, 8),
                "batch": round(math.exp(rng.uniform(math.log(100), math.log(65536)))), "steps": rng.randint(1, 20)}
    return {"kind": "les", "n": rng.choice([32, 64, 128]), "prec": 4, "bf16": rng.random() < 0.75, "kf": 3,
            "steps": rng.randint(1, 6)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def kwave(n, dev):
    i = torch.arange(n, device=dev, dtype=torch.float64)
    return torch.where(i > n // 2, i - n, i)


def cylinder(n):
    """kx and z index of the cylinder columns, kx slowest"""
    xs, zs = [], []
    for x in range(min(int(n * math.sqrt(2.0) / 3.0) + 1, n // 2)):
        cut = int(n * (1.0 - 2.0 * math.sqrt(2.0 / 9.0 - (x / n) ** 2)) / 2)
        z = list(range(n // 2 - cut)) + list(range(n // 2 + cut + 1, n))
        xs += [x] * len(z)
        zs += z
    return torch.tensor(xs), torch.tensor(zs)


def generator(seed, dev):
    g = torch.Generator(device=dev)
    g.manual_seed(int(seed))
    return g


def spectrum_field(n, nv, seed, prec, kpeak=3.0, solenoidal=True):
    """nv random-phase cylinder variables with a broad spectrum, E(k) ~ k^4 /
    (1 + (k/kpeak)^2)^(17/6), smoothed at the truncation; energy 0.5 for the
    velocity (solenoidal, the first three), unit order for scalars.  Returns
    the state in the context's precision (on the device) and sum k^2 E(k)."""
    dev = device()
    g = generator(seed, dev)
    xs, zs = (t.to(dev) for t in cylinder(n))
    kk = kwave(n, dev)
    kx, kz, ky = xs.double()[:, None], kk[zs][:, None], kk[None, :]
    k2 = kx * kx + ky * ky + kz * kz
    y = torch.arange(n, device=dev)
    on = (9 * k2 <= 2 * n * n) & (y != n // 2)[None, :] & (zs != n // 2)[:, None] & (k2 > 0)
    k2s = torch.where(k2 > 0, k2, torch.ones_like(k2))
    e = k2s ** 2 / (1.0 + k2s / kpeak ** 2) ** (17.0 / 6.0) * torch.exp(-3.0 * k2s / (n / 3.0) ** 2)
    amp = torch.where(on, torch.sqrt(e / k2s), torch.zeros_like(e))
    u = torch.view_as_complex(torch.randn((nv, xs.numel(), n, 2), generator=g, device=dev, dtype=torch.float64)) * amp
    if solenoidal:
        p = (kx * u[0] + ky * u[1] + kz * u[2]) / k2s
        u[0] -= kx * p
        u[1] -= ky * p
        u[2] -= kz * p
    # the kx = 0 plane of a real field: u(-k) = conj u(k)
    c0 = torch.nonzero(xs == 0).flatten()
    plane = torch.zeros((nv, n, n), device=dev, dtype=torch.complex128)
    plane[:, zs[c0], :] = u[:, c0, :]
    back = (-y) % n
    plane = 0.5 * (plane + plane[:, back][:, :, back].conj())
    u[:, c0, :] = plane[:, zs[c0], :]
    wt = torch.where(xs == 0, 0.5, 1.0)[:, None]
    e3 = wt * (u[:3].abs() ** 2).sum(0)
    scale = math.sqrt(0.5 / float(e3.sum()))
    d = float((e3 * k2).sum()) * scale ** 2
    u *= scale
    return u.to(torch.complex128 if prec == 8 else torch.complex64), d


def shifts(seed, steps):
    """gsh(3, 2) of some steps: random offsets, the two stages half a cell apart"""
    r = np.random.default_rng(seed)
    a = r.random((steps + 1, 3))
    return [np.concatenate([np.mod(a[i] + 0.5, 1.0), a[i + 1]]) for i in range(steps)]


def viscosity(n, d):
    """nu for k_max eta = 1.5, eps = 2 nu d"""
    return math.sqrt(2.0 * d) * (1.5 / (math.sqrt(2.0) / 3.0 * n)) ** 2


def theta0(seed, scale4):
    """Glorot-uniform weights; the output layer scaled, its first bias an eddy
    viscosity, so that an LES with it runs on"""
    r = np.random.default_rng(seed)
    out = []
    for name, shape in THETA:
        if name[0] == "W":
            a = math.sqrt(6.0 / sum(shape)) * (scale4 if name == "W4" else 1.0)
            out.append(r.uniform(-a, a, shape).ravel())
        else:
            out.append(np.zeros(shape))
    out[-1][0] = -0.05
    return np.concatenate(out).astype(np.float32)


def store(case, seed):
    """stored snapshots of the closure: invariants, tensor basis and stresses of
    the size that turbulence gives them"""
    dev, n, s = device(), case["n"], case["snaps"]
    g = generator(seed, dev)
    lam = torch.randn((s, 5, n, n, n), generator=g, device=dev) * torch.tensor(
        [0.2, 0.2, 0.1, 0.1, 0.1], device=dev)[None, :, None, None, None]
    lam[:, 0] += 0.5
    lam[:, 1] -= 0.5
    basis = 0.3 * torch.randn((s, 4, 6, n, n, n), generator=g, device=dev)
    basis[:, :, 5] = -(basis[:, :, 0] + basis[:, :, 3])
    tau = -0.1 * basis[:, 0] + 0.05 * basis[:, 1] * lam[:, :1] + 0.05 * basis[:, 2] - 0.02 * basis[:, 3]
    tau += 0.02 * torch.randn(tau.shape, generator=g, device=dev)
    return lam, basis, tau


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------
def new_solver(P, case, n, seed):
    """a context with its field; returns it and the viscosity"""
    nc = case.get("nc", 0)
    if n > 512:  # the library's own seeded field
        s = P.Solver(n, case["prec"], viscos=1.0, nc=nc, pr=[1.0] * nc, grad=[(1.0, 0.0, 0.0)] * nc)
        s.init_field(seed=1000003 + seed)
        eps = s.shell_stats(0)[3]
        s.viscos = viscosity(n, eps / 2.0)
        return s, s.viscos
    u, d = spectrum_field(n, 3 + nc, seed, case["prec"], float(case.get("kpeak", 3)))
    nu = viscosity(n, d)
    s = P.Solver(n, case["prec"], viscos=nu, nc=nc, pr=[1.0, 0.7, 2.0][:nc], grad=[(1.0, 0.0, 0.0)] * nc)
    s.put_state(u.cpu().numpy())
    return s, nu


def pinned(shape, dtype):
    if torch.cuda.is_available():
        return torch.empty(shape, dtype=dtype, pin_memory=True)
    return torch.empty(shape, dtype=dtype)


def out_state(s, nv):
    return pinned((nv, s.num_al, s.n), torch.complex128 if s.prec == 8 else torch.complex64)


def read_state(s, buf):
    s._chk(s.L.psdns_get_state(s.h, buf.data_ptr(), 0))
    return buf


def read_sgs(m, which, buf):
    m._chk(m.L.psdns_sgs_get_field(m.h, which, ctypes.cast(buf.data_ptr(), ctypes.POINTER(ctypes.c_float))))
    return buf


def prepare(case, seed):
    P = package()
    kind, st = case["kind"], {"case": case, "at": 0}
    if kind in ("rk2", "rk4", "particles", "les"):
        n = case["n"]
        s, nu = new_solver(P, case, n, seed)
        st["solver"], st["out"] = s, out_state(s, 3 + case.get("nc", 0))
        st["gsh"] = shifts(seed, 64)
        if kind == "particles":
            pp = np.random.default_rng(seed).random((3, case["np"])) * n
            st["run"] = P.Run(s, nu, CFL, kf_shell=case["kf"], particles=pp)
            st["pp"] = pinned((9, case["np"]), torch.float64)
        elif kind == "les":
            st["closure"] = P.Closure(n)
            st["closure"].set_params(theta0(seed, 0.05))
            st["run"] = P.Les(s, nu, CFL, closure=st["closure"], bf16=case["bf16"], kf_shell=case["kf"], fused=True)
        else:
            st["run"] = (P.Run4 if kind == "rk4" else P.Run)(s, nu, CFL, kf_shell=case["kf"])
    elif kind == "stats":
        st["solver"], _ = new_solver(P, case, case["n"], seed)
    elif kind == "snapshot":
        n = case["n"]
        st["fine"], nu = new_solver(P, case, case["nf"], seed)
        st["coarse"] = P.Solver(n, case["prec"], viscos=nu)
        st["closure"] = P.Closure(n, max_snapshots=1)
        st["out"] = [out_state(st["coarse"], 3)] + [pinned((c, n, n, n), torch.float32) for c in (6, 5, 24)]
    else:
        lam, basis, tau = store(case, seed)
        m = st["closure"] = P.Closure(case["n"], max_snapshots=case["snaps"])
        for i in range(case["snaps"]):
            m.put_fields(lam[i].cpu().numpy(), basis[i].cpu().numpy(), tau[i].cpu().numpy())
            m.add_snapshot()
        m.set_params(theta0(seed, 1.0))
        st["sigma2"], st["seed"] = m.target_scale(), 17 + seed
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind in ("rk2", "rk4", "particles", "les"):
        s, r = st["solver"], st["run"]
        for _ in range(case["steps"]):
            r.step(st["gsh"][st["at"] % 64])
            st["at"] += 1
        out = [read_state(s, st["out"])]
        if kind == "particles":
            s._chk(s.L.psdns_lag_get(s.h, ctypes.cast(st["pp"].data_ptr(), ctypes.POINTER(ctypes.c_double)),
                                     case["np"]))
            out.append(st["pp"])
        return out
    if kind == "stats":
        s = st["solver"]
        ek, dk, tke, eps = s.shell_stats()
        du, dw = s.vg_moments()
        if case["prec"] == 4:  # as exact as the transformed FP32 field
            du, dw = du.astype(np.float32), dw.astype(np.float32)
        return {"ek": ek, "dk": dk, "tke": tke, "eps": eps, "dudx": du, "dwdz": dw}
    if kind == "snapshot":
        P = package()
        m = st["closure"]
        m.clear_snapshots()
        P.training_snapshot(m, st["fine"], st["coarse"])
        return [read_state_u(P, st["coarse"], st["out"][0])] + [
            read_sgs(m, w, b) for w, b in zip((P.SGS_TARGET, P.SGS_LAMBDA, P.SGS_BASIS), st["out"][1:])]
    m = st["closure"]
    losses = m.train(case["steps"], case["batch"], 1e-3, st["seed"], st["sigma2"])
    return [m.get_params(), losses.astype(np.float32)]


def read_state_u(P, s, buf):
    """the cylinder slots u of a context (where xktran leaves the coarse field)"""
    s._chk(s.L.psdns_get_field(s.h, P.FIELD_U, buf.shape[0], buf.data_ptr()))
    return buf


# ---------------------------------------------------------------------------
# what one pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    kind = case["kind"]

    def grid(n, prec):
        na = int(cylinder(n)[0].numel())
        fft = 2.5 * n ** 3 * 3 * math.log2(n)  # a real 3-D transform
        return 2 * prec * na * n, fft  # bytes of a cylinder variable

    if kind in ("rk2", "rk4", "particles", "les"):
        n, prec, nc = case["n"], case["prec"], case.get("nc", 0)
        cyl, fft = grid(n, prec)
        stages = 4 if kind == "rk4" else 2
        step_b = 2 * (3 + nc) * cyl  # the state in and out
        step_f = stages * ((8 + 4 * nc) * fft + 30 * (3 + nc) * n ** 3)
        if kind == "particles":
            step_b += 2 * 72 * case["np"] + 3 * 64 * prec * case["np"]
            step_f += 3 * fft + 400 * case["np"]
        if kind == "les":
            step_f += stages * (9 * fft + 2 * 12164 * n ** 3)
        out = (3 + nc) * cyl
        return {"bytes": case["steps"] * step_b + out, "flops": case["steps"] * step_f}
    if kind == "stats":
        cyl, fft = grid(case["n"], case["prec"])
        return {"bytes": 3 * cyl + 2 * cyl, "flops": 2 * fft + 40 * case["n"] ** 3}
    if kind == "snapshot":
        cyl, fft = grid(case["nf"], case["prec"])
        ccyl, cfft = grid(case["n"], case["prec"])
        p = case["n"] ** 3
        return {"bytes": 3 * cyl + 3 * ccyl + 2 * 35 * 4 * p, "flops": 3 * fft + 15 * case["nf"] ** 3 + 12 * cfft + 400 * p}
    b = case["batch"]
    return {"bytes": case["steps"] * (b * 4 * (135 + 24 + 6) + 7 * 4 * 12164), "flops": case["steps"] * 6.0 * b * 12164}


# ---------------------------------------------------------------------------
# 64-bit results
# ---------------------------------------------------------------------------
class Box:
    """dense spectral arrays uhat[y][z][kx] of an n^3 box, FP64"""

    def __init__(self, n):
        self.n, self.dev = n, device()
        k = kwave(n, self.dev)
        self.kx = torch.arange(n // 2 + 1, device=self.dev, dtype=torch.float64)[None, None, :]
        self.ky, self.kz = k[:, None, None], k[None, :, None]
        self.k2 = self.kx ** 2 + self.ky ** 2 + self.kz ** 2
        i = torch.arange(n, device=self.dev)
        ok = i != n // 2
        self.mask = (9 * self.k2 <= 2 * n * n) & ok[:, None, None] & ok[None, :, None]
        self.xs, self.zs = (t.to(self.dev) for t in cylinder(n))

    def dense(self, u):
        d = torch.zeros((u.shape[0], self.n, self.n, self.n // 2 + 1), device=self.dev, dtype=torch.complex128)
        d[:, :, self.zs, self.xs] = u.to(self.dev).to(torch.complex128).transpose(1, 2)
        return d

    def columns(self, d):
        return d[:, :, self.zs, self.xs].transpose(1, 2).contiguous()

    def phys(self, d):
        return torch.fft.irfftn(d, s=(self.n,) * 3, dim=(-3, -2, -1), norm="forward")

    def spec(self, f):
        return torch.fft.rfftn(f, dim=(-3, -2, -1), norm="forward")

    def shift(self, g):
        w = 2.0 * math.pi / self.n
        return torch.polar(torch.ones((), device=self.dev, dtype=torch.float64),
                           w * (self.kx * g[0] + self.ky * g[1] + self.kz * g[2]))

    def project(self, u):
        k2 = torch.where(self.k2 > 0, self.k2, torch.ones_like(self.k2))
        p = (self.kx * u[0] + self.ky * u[1] + self.kz * u[2]) / k2
        u[0] -= self.kx * p
        u[1] -= self.ky * p
        u[2] -= self.kz * p
        return u

    def shells(self, u, nshell):
        """E(ik), D(ik) / (2 nu) for ik = int(|k| + 1.5) = 1 .. nshell"""
        sel = torch.nonzero((self.mask & (self.k2.sqrt() + 1.5 < nshell + 1)).flatten()).flatten()
        e = (torch.where(self.kx == 0, 0.5, 1.0) * (u[:3].abs() ** 2).sum(0)).flatten()[sel].cpu().numpy()
        k2 = self.k2.flatten()[sel].cpu().numpy()
        ik = (np.sqrt(k2) + 1.5).astype(np.int64)
        ek, dk = np.bincount(ik, e, nshell + 1), np.bincount(ik, e * k2, nshell + 1)
        return torch.from_numpy(ek[1:]).to(self.dev), torch.from_numpy(dk[1:]).to(self.dev)

    def gradient(self, u):
        return torch.stack([torch.stack([self.phys(1j * k * u[i] * self.mask) for k in (self.kx, self.ky, self.kz)])
                            for i in range(3)])

    def nonlinear(self, u, g, dt, nc=0, tau=None):
        """velmax and the terms N of the velocity and the scalars (dt attached by
        a function of velmax on the first stage)"""
        sh = self.shift(g)
        us = torch.where(self.mask, u[:3] * sh, torch.zeros((), device=self.dev, dtype=torch.complex128))
        v = torch.stack([self.phys(us[i]) for i in range(3)])
        velmax = float(v.abs().sum(0).max()) * self.n
        if callable(dt):
            dt = dt(velmax)
        pairs = [v[0] ** 2 - v[1] ** 2, v[0] * v[1], v[2] ** 2 - v[1] ** 2, v[1] * v[2], v[0] * v[2]]
        if tau is not None:
            for q, t in zip(pairs, (tau[0] - tau[3], tau[1], tau[5] - tau[3], tau[4], tau[2])):
                q += t
        p = [self.spec(q) for q in pairs]
        f = torch.where(self.mask, -(dt / 2.0) * sh.conj(), torch.zeros((), device=self.dev, dtype=torch.complex128))
        kx, ky, kz = self.kx, self.ky, self.kz
        out = [f * 1j * (kx * p[0] + kz * p[4] + ky * p[1]), f * 1j * (kx * p[1] + kz * p[3]),
               f * 1j * (kx * p[4] + kz * p[2] + ky * p[3])]
        for i in range(nc):
            ph = torch.where(self.mask, u[3 + i] * sh, torch.zeros((), device=self.dev, dtype=torch.complex128))
            t = v[0] * (1.0 + self.phys(1j * kx * ph)) + v[1] * self.phys(1j * ky * ph) + v[2] * self.phys(1j * kz * ph)
            out.append(f * self.spec(t))
        return dt, torch.stack(out)


def force(box, un, kf, ekinf):
    if kf:
        ek = box.shells(un, kf + 1)[0]
        ratio = torch.sqrt(ekinf / torch.where(ek > 0, ek, torch.ones_like(ek)))
        ratio[0] = 0.0
        ik = (box.k2.sqrt() + 1.5).long()
        scale = torch.where(ik <= kf, ratio[(ik - 1).clamp(max=kf)], torch.ones_like(box.k2))
        un[:3] *= scale


def factors(box, nu, dt, nc):
    f = torch.exp(-nu * box.k2 * dt)
    return torch.stack([f] * 3 + [f ** (1.0 / pr) for pr in [1.0, 0.7, 2.0][:nc]])


def exact_steps(case, seed):
    n, nc, rk4 = case["n"], case.get("nc", 0), case["kind"] == "rk4"
    if n > 512:
        return None
    u0, d = spectrum_field(n, 3 + nc, seed, case["prec"], float(case.get("kpeak", 3)))
    box, nu = Box(n), viscosity(n, d)
    un = box.dense(u0)
    kf = case["kf"]
    ekinf = box.shells(un, kf + 1)[0] if kf else None
    net = unpack(torch.from_numpy(theta0(seed, 0.05)).to(box.dev).double()) if case["kind"] == "les" else None
    part = None
    if case["kind"] == "particles":
        part = torch.zeros((9, case["np"]), device=box.dev, dtype=torch.float64)
        part[:3] = torch.from_numpy(np.random.default_rng(seed).random((3, case["np"])) * n).to(box.dev)
    dt_of, dt = (lambda vm: CFL / vm), None
    for g in shifts(seed, case["steps"]):
        if part is not None:
            advance_particles(box, un, g, part, dt)
        u = un
        stages = (0, 1, 0, 1) if rk4 else (0, 1)
        for k, st in enumerate(stages):
            gs = g[3 * st:3 * st + 3]
            tau = closure_stress(box, u, gs, net) if net is not None else None
            dt, N = box.nonlinear(u, gs, dt_of if k == 0 else dt, nc, tau)
            if k == 0:
                F = factors(box, nu, dt, nc)
            if rk4:
                if k == 0:
                    u1, u = F * (un + N / 3.0), F * (un + N)
                elif k < 3:
                    u1, u = u1 + 2.0 * N / 3.0, un + N * (1.0 if k == 1 else 2.0)
                else:
                    u = u1 + N / 3.0
            elif k == 0:
                u, un = F * (un + 2.0 * N), F * (un + N)
            else:
                u = un + N
            u = box.project(u * box.mask)
        u[:, 0, 0, 0] = 0.0
        un = u
        force(box, un, kf, ekinf)
    out = [box.columns(un)]
    return out + [part] if part is not None else out


def advance_particles(box, un, g, pp, dt):
    n = box.n
    if dt is not None:
        f = dt / (2.0 * math.pi) * n * 0.5
        pp[6:9] = pp[:3] + f * pp[3:6]
        pp[:3] = pp[6:9] + f * pp[3:6]
    eig = [6.0 / (4.0 + 2.0 * torch.cos(2.0 * math.pi * k / n)) for k in (box.kx, box.ky, box.kz)]
    sp = box.shift(g[:3]) * eig[0] * eig[1] * eig[2] * box.mask
    c = torch.stack([box.phys(un[i] * sp) for i in range(3)]).reshape(3, -1)
    w, at = [], []
    for j in range(3):
        x = torch.remainder(pp[j] - (float(g[j]) + 1.0), float(n))
        ib = x.floor()
        p = x - ib
        m = 1.0 - p
        w0, w3 = m ** 3 / 6.0, p ** 3 / 6.0
        w1 = 2.0 / 3.0 + 0.5 * p * (m * m - 1.0)
        w.append([w0, w1, 1.0 - w0 - w1 - w3, w3])
        at.append([torch.remainder(ib.long() + i - 1, n) for i in range(4)])
    pp[3:6] = 0.0
    for iy in range(4):
        for iz in range(4):
            for ix in range(4):
                pp[3:6] += w[0][ix] * w[1][iy] * w[2][iz] * c[:, (at[1][iy] * n + at[2][iz]) * n + at[0][ix]]
    if dt is not None:
        pp[:3] = pp[6:9] + f * pp[3:6]


def invariants(A, n):
    """the closure's 5 invariants and 4 x 6 tensor basis of the gradient A"""
    def mm(a, b):
        return torch.stack([torch.stack([sum(a[i, k] * b[k, j] for k in range(3)) for j in range(3)]) for i in range(3)])

    def tr(m):
        return m[0, 0] + m[1, 1] + m[2, 2]

    t3 = tr(A) / 3.0
    S, W = 0.5 * (A + A.transpose(0, 1)), 0.5 * (A - A.transpose(0, 1))
    for i in range(3):
        S[i, i] = S[i, i] - t3
    S2, W2 = mm(S, S), mm(W, W)
    s2, w2 = tr(S2), tr(W2)
    q = torch.clamp(s2 - w2, min=1e-30)
    lam = torch.stack([s2 / q, w2 / q, tr(mm(S2, S)) / q ** 1.5, tr(mm(W2, S)) / q ** 1.5, tr(mm(W2, S2)) / q ** 2])
    d2, sw = (2.0 * math.pi / n) ** 2, mm(S, W) - mm(W, S)
    eye = torch.eye(3, device=A.device, dtype=A.dtype)
    return lam, torch.stack([torch.stack([d2 * t for t in (torch.sqrt(2.0 * s2) * S[i, j], sw[i, j],
                                                           S2[i, j] - s2 / 3.0 * eye[i, j],
                                                           W2[i, j] - w2 / 3.0 * eye[i, j])]) for i, j in SYM], dim=1)


def unpack(theta):
    out, o = {}, 0
    for name, shape in THETA:
        c = math.prod(shape)
        out[name] = theta[o:o + c].reshape(shape)
        o += c
    return out


def network(p, x0, lam, T):
    """x0 (B, 135), lam (B, 5), T (B, 4, 6) -> stress (B, 6)"""
    h = torch.cat([lam, torch.tanh(x0 @ p["W0"].T + p["b0"])], 1)
    for i in "123":
        h = torch.tanh(h @ p["W" + i].T + p["b" + i])
    g = h @ p["W4"].T + p["b4"]
    return sum(g[:, i:i + 1] * T[:, i] for i in range(4))


def neighbours(lam):
    """the 135 convolution inputs of every point: (P, 135)"""
    return torch.stack([torch.roll(lam[c], (-dy, -dz, -dx), (0, 1, 2)).flatten() for c in range(5)
                        for dy in (-1, 0, 1) for dz in (-1, 0, 1) for dx in (-1, 0, 1)], 1)


def closure_stress(box, u, g, net):
    lam, T = invariants(box.gradient(u[:3] * box.shift(g)), box.n)
    x0, n = neighbours(lam), box.n
    lp, Tp = lam.reshape(5, -1).T, T.reshape(4, 6, -1).permute(2, 0, 1)
    out = torch.cat([network(net, x0[i:i + (1 << 18)], lp[i:i + (1 << 18)], Tp[i:i + (1 << 18)])
                     for i in range(0, n ** 3, 1 << 18)])
    return out.T.reshape(6, n, n, n)


def box_filter(f, r):
    w = [(0.5 if abs(o) == r // 2 else 1.0) / r for o in range(-(r // 2), r // 2 + 1)]
    for ax in range(3):
        n = f.shape[ax]
        at = torch.arange(0, n, r, device=f.device)
        f = sum(wi * f.index_select(ax, torch.remainder(at + o - r // 2, n)) for o, wi in enumerate(w))
    return f


def exact_snapshot(case, seed):
    nf, n = case["nf"], case["n"]
    r, fine, coarse = nf // n, Box(nf), Box(n)
    u0, _ = spectrum_field(nf, 3, seed, case["prec"], float(case.get("kpeak", 3)))
    ud = fine.dense(u0)
    v = [fine.phys(ud[i]) for i in range(3)]
    ub = [box_filter(x, r) for x in v]
    tau = torch.stack([box_filter(v[i] * v[j], r) - ub[i] * ub[j] for i, j in SYM])
    t3 = (tau[0] + tau[3] + tau[5]) / 3.0
    for c in (0, 3, 5):
        tau[c] -= t3
    uc = torch.stack([coarse.spec(x) for x in ub])
    lam, T = invariants(coarse.gradient(uc), n)
    return [coarse.columns(uc), tau, lam, T.reshape(24, n, n, n)]


M64 = (1 << 64) - 1


def splitmix(x):
    """splitmix64's finaliser (Steele, Lea and Flood 2014) on uint64 arrays"""
    x = x + np.uint64(0x9E3779B97F4A7C15)
    x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return x ^ (x >> np.uint64(31))


def exact_train(case, seed):
    dev, n, s, B = device(), case["n"], case["snaps"], case["batch"]
    lam, basis, tau = (t.double() for t in store(case, seed))
    P = n ** 3
    cw = torch.tensor(CW, device=dev, dtype=torch.float64)
    sigma2 = float((cw[None, :, None] * tau.reshape(s, 6, P) ** 2).sum() / (s * P))
    theta = torch.from_numpy(theta0(seed, 1.0)).to(dev).double()
    m, v, losses = torch.zeros_like(theta), torch.zeros_like(theta), []
    off = [(dy, dz, dx) for dy in (-1, 0, 1) for dz in (-1, 0, 1) for dx in (-1, 0, 1)]
    for t in range(1, case["steps"] + 1):
        with np.errstate(over="ignore"):
            base = splitmix(np.array([((17 + seed) * 0xD1B54A32D192ED03 + t) & M64], np.uint64))
            idx = splitmix(base + np.arange(B, dtype=np.uint64)) % np.uint64(s * P)
        idx = torch.from_numpy(idx.astype(np.int64)).to(dev)
        sn, p = idx // P, idx % P
        y, z, x = p // (n * n), (p // n) % n, p % n
        x0 = torch.stack([lam[sn, c, (y + a) % n, (z + b) % n, (x + d) % n] for c in range(5) for a, b, d in off], 1)
        th = theta.clone().requires_grad_(True)
        e = network(unpack(th), x0, lam[sn, :, y, z, x], basis[sn, :, :, y, z, x]) - tau[sn, :, y, z, x]
        loss = (cw * e * e).sum() / (B * sigma2)
        g, = torch.autograd.grad(loss, th)
        losses.append(float(loss.detach()))
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        theta = theta - 1e-3 * (m / (1.0 - 0.9 ** t)) / (torch.sqrt(v / (1.0 - 0.999 ** t)) + 1e-8)
    return [theta, np.array(losses)]


def exact_stats(case, seed):
    n = case["n"]
    u0, d = spectrum_field(n, 3, seed, case["prec"], float(case.get("kpeak", 3)))
    box, nu = Box(n), viscosity(n, d)
    u = box.dense(u0)
    ek, dk = box.shells(u, n)
    mom = []
    for f in (box.phys(1j * box.kx * u[0] * box.mask), box.phys(1j * box.kz * u[2] * box.mask)):
        mom.append(torch.stack([(f ** p).mean() for p in range(1, 9)]))
    # the first moment of a gradient is zero: its value is rounding
    for q in mom:
        q[0] = 0.0
    return {"ek": ek, "dk": 2.0 * nu * dk, "tke": float(ek.sum()), "eps": float(2.0 * nu * dk.sum()), "dudx": mom[0],
            "dwdz": mom[1]}


def exact(case, seed):
    with torch.no_grad():
        if case["kind"] in ("rk2", "rk4", "particles", "les"):
            return exact_steps(case, seed)
        if case["kind"] == "snapshot":
            return exact_snapshot(case, seed)
        if case["kind"] == "stats":
            return exact_stats(case, seed)
    return exact_train(case, seed)
