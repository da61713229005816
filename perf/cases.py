"""What the framework is timed on: whole calls through its public entry
points, over the range of sizes and options that its programs use.

A case is a dict of plain values.  `prepare` makes what a program holds before
the call (a configured system, a batch, a network with its training set, or
device arrays), `run` is one pass, `work` the bytes and operations that pass
cannot do without, `exact` the same outputs in 64 bits from plain torch.

Kinds of case:
  run        steps of one system, then the field, unwrapped positions and
             forces read back, as a program does between two dumps
  batch      steps of several independent systems advanced together
  surrogate  blocks of K steps advanced by the trained network
  train      steps of the network's trainer on a resident training set
  gradient   the gradient of a field on device arrays, without allocation
"""
import ctypes
import math
import os

import numpy as np
import torch

import phafd_amd as P

PI = 3.141592          # the wavevectors' pi
LJ = (1.122462048, 1.0, 1.0)
SKIN, DT = 0.5, 1e-3
CHAIN = dict(r0=1.0, kbond=100.0, kbend=10.0, drag=1.0)
HARMONIC = (1.0, 20.0)
ROD = dict(bondlength=1.0, zeta_para=1.0, zeta_perp=2.0, bending=2.0, temp=0.2)
NOISE_TEMP = 1e-3      # the noise's temperature; temp * gamma stays 1
EPSILON = {"gaussian": 1.0, "ljish": 1.0, "linear": 0.2}
STYLE = {"gaussian": 0, "ljish": 1, "linear": 3}
CUT = {"gaussian": 3.0, "ljish": 2.5, "linear": 3.0}
RANGE = {"gaussian": 1.0, "ljish": 2.5, "linear": 2.0}   # nucleus width: how far a bead reaches
NETWORK = os.path.join(os.path.dirname(os.path.abspath(P.__file__)), "data", "surrogate_gaussian128_k10.npz")


def system(nx, ny, nz, chains, beads, steps, coupling="gaussian", fp32=False, integrator="chain", noise=False,
           phi0=0.4, var=0.04, chi=2.5):
    return dict(kind="run", nx=nx, ny=ny, nz=nz, chains=chains, beads=beads, steps=steps, coupling=coupling,
                fp32=fp32, integrator=integrator, noise=noise, phi0=phi0, var=var, chi=chi)


def listed():
    return [
        # the smallest call: one step of a small box, as the quick check of an installation or a
        # program that looks at the system after every step makes it
        dict(system(32, 32, 32, 6, 20, 1, phi0=0.5, var=0.02, chi=3.0), name="step_32"),
        # the 64^3 reference case (20 chains of 50): a run whose launches count, not its bytes
        dict(system(64, 64, 64, 20, 50, 50, phi0=0.5, var=0.02, chi=3.0), name="run_64"),
        # the example script's coupling with thermal noise, one replica of the batched workload's size
        dict(system(128, 128, 128, 499, 101, 40, coupling="linear", noise=True, chi=2.2), name="run_128_noise"),
        # bead-rod polymers (atom/semiflexible) in a small box
        dict(system(64, 64, 64, 81, 25, 20, coupling="linear", integrator="rod", phi0=0.5, var=0.02, chi=3.0),
             name="rods_64"),
        # a flat box with three different axis lengths, free beads under drag pushed apart by the
        # harmonic style, the wide coupling
        dict(system(512, 128, 32, 3001, 21, 30, coupling="ljish", integrator="drag"), name="slab_drag"),
        # the production case: 256^3, 500 000 beads, FP64
        dict(system(256, 256, 256, 5000, 100, 50), name="run_256"),
        # the same with FP32 fields and compensated sums
        dict(system(256, 256, 256, 5000, 100, 50, fp32=True), name="run_256_fp32"),
        # the largest box: 512^3, 2M beads, the wide LJish coupling, FP32 fields
        dict(system(512, 512, 512, 19968, 100, 20, coupling="ljish", fp32=True), name="run_512_fp32"),
        # replicas of 128^3 with 10k to 60k beads each, advanced together
        dict(kind="batch", n=128, members=10, steps=10, name="batch_128"),
        # the surrogate with its deployed network on the production case, 2 blocks of 10 steps
        dict(kind="surrogate", n=256, chains=5000, beads=100, K=10, steps=20, name="surrogate_256"),
        # training that network: minibatches of 8 samples of 64^3
        dict(kind="train", nx=64, ny=64, nz=64, samples=16, batch=8, steps=3, name="train_64"),
        # the gradient entry point for callers that hold device arrays
        dict(kind="gradient", nx=128, ny=128, nz=128, name="gradient_128"),
    ]


def draw(rng):
    def log2(lo, hi):
        return 2 ** rng.randint(int(math.log2(lo)), int(math.log2(hi)))

    kind = rng.choice(["run"] * 8 + ["batch", "surrogate", "train", "gradient"])
    if kind == "run":
        nx, ny, nz = log2(32, 512), log2(32, 512), log2(32, 512)
        while nx * ny * nz > 1 << 24:
            nx, ny, nz = max(32, nx // 2), max(32, ny // 2), max(32, nz // 2)
        points = nx * ny * nz
        coupling = rng.choice(["gaussian", "gaussian", "ljish", "linear"])
        integrator = rng.choice(["chain", "chain", "chain", "drag", "rod"])
        beads = rng.randint(20, 130) if integrator != "rod" else rng.randint(10, 40)
        density = math.exp(rng.uniform(math.log(0.003), math.log(0.03)))
        chains = max(3, int(density * points / beads)) | 1
        if integrator == "rod":
            chains = min(chains, 2001)
        steps = max(1, min(60, int(4e7 / points * rng.uniform(0.5, 1.5))))
        fp32, noise = rng.random() < 0.35, rng.random() < 0.25
        return system(nx, ny, nz, chains, beads, steps, coupling, fp32, integrator, noise,
                      round(rng.uniform(0.35, 0.5), 3), 0.04, round(rng.uniform(2.0, 2.4 if noise else 3.2), 3))
    if kind == "batch":
        return dict(kind="batch", n=rng.choice([32, 64, 64, 128]), members=rng.randint(2, 9), steps=rng.randint(4, 12))
    if kind == "surrogate":
        n = rng.choice([64, 128, 128])
        return dict(kind="surrogate", n=n, chains=int(n ** 3 * rng.uniform(0.005, 0.03) / 50) | 1, beads=50, K=10,
                    steps=10 * rng.randint(1, 4))
    if kind == "train":
        return dict(kind="train", nx=64 * rng.randint(1, 2), ny=32 * rng.randint(1, 3), nz=4 * rng.randint(2, 18),
                    samples=rng.randint(4, 12), batch=rng.randint(2, 8), steps=rng.randint(1, 3))
    while True:
        nx, ny, nz = log2(16, 256), log2(16, 256), log2(16, 256)
        if (nx // 2 + 1) * ny * nz <= 1308672:
            return dict(kind="gradient", nx=nx, ny=ny, nz=nz)


# ------------------------------------------------------------------ inputs
def _noisy(shape, phi0, var, seed):
    """phi0 + uniform noise of total width var."""
    d = "cuda" if torch.cuda.is_available() else "cpu"
    g = torch.Generator(device=d).manual_seed(int(seed))
    return phi0 + var * (torch.rand(shape, generator=g, device=d, dtype=torch.float64) - 0.5)


def _chains(nchains, nbeads, n, seed):
    """Random-walk chains, no two beads closer than a bond: drawn in a box of at
    most 128 a side and repeated along the axes of a larger one.  Coordinates run on past the faces."""
    sub = [min(v, 128) for v in n]
    copies = [a // b for a, b in zip(n, sub)]
    total = copies[0] * copies[1] * copies[2]
    per = max(1, nchains // total)
    xyz, _ = P.ic_random_chains(per, nbeads, 1.0, 1.0, [0, 0, 0], [float(v) for v in sub], int(seed))
    shift = np.array([(i, j, k) for i in range(copies[0]) for j in range(copies[1]) for k in range(copies[2])], float)
    xyz = (xyz[None] + (shift * np.array(sub, float))[:, None, :]).reshape(-1, 3)
    return np.ascontiguousarray(xyz), per * total


def _inputs(case, seed):
    n = (case["nx"], case["ny"], case["nz"])
    phi = _noisy(n[::-1], case["phi0"], case["var"], seed)
    xyz, nchains = _chains(case["chains"], case["beads"], n, seed + 1)
    return phi, xyz, nchains


def _configure(s, case, phi, xyz, nchains):
    nb = case["beads"]
    s.set_field(P.PHI, phi.cpu().numpy())
    mol = np.repeat(np.arange(nchains, dtype=np.int32), nb)
    s.set_atoms(xyz, np.zeros(len(xyz), np.int32), mols=mol)
    ip = s.pair_gridatom(STYLE[case["coupling"]], CUT[case["coupling"]])
    s.pair_coeff(ip, 0, EPSILON[case["coupling"]], 0.1, RANGE[case["coupling"]])
    if case["integrator"] == "drag":
        s.pair_harmoniccut(*HARMONIC)
    else:
        s.pair_ljcut(*LJ)
    temp = NOISE_TEMP if case["noise"] else 1.0
    s.fix_conjugate(5678, 1.0, temp, 1.0, 1.0 / temp, P.NOISE_DEVICE if case["noise"] else P.NOISE_OFF)
    s.fix_floryhuggins(1.0, 1.0, case["chi"])
    st = np.arange(nchains, dtype=np.int32) * nb
    if case["integrator"] == "chain":
        s.fix_chain(st, st + nb, **CHAIN)
    elif case["integrator"] == "rod":
        s.fix_semiflexible(0, st, st + nb, 99, **ROD)
    else:
        s.fix_drag(st, st + nb, 1.0)
    s.neighbor(SKIN)


class Host:
    """Host buffers that a program reads a system's state into after each call."""

    def __init__(self, s, natoms):
        self.phi = torch.empty(s.shape, dtype=torch.float64, pin_memory=torch.cuda.is_available())
        self.x = np.empty((natoms, 3))
        self.F = np.empty((natoms, 3))

    def read(self, s, wrapped):
        L, dp = P.lib(), ctypes.POINTER(ctypes.c_double)
        x = self.x.ctypes.data_as(dp)
        for rc in (L.phafd_hip_get_field(s.h, P.PHI, ctypes.cast(self.phi.data_ptr(), dp)),
                   L.phafd_hip_get_atoms(s.h, x if wrapped else None, None if wrapped else x, None),
                   L.phafd_hip_get_forces(s.h, self.F.ctypes.data_as(dp))):
            if rc < 0:
                raise RuntimeError(L.phafd_hip_last_error(s.h).decode())
        return {"phi": self.phi, "x": self.x, "F": self.F}


def _batch_members(case, seed):
    """Replicas of one grid with their own chi, mean composition and bead count."""
    rng = np.random.default_rng(case["members"])   # the members' make-up is the case's, their state the seed's
    n = case["n"]
    out = []
    for i in range(case["members"]):
        nb = int(rng.integers(50, 201)) if n >= 64 else 20
        beads = n ** 3 * math.exp(rng.uniform(math.log(0.005), math.log(0.03)))
        m = system(n, n, n, max(1, int(beads / nb)), nb, case["steps"], phi0=float(rng.uniform(0.3, 0.5)),
                   chi=float(rng.uniform(2.0, 4.0)))
        out.append((m,) + _inputs(m, seed * 1000 + i))
    return out


def _new_system(case):
    n = (case["nx"], case["ny"], case["nz"])
    return P.System(*n, [0, 0, 0], [float(v) for v in n], zghost=P.ZGHOST_PERIODIC,
                    precision=P.FP32 if case["fp32"] else P.FP64)


def _surrogate_case(case):
    n = case["n"]
    return system(n, n, n, case["chains"], case["beads"], case["steps"])


def _train_data(case, seed):
    """Samples with the scales and smoothness of the network's inputs and targets."""
    g = torch.Generator().manual_seed(int(seed))
    shape = (case["nz"], case["ny"], case["nx"])
    for _ in range(case["samples"]):
        x = torch.randn((4,) + shape, generator=g)
        x = (x + x.roll(1, 1) + x.roll(1, 2) + x.roll(1, 3)) * 0.5
        x[1:3] = x[1:3].clamp(min=0) * 0.3
        x[3] = x[3].mean()
        y = 0.5 * x[0] - x[2] + x[1] * x[0] + 0.1 * torch.randn(shape, generator=g)
        yield x.numpy(), y.contiguous().numpy()


def prepare(case, seed):
    kind = case["kind"]
    st = {"kind": kind, "case": case}
    if kind in ("run", "surrogate"):
        c = case if kind == "run" else _surrogate_case(case)
        phi, xyz, nchains = _inputs(c, seed)
        s = _new_system(c)
        _configure(s, c, phi, xyz, nchains)
        s.setup(DT)
        st.update(s=s, host=Host(s, len(xyz)))
        if kind == "surrogate":
            st["net"] = P.UNet(seed=1)
            st["net"].load(NETWORK)
            st["tol"] = float(np.load(NETWORK)["tol"][0])
            s.run_surrogate(st["net"], 0, case["K"], st["tol"])
    elif kind == "batch":
        n = case["n"]
        b = P.Batch(n, n, n, [0, 0, 0], [float(n)] * 3, case["members"], zghost=P.ZGHOST_PERIODIC)
        hosts = []
        for i, (m, phi, xyz, nchains) in enumerate(_batch_members(case, seed)):
            _configure(b.member(i), m, phi, xyz, nchains)
            hosts.append(Host(b.member(i), len(xyz)))
        b.setup(DT)
        st.update(b=b, hosts=hosts)
    elif kind == "train":
        net = P.UNet(seed=int(seed) & 0xFFFF)
        net.data_alloc(case["nx"], case["ny"], case["nz"], case["samples"])
        for i, (x, y) in enumerate(_train_data(case, seed)):
            net.data_put(i, x, y)
        st["net"] = net
    else:
        shape = (case["nz"], case["ny"], case["nx"])
        st["phi"] = _noisy(shape, 0.4, 0.04, seed)
        st["out"] = [torch.empty_like(st["phi"]) for _ in range(3)]
        st["period"] = (ctypes.c_double * 3)(*[float(v) for v in shape[::-1]])
    return st


def run(st):
    case, kind = st["case"], st["kind"]
    if kind == "run":
        st["s"].run(case["steps"])
        return st["host"].read(st["s"], case["integrator"] == "drag")
    if kind == "batch":
        st["b"].run(case["steps"])
        return [h.read(st["b"].member(i), False) for i, h in enumerate(st["hosts"])]
    if kind == "surrogate":
        st["s"].run_surrogate(st["net"], case["steps"], case["K"], st["tol"])
        return st["host"].read(st["s"], False)
    if kind == "train":
        losses = st["net"].train(case["steps"], case["batch"], case["samples"], 1e-3)
        return {"losses": losses, "params": st["net"].get_params()}
    v = ctypes.c_void_p
    rc = P.lib().phafd_hip_gradphi_noalloc(case["nx"], case["ny"], case["nz"], st["period"], v(st["phi"].data_ptr()),
                                           *[v(g.data_ptr()) for g in st["out"]],
                                           v(torch.cuda.current_stream().cuda_stream))
    if rc < 0:
        raise RuntimeError(P.lib().phafd_hip_last_error(None).decode())
    return st["out"]


# -------------------------------------------------------------------- work
CONV_FLOPS = 2 * (4 * 16 * 27 + 16 * 16 * 27 * 2 + 16 + (16 * 32 * 27 + 32 * 32 * 27 + 32 * 16) / 8
                  + (32 * 64 * 27 + 64 * 32) / 64)   # the network, per grid point


def _step_work(points, beads, size, coupling):
    """One step: the field read and written, each bead's position read and written and its force
    written; two transforms there and back, three of the gradient, the coupling's and the chains' arithmetic."""
    pairs = 4.19 * RANGE[coupling] ** 3 * beads
    return (2.0 * size * points + 72.0 * beads,
            5 * 2.5 * points * math.log2(points) + 40.0 * points + 40.0 * pairs + 300.0 * beads)


def work(case):
    kind = case["kind"]
    if kind == "run":
        b, f = _step_work(case["nx"] * case["ny"] * case["nz"], case["chains"] * case["beads"],
                          4 if case["fp32"] else 8, case["coupling"])
        return {"bytes": b * case["steps"], "flops": f * case["steps"]}
    if kind == "batch":
        points = case["n"] ** 3
        b, f = _step_work(points, 0.0135 * points, 8, "gaussian")
        return {"bytes": b * case["steps"] * case["members"], "flops": f * case["steps"] * case["members"]}
    if kind == "surrogate":
        points, beads, blocks = case["n"] ** 3, case["chains"] * case["beads"], case["steps"] // case["K"]
        return {"bytes": 16.0 * points * blocks + 72.0 * beads * case["steps"],
                "flops": (CONV_FLOPS + 5 * 2.5 * math.log2(points)) * points * blocks + 400.0 * beads * case["steps"]}
    if kind == "train":
        points, n = case["nx"] * case["ny"] * case["nz"], case["batch"] * case["steps"]
        return {"bytes": 20.0 * points * n, "flops": 3 * CONV_FLOPS * points * n}
    points = case["nx"] * case["ny"] * case["nz"]
    return {"bytes": 32.0 * points, "flops": 4 * 2.5 * points * math.log2(points)}


# ------------------------------------------------------------------- exact
def _wave(n, period, dev):
    i = torch.arange(n, device=dev)
    return torch.where(i > n // 2, i - n, i).double() * (2 * PI / period)


class Exact:
    """The same time step in plain 64-bit torch: transforms of the whole field, every bead's
    grid points one offset at a time, bead pairs from a cell grid."""

    def __init__(self, case, phi, xyz, nchains):
        self.c, self.phi = case, phi.clone()
        self.dev = dev = phi.device
        self.n = [case["nx"], case["ny"], case["nz"]]
        self.L = torch.tensor([float(v) for v in self.n], device=dev, dtype=torch.float64)
        self.u = torch.from_numpy(xyz).to(dev)
        self.nchains = nchains
        nx, ny, nz = self.n
        kx = torch.arange(nx // 2 + 1, device=dev).double() * (2 * PI / nx)
        self.k = (kx.view(1, 1, -1), _wave(ny, ny, dev).view(1, -1, 1), _wave(nz, nz, dev).view(-1, 1, 1))
        self.q2 = self.k[0] ** 2 + self.k[1] ** 2 + self.k[2] ** 2
        self.pairs = None

    def inverse(self, s):
        """Of a half spectrum that need not be Hermitian: the kx = 0 and kx = Nx/2 bins give their real part."""
        t = torch.fft.ifft2(s, dim=(0, 1))
        t[..., 0].imag.zero_()
        t[..., -1].imag.zero_()
        return torch.fft.irfft(t, n=self.n[0], dim=2)

    def couple(self, grad):
        c, dev = self.c, self.dev
        nx, ny, nz = self.n
        w = RANGE[c["coupling"]]
        x = torch.remainder(self.u, self.L)
        base = torch.floor(x)
        frac = x - base
        bi = base.long()
        F = torch.zeros_like(x)
        mu = torch.zeros(nx * ny * nz, device=dev, dtype=torch.float64)
        phi, g = self.phi.reshape(-1), [v.reshape(-1) for v in grad]
        reach = int(math.ceil(w))
        e05 = math.exp(-0.5)
        for dz in range(-reach, reach + 2):
            for dy in range(-reach, reach + 2):
                for dx in range(-reach, reach + 2):
                    d = torch.tensor([dx, dy, dz], device=dev, dtype=torch.float64) - frac
                    r2 = (d * d).sum(1) / (w * w)
                    at = torch.nonzero(r2 < 1).reshape(-1)
                    if not len(at):
                        continue
                    r2 = r2[at]
                    b = bi[at]
                    p = (((b[:, 2] + dz) % nz) * ny + (b[:, 1] + dy) % ny) * nx + (b[:, 0] + dx) % nx
                    if c["coupling"] == "gaussian":
                        e = (torch.exp(-r2 / 2) - e05) / e05
                    else:
                        e = torch.exp(1 - 1 / (1 - r2))
                    e = e * EPSILON[c["coupling"]] * (-1 if c["coupling"] == "linear" else 2 * (phi[p] - 0.1))
                    mu.index_add_(0, p, e)
                    for k in range(3):
                        F[at, k] -= g[k][p] * e
        return mu.view(nz, ny, nx), F

    def near(self, cut):
        """Bead pairs (i, j) closer than cut plus half a unit, from cells at least that wide."""
        dev, N = self.dev, len(self.u)
        wide = cut + 0.5
        m = [max(1, int(v // wide)) for v in self.n]
        x = torch.remainder(self.u, self.L)
        ci = torch.minimum((x / self.L * torch.tensor(m, device=dev)).long(), torch.tensor(m, device=dev) - 1)
        cell = (ci[:, 2] * m[1] + ci[:, 1]) * m[0] + ci[:, 0]
        order = torch.argsort(cell)
        count = torch.bincount(cell, minlength=m[0] * m[1] * m[2])
        start = torch.cumsum(count, 0) - count
        most = int(count.max())
        me = torch.arange(N, device=dev)
        I, J = [], []
        for dz in (-1, 0, 1):
            for dy in (-1, 0, 1):
                for dx in (-1, 0, 1):
                    o = ((ci[:, 2] + dz) % m[2] * m[1] + (ci[:, 1] + dy) % m[1]) * m[0] + (ci[:, 0] + dx) % m[0]
                    for k in range(most):
                        ok = k < count[o]
                        j = order[torch.clamp(start[o] + k, max=N - 1)]
                        d = self.u - self.u[j]
                        d = d - self.L * torch.round(d / self.L)
                        at = torch.nonzero(ok & (j > me) & ((d * d).sum(1) < wide * wide)).reshape(-1)
                        I.append(me[at])
                        J.append(j[at])
        self.pairs, self.at = (torch.cat(I), torch.cat(J)), self.u.clone()

    def bead_pairs(self):
        soft = self.c["integrator"] == "drag"
        cut = HARMONIC[0] if soft else LJ[0]
        if self.pairs is None or float(((self.u - self.at) ** 2).sum(1).max()) > 0.2 ** 2:
            self.near(cut)
        i, j = self.pairs
        d = self.u[i] - self.u[j]
        d = d - self.L * torch.round(d / self.L)
        r2 = (d * d).sum(1)
        if soft:
            r = torch.sqrt(r2)
            f = torch.where(r < cut, -HARMONIC[1] * (r - cut) / r, torch.zeros_like(r))
        else:
            s6 = 1 / r2 ** 3
            f = torch.where(r2 < cut * cut, s6 * (48 * s6 - 24) / r2, torch.zeros_like(r2))
        F = torch.zeros_like(self.u)
        F.index_add_(0, i, d * f[:, None])
        F.index_add_(0, j, -d * f[:, None])
        return F

    def bonded(self):
        u = self.u.view(self.nchains, -1, 3)
        b = u[:, 1:] - u[:, :-1]
        r = b.norm(dim=2, keepdim=True)
        F = torch.zeros_like(u)
        t = -CHAIN["kbond"] * (r - CHAIN["r0"]) / r * b
        F[:, 1:] += t
        F[:, :-1] -= t
        if b.shape[1] > 1:
            a, c = b[:, :-1], b[:, 1:]
            ra, rc = r[:, :-1], r[:, 1:]
            cs = (a * c).sum(2, keepdim=True) / (ra * rc)
            ga = CHAIN["kbend"] * (c / (ra * rc) - cs * a / ra ** 2)
            gc = CHAIN["kbend"] * (a / (ra * rc) - cs * c / rc ** 2)
            F[:, :-2] -= ga
            F[:, 1:-1] += ga - gc
            F[:, 2:] += gc
        return F.reshape(-1, 3)

    def step(self):
        c = self.c
        hat = torch.fft.rfftn(self.phi)
        grad = [self.inverse(1j * k * hat) for k in self.k]
        mu, F = self.couple(grad)
        del grad
        self.F = F = F + self.bead_pairs()
        for _ in range(2):
            self.u = self.u + (0.5 * DT) * ((F + self.bonded()) * CHAIN["drag"] if c["integrator"] == "chain" else F)
        p = self.phi
        p = torch.where(p <= 0, -p, torch.where(p >= 1, 2 - p, p))
        mu = mu + torch.log(p / (1 - p)) + c["chi"] * (1 - 2 * p)
        hat = hat - DT * self.q2 * (torch.fft.rfftn(mu) + self.q2 * hat)
        self.phi = self.inverse(hat)

    def run(self, steps):
        for _ in range(steps):
            self.step()
        x = None if self.c["integrator"] == "drag" else self.u
        return {"phi": self.phi, "x": x, "F": self.F}


def exact(case, seed):
    kind = case["kind"]
    if kind == "run":
        # no plain restatement of the rods' and the noise's random streams; the largest box takes too long
        if case["noise"] or case["integrator"] == "rod" or case["nx"] * case["ny"] * case["nz"] > 1 << 24:
            return None
        return Exact(case, *_inputs(case, seed)).run(case["steps"])
    if kind == "batch":
        return [Exact(*m).run(case["steps"]) for m in _batch_members(case, seed)]
    if kind == "gradient":
        n = (case["nx"], case["ny"], case["nz"])
        c = system(*n, 1, 1, 1)
        e = Exact(c, _noisy(n[::-1], 0.4, 0.04, seed), np.zeros((1, 3)), 1)
        hat = torch.fft.rfftn(e.phi)
        return [e.inverse(1j * k * hat) for k in e.k]
    return None   # a trained network in 16 bits, and its trainer's own random draws
