"""The workloads this engine is timed on, as a program calls it.

Every case is a call sequence of a driver: an engine or an ensemble with its
parameters and its state resident on the GPU (`prepare`), and one block of
steps with what the program takes from it (`run`).  Lattices, potentials and
time steps are those of the repository's benchmark, workloads and tests, and
the lengths between them that the engine supports.  `exact` restates each
block in plain FP64 torch.
"""
import math

import numpy as np
import torch

from libcugpe_amd import adjoint as A
from libcugpe_amd import engine as E

LENGTHS = (8, 12, 16, 24, 32, 48, 64, 96, 128, 192, 256, 512)
PREC = {"c64": E.C64, "c128": E.C128}
DT = 0.02        # step of the uniform-lattice workloads
A_SCAT = 0.008   # scattering length of the uniform-lattice workloads
MOST = 8.0 * 134217728  # bytes of one state array times steps of the largest listed case: 512^3 complex64


def listed():
    return [
        # a loop that takes one step per call on a small lattice (a driver
        # watching every step; the tests' sizes): latency and launches
        {"name": "rt step 16x24x32 c128", "kind": "rt", "nx": 16, "ny": 24, "nz": 32, "prec": "c128", "nt": 1},
        # blocks of steps on the smallest cube of the benchmark's size table
        {"name": "rt 32 c64", "kind": "rt", "nx": 32, "ny": 32, "nz": 32, "prec": "c64", "nt": 50},
        # an elongated box with lengths that are not powers of two
        {"name": "rt 96x192x48 c64", "kind": "rt", "nx": 96, "ny": 192, "nz": 48, "prec": "c64", "nt": 20},
        # the headline workload: turbulence on 256^3 in complex64
        {"name": "rt 256 c64", "kind": "rt", "nx": 256, "ny": 256, "nz": 256, "prec": "c64", "nt": 20},
        # the largest lattice length in all three directions
        {"name": "rt 512 c64", "kind": "rt", "nx": 512, "ny": 512, "nz": 512, "prec": "c64", "nt": 4},
        # a real-time run in complex128 that reports its energy and its
        # vortices after every block of steps
        {"name": "monitor 128 c128", "kind": "monitor", "nx": 128, "ny": 128, "nz": 128, "prec": "c128", "nt": 20},
        # trapped ground state in imaginary time with the chemical potential
        {"name": "ite 32 c128", "kind": "ite", "nx": 32, "ny": 32, "nz": 32, "prec": "c128", "nt": 50},
        # imaginary time with a vortex line pinned, in complex64
        {"name": "ite vortex 128x128x64 c64", "kind": "itev", "nx": 128, "ny": 128, "nz": 64, "prec": "c64", "nt": 20},
        # unitary Fermi gas with quantum friction and a vortex line
        {"name": "qf 128 c64", "kind": "qf", "nx": 128, "ny": 128, "nz": 128, "prec": "c64", "nt": 20},
        # dipolar bosons in a trap, real time
        {"name": "dipolar 96x64x128 c128", "kind": "dipolar", "nx": 96, "ny": 64, "nz": 128, "prec": "c128", "nt": 10},
        # truncated-Wigner ensemble of uneven cubes (the benchmark's mix, a
        # quarter of its lattices): a block of steps and the mean densities
        {"name": "ensemble 24-64 c64", "kind": "ensemble", "count": 64, "prec": "c64", "nt": 50},
        # gradient of an overlap with respect to the potential
        {"name": "adjoint 64 c64", "kind": "adjoint", "nx": 64, "ny": 64, "nz": 64, "prec": "c64", "nt": 32},
    ]


def draw(rng):
    kind = rng.choice(["rt", "rt", "rt", "rt", "monitor", "ite", "itev", "qf", "dipolar", "ensemble", "adjoint"])
    prec = rng.choice(["c64", "c128"])
    if kind in ("monitor",):
        prec = "c128"  # its energies are compared in FP64
    if kind == "ensemble":
        return {"kind": kind, "count": rng.choice([16, 32, 64, 128]), "prec": "c64",
                "nt": int(round(math.exp(rng.uniform(math.log(10), math.log(100)))))}
    # sizes and block lengths up to what the listed cases of the kind cost
    top = {"rt": 27, "monitor": 24, "ite": 22, "itev": 22, "qf": 22, "dipolar": 20, "adjoint": 18}[kind]
    size = rng.uniform(13 if kind == "rt" else 15, top)
    while True:
        n = [rng.choice(LENGTHS) for _ in range(3)]
        if abs(math.log2(n[0] * n[1] * n[2]) - size) < 0.6 and math.log2(n[0] * n[1] * n[2]) <= top:
            break
    nt = int(round(math.exp(rng.uniform(0.0 if kind == "rt" else math.log(5), math.log(50)))))
    es = 8 if prec == "c64" else 16
    points = n[0] * n[1] * n[2]
    nt = max(1, min(nt, int(4 * MOST / (es * points))))
    if kind == "adjoint":
        nt = min(nt, 32)
    return {"kind": kind, "nx": n[0], "ny": n[1], "nz": n[2], "prec": prec, "nt": nt}


# ------------------------------------------------------------------ inputs


def shape_of(case):
    return (case["nx"], case["ny"], case["nz"])


def generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def grids(shape):
    """Lattice coordinates from the centre, one broadcastable FP64 tensor per axis."""
    out = []
    for a, n in enumerate(shape):
        x = torch.arange(n, dtype=torch.float64, device="cuda") - n // 2
        out.append(x.reshape([n if i == a else 1 for i in range(3)]))
    return out


def noise(shape, gen):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)


def vortex_state(shape, seed, lines=8):
    """Near-uniform density, a random phase per site and z-line vortices."""
    g = generator(seed)
    x, y, _ = grids(shape)
    p = torch.rand((lines, 3), generator=g, device="cuda", dtype=torch.float64)
    ph = torch.zeros((shape[0], shape[1], 1), dtype=torch.float64, device="cuda")
    for j in range(lines):
        w = torch.where(p[j, 2] < 0.5, -1.0, 1.0)
        ph = ph + w * torch.atan2(y - (p[j, 1] - 0.5) * shape[1], x - (p[j, 0] - 0.5) * shape[0])
    amp = 1.0 + 0.02 * noise(shape, g).clamp(-3, 3)
    return torch.polar(amp.double(), ph + 0.1 * noise(shape, g))


def trap_state(shape, seed):
    """Gaussian cloud with noise in the middle of the box."""
    g = generator(seed)
    r2 = sum((c / n) ** 2 for c, n in zip(grids(shape), shape))
    return (torch.exp(-r2 * 40.0) * (1 + 0.05 * noise(shape, g))).to(torch.complex128)


def fermi_state(shape, seed):
    """Thomas-Fermi cloud of the friction workload with 1% noise and a vortex line."""
    g = generator(seed)
    x, y, z = (c * (32.0 / n) for c, n in zip(grids(shape), shape))
    rho = (1.0 - 0.5 * (x * x + y * y + 0.25 * z * z) / 25.0).clamp_min(0.0) ** 1.5
    rho = rho * (1 + 0.01 * torch.rand(shape, generator=g, device="cuda", dtype=torch.float64))
    return torch.polar(rho.sqrt(), torch.atan2(y + 0.5 * (32.0 / shape[1]), x + 0.5 * (32.0 / shape[0])).expand(shape))


def setup(case):
    """(interactions, vext, alpha, beta, dt, npart, user parameters, start state) of a case."""
    kind, shape = case["kind"], shape_of(case)
    n = float(np.prod(shape))
    if kind in ("rt", "monitor"):
        return E.CONTACT, E.COSINE, 1.0, 0.0, DT, n, [0.1, 4.0, 0.0, A_SCAT], vortex_state
    if kind == "ite":
        return E.CONTACT, E.HARMONIC, 0.0, 1.0, 2.56e-3, 1.0e4, [12.5 / m for m in shape] + [0.159], trap_state
    if kind == "itev":
        return E.UFG, E.HARMONIC, 0.0, 1.0, 8e-3, 1.0e4, [6.0 / m for m in shape], trap_state
    if kind == "qf":
        om = [w * (32.0 / m) ** 2 for w, m in zip((1.0, 1.0, 0.5), shape)]
        return E.UFG, E.HARMONIC, 1.0, 0.0, 8e-3, 1.0e4, om, fermi_state
    if kind == "dipolar":
        return E.DIPOLAR, E.HARMONIC, 1.0, 0.0, DT, 0.1 * n, [2.0 / m for m in shape] + [0.02, 0.015], trap_state
    raise ValueError(kind)


class DevicePsi:
    """An engine's wave function as torch sees it (the engine's own memory)."""

    def __init__(self, eng):
        self.eng = eng
        self.__cuda_array_interface__ = {"shape": eng.shape, "typestr": "<c8" if eng.precision == E.C64 else "<c16",
                                         "data": (eng.device_psi(), False), "version": 2}


def device_psi(eng):
    return torch.as_tensor(DevicePsi(eng), device="cuda")


ENS_LENGTHS = ((24, 4), (32, 2), (48, 1), (64, 1))  # lattices per 8 of the mix


def ens_state(L, count, seed):
    """Uniform density plus complex noise of variance 1/2 per plane-wave mode."""
    g = generator(seed * 1000 + L)
    b = torch.randn((count, L, L, L, 2), generator=g, device="cuda", dtype=torch.float64) * 0.5
    return 1.0 + torch.fft.ifftn(torch.view_as_complex(b), dim=(1, 2, 3)) * math.sqrt(float(L ** 3))


def adjoint_inputs(case, seed):
    g = generator(seed)
    shape = shape_of(case)

    def smooth():
        k = torch.rand((3, 2), generator=g, device="cuda", dtype=torch.float64)
        return sum((0.3 + k[a, 0]) * torch.cos(2 * math.pi * c / n + 6 * k[a, 1])
                   for a, (c, n) in enumerate(zip(grids(shape), shape)))

    v = 0.2 * smooth() + 0.02 * noise(shape, g)
    psi0 = torch.polar(1 + 0.1 * torch.rand(shape, generator=g, device="cuda", dtype=torch.float64), smooth())
    psit = torch.polar(1 + 0.1 * torch.rand(shape, generator=g, device="cuda", dtype=torch.float64), smooth())
    return v.to(torch.float32 if case["prec"] == "c64" else torch.float64), psi0, psit


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind == "ensemble":
        lat = [(L, case["count"] * c // 8) for L, c in ENS_LENGTHS]
        ens = E.Ensemble([(L,) * 3 for L, c in lat for _ in range(c)], 1.0, 0.0, DT, 1.0, E.CONTACT, E.COSINE, 0,
                         PREC[case["prec"]])
        ens.set_user_params([0.1, 4.0, 0.0, A_SCAT])
        i = 0
        for L, c in lat:
            for psi in ens_state(L, c, seed).cpu().numpy():
                ens.set_psi(i, psi)
                i += 1
        ens.autotune(3)
        return {**st, "ens": ens, "first": [sum(c for _, c in lat[:j]) for j in range(len(lat))]}
    if kind == "adjoint":
        v, psi0, psit = adjoint_inputs(case, seed)
        eng = E.Engine(shape_of(case), 1.0, 0.0, 1e-2, 1.0, E.UFG, E.VARRAY, 0, PREC[case["prec"]])
        return {**st, "eng": eng, "v": v.requires_grad_(True), "psi0": psi0.cpu().numpy(), "psit": psit.cpu().numpy()}
    inter, vext, alpha, beta, dt, npart, up, state = setup(case)
    eng = E.Engine(shape_of(case), alpha, beta, dt, npart, inter, vext, 0, PREC[case["prec"]])
    eng.set_user_params(up)
    if kind == "qf":
        eng.set_quantum_friction_coeff(0.1)
    if kind == "itev":
        eng.set_vortex(0.5, 0.5, 1)
    eng.set_psi(state(shape_of(case), seed).cpu().numpy())
    if kind != "qf":
        eng.normalize_psi()
    eng.synchronize()
    return {**st, "eng": eng, "psi": device_psi(eng)}


def run(state):
    case = state["case"]
    kind, nt = case["kind"], case["nt"]
    if kind == "ensemble":
        # the mean density of every group, and one realisation of each; both
        # carry the precision of the complex64 states
        ens = state["ens"]
        ens.evolve(nt)
        return {"density": [ens.mean_density(g).astype(np.float32) for g in range(len(state["first"]))],
                "psi": [ens.get_psi(i)[0].astype(np.complex64) for i in state["first"]]}
    eng = state["eng"]
    if kind == "adjoint":
        v = state["v"]
        v.grad = None
        loss = A.overlap_loss(v, eng, state["psi0"], state["psit"], nt)
        loss.backward()
        return {"loss": loss.detach(), "grad": v.grad}
    if kind in ("rt", "qf"):
        eng.evolve_qf(nt)
        return state["psi"]
    if kind == "ite":
        mu = eng.evolve_qf(nt, want_mu=True)
        return {"psi": state["psi"], "mu": mu if case["prec"] == "c128" else np.float32(mu)}
    if kind == "itev":
        eng.evolve_vortex(nt)
        return state["psi"]
    if kind == "dipolar":
        eng.evolve_dipolar(nt)
        return state["psi"]
    eng.evolve_qf(nt)
    _, ekin, eint, eext = eng.energy()
    return {"psi": state["psi"], "energy": [ekin, eint, eext], "vortices": eng.detect_vortices(0.05, False)[1]}


def work(case):
    if case["kind"] == "ensemble":
        n = sum(L ** 3 * (case["count"] * c // 8) for L, c in ENS_LENGTHS)
        logn = 16.0
    else:
        n = case["nx"] * case["ny"] * case["nz"]
        logn = math.log2(n)
    s = n * (8 if case["prec"] == "c64" else 16)
    # a step reads and writes the state once and takes four transforms (the
    # predictor's and the corrector's kinetic factors), friction two more, a
    # dipolar step six; a gradient runs the steps twice and three kinetic
    # factors more, and reads and writes the state and its adjoint going back
    steps = {"adjoint": 4.0}.get(case["kind"], 1.0) * case["nt"]
    transforms = {"qf": 6, "dipolar": 6, "adjoint": 14}.get(case["kind"], 4) * case["nt"]
    extra = {"monitor": 2.0}.get(case["kind"], 0.0)  # the energy rescales the state; both queries read it
    return {"bytes": (2.0 * steps + 2.0 * extra) * s, "flops": transforms * 5.0 * n * logn + 60.0 * n * case["nt"]}


# ------------------------------------------------------- FP64 restatement


def wave_numbers(shape):
    out = []
    for a, n in enumerate(shape):
        k = 2 * math.pi * torch.fft.fftfreq(n, dtype=torch.float64, device="cuda")
        out.append(k.reshape([n if i == a else 1 for i in range(3)]))
    return out


def potential(vext, up, shape):
    if vext == E.HARMONIC:
        return sum(0.5 * (c * w) ** 2 for c, w in zip(grids(shape), up))
    return up[0] * sum(torch.cos(2 * math.pi * up[1] * torch.arange(n, dtype=torch.float64, device="cuda") / n)
                       .reshape([n if i == a else 1 for i in range(3)]) for a, n in enumerate(shape))


def mean_field(inter, up, rho):
    if inter == E.UFG:
        return 0.37 * (3 * math.pi ** 2 * rho) ** (2.0 / 3.0) / 2.0
    return 4 * math.pi * up[3] * rho


class Exact:
    def __init__(self, shape, inter, vext, alpha, beta, dt, npart, up, v=None):
        self.inter, self.up, self.beta, self.dt, self.npart = inter, up, beta, dt, npart
        self.gamma = 2.0 if inter == E.UFG else 1.0
        self.c = self.gamma * 0.5 * dt / complex(-beta, alpha)
        self.k2 = sum(k * k for k in wave_numbers(shape))
        self.K = torch.exp(self.c * self.k2 / self.gamma ** 2)
        self.v = potential(vext, up, shape) if v is None else v

    def rho(self, p):
        return self.gamma * (p.real ** 2 + p.imag ** 2)

    def g(self, p):
        return mean_field(self.inter, self.up, self.rho(p))

    def kinetic(self, p):
        return torch.fft.ifftn(self.K * torch.fft.fftn(p, dim=(-3, -2, -1)), dim=(-3, -2, -1))

    def normalize(self, p):
        s = self.rho(p).sum()
        return p * torch.sqrt(self.npart / s), s

    def step(self, p, qf=0.0, pin=None):
        """One predictor-corrector split step; returns psi and the norm sum before the last rescaling."""
        if pin is not None:
            p = pin(p)
        q = 0.0
        if qf:
            w = torch.fft.ifftn(self.k2 * torch.fft.fftn(p)) * (qf / self.gamma)
            q = (p.conj() * w).imag / (self.rho(p) + 1e-12)
        v0 = self.v + self.g(p) + q
        e0 = torch.exp(self.c * v0)
        p3 = self.kinetic(p * e0) * e0
        if self.beta:
            p3, _ = self.normalize(p3)
        v1 = 0.5 * (v0 + self.v + self.g(p3) + q)
        if pin is not None and self.beta:
            p = pin(p)
        w = torch.exp(self.c * v1)
        p = self.kinetic(p * w) * w
        s = None
        if self.beta:
            p, s = self.normalize(p)
        return p, s

    def dipolar_step(self, p, shape):
        kx, ky, kz = wave_numbers(shape)
        k2 = kx * kx + ky * ky + kz * kz
        vpp = 4 * math.pi * (self.up[3] + self.up[4] * (3 * kz * kz / k2.clamp_min(1e-30) - 1))
        vpp[0, 0, 0] = 4 * math.pi * self.up[3]
        for half in range(2):
            vd = torch.fft.ifftn(vpp * torch.fft.fftn(self.rho(p).to(torch.complex128))).real
            p = p * torch.exp(self.c * (self.v + vd))
            if half == 0:
                p = self.kinetic(p)
        return p


def exact(case, seed):
    kind, nt = case["kind"], case["nt"]
    if kind == "ensemble":
        den, one = [], []
        for L, c in ENS_LENGTHS:
            x = Exact((L,) * 3, E.CONTACT, E.COSINE, 1.0, 0.0, DT, 1.0, [0.1, 4.0, 0.0, A_SCAT])
            p = ens_state(L, case["count"] * c // 8, seed)
            for _ in range(nt):
                p, _ = x.step(p)
            den.append(x.rho(p).mean(dim=0).cpu().numpy())
            one.append(p[0].cpu().numpy())
        return {"density": den, "psi": one}
    shape = shape_of(case)
    if kind == "adjoint":
        v, psi0, psit = adjoint_inputs(case, seed)
        v = v.double().requires_grad_(True)
        x = Exact(shape, E.UFG, E.VARRAY, 1.0, 0.0, 1e-2, 1.0, [], v)
        p = psi0
        for _ in range(nt):
            p, _ = x.step(p)
        o = (psit.conj() * p).sum()
        loss = 1.0 - (o.real ** 2 + o.imag ** 2) / ((psit.abs() ** 2).sum() * (psi0.abs() ** 2).sum())
        loss.backward()
        return {"loss": loss.detach(), "grad": v.grad}
    inter, vext, alpha, beta, dt, npart, up, state = setup(case)
    x = Exact(shape, inter, vext, alpha, beta, dt, npart, up)
    p = state(shape, seed)
    if kind != "qf":
        p, _ = x.normalize(p)
    if kind == "dipolar":
        for _ in range(nt):
            p = x.dipolar_step(p, shape)
        return p
    pin = None
    if kind == "itev":
        gx, gy, _ = grids(shape)
        turn = torch.polar(torch.ones((), dtype=torch.float64, device="cuda"), torch.atan2(gx - 0.5, gy - 0.5))
        pin = lambda q: q.abs() * turn  # noqa: E731
    s = None
    for _ in range(nt):
        p, s = x.step(p, qf=0.1 if kind == "qf" else 0.0, pin=pin)
    if kind == "ite":
        return {"psi": p, "mu": float(-0.5 * torch.log(s / npart) / dt)}
    if kind == "monitor":
        p, _ = x.normalize(p)
        rho = x.rho(p)
        n = float(np.prod(shape))
        ekin = (x.k2 * torch.fft.fftn(p).abs() ** 2).sum() / (2.0 * x.gamma * n)
        return {"psi": p, "energy": [float(ekin), float((2 * math.pi * up[3] * rho * rho).sum()),
                                     float((rho * x.v).sum())], "vortices": None}
    return p
