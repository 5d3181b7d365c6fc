"""The work a user of this framework has it do, as cases that can be timed.

A case is one call sequence through the public entry points: advance the spins
of a System or of a ReplicaBatch by a number of steps (or sweeps, samples, or
one trajectory gradient) and read the resulting state back, as a simulation
script does between two measurements.  Sizes are those of the repository's own
workloads (cubic 16^3 and 64^3, pyrochlore 32^3 x 16, dipolar pyrochlore
16^3 x 16, 64 uneven SU(3) triangular replicas), with ragged ones beside them.

listed() and draw(rng) give cases, prepare(case, seed) builds what the script
holds before the call, run(state) makes one pass, work(case) counts what the
pass cannot do without, and exact(case, seed) computes the same outputs in
64 bits with plain torch.
"""
from __future__ import annotations

import itertools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "sunny.jl_amd"))

import sunnyhip as sh  # noqa: E402

MU0_MUB2 = 0.6745817653324668  # meV A^3
GOLDEN = 0x9E3779B97F4A7C15    # key increment from one replica to the next
MASK32 = 0xFFFFFFFF


# ---------------------------------------------------------------------------
# Cases

def listed():
    return [
        # a small ragged magnet, as in a notebook: every call is latency
        {"name": "cubic-small-langevin-f64", "kind": "langevin", "model": "cubic", "L1": 6, "L2": 7, "L3": 9, "R": 1,
         "bits": 64, "nsteps": 100, "dt": 0.05, "damping": 0.1, "kT": 0.5},
        # simple cubic 16^3 in plain FP64: thermalisation between two measurements
        {"name": "cubic16-langevin-f64", "kind": "langevin", "model": "cubic", "L1": 16, "L2": 16, "L3": 16, "R": 1,
         "bits": 64, "nsteps": 200, "dt": 0.05, "damping": 0.1, "kT": 0.5},
        # the same magnet's energy-conserving dynamics at the default tolerance
        {"name": "cubic16-midpoint-f64", "kind": "midpoint", "model": "cubic", "L1": 16, "L2": 16, "L3": 16, "R": 1,
         "bits": 64, "nsteps": 50, "dt": 0.05, "tol": 1e-12, "kT": 0.5},
        # one large pyrochlore (18 bonds a site) in FP64, dims that divide nothing
        {"name": "pyro-ragged-langevin-f64", "kind": "langevin", "model": "pyro", "L1": 31, "L2": 26, "L3": 29, "R": 1,
         "bits": 64, "nsteps": 400, "dt": 0.025, "damping": 0.2, "kT": 0.3},
        # the headline model as a batch of FP32 replicas: thermalisation
        {"name": "pyro32-batch-langevin-f32", "kind": "langevin", "model": "pyro", "L1": 32, "L2": 32, "L3": 32, "R": 8,
         "bits": 32, "nsteps": 500, "dt": 0.025, "damping": 0.5, "kT": 0.3},
        # and its energy-conserving dynamics
        {"name": "pyro32-batch-midpoint-f32", "kind": "midpoint", "model": "pyro", "L1": 32, "L2": 32, "L3": 32, "R": 8,
         "bits": 32, "nsteps": 100, "dt": 0.025, "tol": 1e-5, "kT": 0.3},
        # long-range dipolar interactions: one replica, and a batch sharing the tensor
        {"name": "ewald16-langevin-f32", "kind": "langevin", "model": "dipolar", "L1": 16, "L2": 16, "L3": 16, "R": 1,
         "bits": 32, "nsteps": 200, "dt": 0.025, "damping": 0.2, "kT": 0.3},
        {"name": "ewald16-batch-langevin-f32", "kind": "langevin", "model": "dipolar", "L1": 16, "L2": 16, "L3": 16,
         "R": 32, "bits": 32, "nsteps": 200, "dt": 0.025, "damping": 0.2, "kT": 0.3},
        # parallel tempering's shape: 64 SU(3) replicas of uneven size at 64 temperatures
        {"name": "sun3-batch-langevin-f32", "kind": "langevin", "model": "sun3", "L1": 32, "L2": 256, "L3": 1, "R": 64,
         "bits": 32, "nsteps": 1000, "dt": 0.02, "damping": 0.5, "kT": 0.1},
        # a fit's gradient through a trajectory: record forward, sweep backward
        {"name": "cubic64-adjoint-f64", "kind": "adjoint", "model": "cubic", "L1": 64, "L2": 64, "L3": 64, "R": 1,
         "bits": 64, "nsteps": 100, "dt": 0.05, "tol": 1e-12, "kT": 0.5},
        # dynamical structure factor: trajectories sampled into correlations
        {"name": "cubic20-correlations-f64", "kind": "correlations", "model": "cubic", "L1": 20, "L2": 20, "L3": 20,
         "R": 1, "bits": 64, "nsteps": 3, "dt": 0.05, "tol": 1e-12, "kT": 0.3, "nomega": 26, "omega_max": 6.0},
        # Metropolis sweeps of the headline model
        {"name": "pyro32-metropolis-f32", "kind": "metropolis", "model": "pyro", "L1": 32, "L2": 32, "L3": 32, "R": 1,
         "bits": 32, "nsteps": 50, "kT": 0.3},
    ]


def _logint(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["small", "cubic-mid", "pyro64", "pyro-batch", "pyro-batch-mid", "dipolar", "dipolar-batch",
                       "sun3", "adjoint", "correlations", "metropolis"])

    def dims(lo, hi):
        return {"L1": rng.randint(lo, hi), "L2": rng.randint(lo, hi), "L3": rng.randint(lo, hi)}

    if kind == "small":
        L = _logint(rng, 4, 20)
        return {"kind": "langevin", "model": "cubic", "L1": L, "L2": rng.randint(4, 20), "L3": rng.randint(4, 20),
                "R": 1, "bits": 64, "nsteps": rng.randint(50, 300), "dt": 0.05, "damping": 0.1, "kT": 0.5}
    if kind == "cubic-mid":
        return {"kind": "midpoint", "model": "cubic", **dims(6, 20), "R": 1, "bits": 64,
                "nsteps": rng.randint(20, 80), "dt": 0.05, "tol": 1e-12, "kT": 0.5}
    if kind == "pyro64":
        return {"kind": "langevin", "model": "pyro", "L1": _logint(rng, 5, 32), "L2": _logint(rng, 5, 32),
                "L3": _logint(rng, 5, 32), "R": 1, "bits": 64, "nsteps": rng.randint(100, 400), "dt": 0.025,
                "damping": 0.2, "kT": 0.3}
    if kind == "pyro-batch":
        return {"kind": "langevin", "model": "pyro", **dims(12, 32), "R": _logint(rng, 1, 8), "bits": 32,
                "nsteps": rng.randint(150, 500), "dt": 0.025, "damping": 0.5, "kT": 0.3}
    if kind == "pyro-batch-mid":
        return {"kind": "midpoint", "model": "pyro", **dims(12, 32), "R": _logint(rng, 1, 8), "bits": 32,
                "nsteps": rng.randint(30, 100), "dt": 0.025, "tol": 1e-5, "kT": 0.3}
    if kind == "dipolar":
        return {"kind": "langevin", "model": "dipolar", **dims(6, 16), "R": 1, "bits": 32,
                "nsteps": rng.randint(80, 250), "dt": 0.025, "damping": 0.2, "kT": 0.3}
    if kind == "dipolar-batch":
        L = rng.choice([8, 10, 12, 15, 16])
        return {"kind": "langevin", "model": "dipolar", "L1": L, "L2": L, "L3": rng.choice([8, 9, 12, 16]),
                "R": _logint(rng, 2, 32), "bits": 32, "nsteps": rng.randint(60, 150), "dt": 0.025, "damping": 0.2,
                "kT": 0.3}
    if kind == "sun3":
        lo = _logint(rng, 16, 64)
        return {"kind": "langevin", "model": "sun3", "L1": lo, "L2": rng.randint(lo + 32, 256), "L3": 1,
                "R": rng.randint(8, 64), "bits": 32, "nsteps": rng.randint(300, 1000), "dt": 0.02, "damping": 0.5,
                "kT": 0.1}
    if kind == "adjoint":
        return {"kind": "adjoint", "model": "cubic", "L1": 8 * rng.randint(2, 8), "L2": 8 * rng.randint(2, 8),
                "L3": 8 * rng.randint(2, 8), "R": 1, "bits": 64, "nsteps": rng.randint(30, 100), "dt": 0.05,
                "tol": 1e-12, "kT": 0.5}
    if kind == "correlations":
        return {"kind": "correlations", "model": "cubic", "L1": 2 * rng.randint(4, 10), "L2": rng.randint(8, 20),
                "L3": rng.randint(8, 20), "R": 1, "bits": 64, "nsteps": rng.randint(1, 3), "dt": 0.05, "tol": 1e-12,
                "kT": 0.3, "nomega": rng.randint(16, 26), "omega_max": 6.0}
    return {"kind": "metropolis", "model": "pyro", **dims(10, 32), "R": 1, "bits": 32, "nsteps": rng.randint(20, 60),
            "kT": 0.3}


# ---------------------------------------------------------------------------
# The models, restated in plain torch (64 bits).  Sites are numbered in the
# framework's order, c1 + L1 (c2 + L2 (c3 + L3 i)), replica after replica.

PYRO_POS = [np.mod((np.array(b) + np.array(t)) / 4.0, 1.0)
            for t in ((0, 0, 0), (0, 2, 2), (2, 0, 2), (2, 2, 0))
            for b in ((0, 0, 0), (3, 1, 2), (1, 2, 3), (2, 3, 1))]

LATTICE = {  # positions, lattice vectors (columns)
    "cubic": ([np.zeros(3)], np.eye(3)),
    "pyro": (PYRO_POS, 10.0 * np.eye(3)),
    "dipolar": (PYRO_POS, 10.0 * np.eye(3)),
    "sun3": ([np.zeros(3)], np.array([[4.0, -2.0, 0.0], [0.0, 2 * math.sqrt(3.0), 0.0], [0.0, 0.0, 6.75]])),
}
NN = 10.0 * math.sqrt(2.0) / 4
SHELLS = {  # (bond length, J)
    "cubic": [(1.0, 1.0)],
    "pyro": [(NN, 1.0), (10.0 * math.sqrt(6.0) / 4, 0.1)],
    "dipolar": [(NN, 0.05)],
    "sun3": [(4.0, -0.24), (4.0 * math.sqrt(3.0), 0.05), (8.0, 0.2)],
}
KAPPA = {"cubic": 1.0, "pyro": 1.5, "dipolar": 3.5, "sun3": 1.0}


def _dims(case):
    """Dims of every replica (the SU(3) batch: sides uniform in L1..L2)."""
    if case["model"] == "sun3":
        r = np.random.default_rng(0)
        return [(int(L), int(L), 1) for L in r.integers(case["L1"], case["L2"] + 1, size=case["R"])]
    return [(case["L1"], case["L2"], case["L3"])] * case["R"]


def _kTs(case):
    """One temperature for all replicas; tempering: geometric up to 2."""
    if case["model"] == "sun3":
        return case["kT"] * (2.0 / case["kT"]) ** (np.arange(case["R"]) / max(1, case["R"] - 1))
    return np.full(case["R"], case["kT"])


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


class _Model:
    """Neighbour tables and couplings of all replicas of a case."""

    def __init__(self, case):
        self.name, self.dev = case["model"], _device()
        self.dims, self.kappa = _dims(case), KAPPA[case["model"]]
        pos, lv = LATTICE[self.name]
        self.pos, self.lv, self.na = pos, lv, len(pos)
        rng = range(-2, 3)
        slots = []  # slots[s][i] = (j, n): neighbour s of sublattice i
        self.J = []
        for d, J in SHELLS[self.name]:
            per = [[(j, n) for j in range(self.na) for n in itertools.product(rng, rng, rng)
                    if abs(np.linalg.norm(lv @ (pos[j] + np.array(n) - pos[i])) - d) < 1e-6] for i in range(self.na)]
            for s in range(len(per[0])):
                slots.append([p[s] for p in per])
                self.J.append(J)
        table, site, rep, off, cache = [], [], [], 0, {}
        for r, L in enumerate(self.dims):
            if L not in cache:
                c = torch.stack(torch.meshgrid(*[torch.arange(x, device=self.dev) for x in L[::-1]], indexing="ij"))
                c3, c2, c1 = (x.reshape(-1) for x in c)
                nc = c1.numel()
                rows = []
                for sl in slots:
                    rows.append(torch.cat([((c1 + n[0]) % L[0]) + L[0] * (((c2 + n[1]) % L[1]) +
                                           L[1] * ((c3 + n[2]) % L[2])) + nc * j for j, n in sl]))
                cache[L] = torch.stack(rows)
            t = cache[L]
            table.append(t + off)
            n = t.shape[1]
            site.append(torch.arange(n, device=self.dev))
            rep.append(torch.full((n,), r, device=self.dev))
            off += n
        self.nbr, self.site, self.rep, self.total = torch.cat(table, 1), torch.cat(site), torch.cat(rep), off
        self.ni = [len(s) for s in site]
        self.axes = None
        if self.name == "pyro":  # local <111> axes: from the tetrahedron's centre to the site
            ax = []
            for i in range(self.na):
                v = [lv @ (pos[j] + np.array(n) - pos[i]) for j in range(self.na) for n in itertools.product(rng, rng, rng)]
                v = [x for x in v if abs(np.linalg.norm(x) - NN) < 1e-6]
                tet = [x for x in v if np.linalg.norm(x - v[0]) < NN + 1e-6]
                ax.append(sum(tet) / np.linalg.norm(sum(tet)))
            nc = [int(np.prod(L)) for L in self.dims]
            self.axes = torch.cat([torch.tensor(np.repeat(np.array(ax), n, axis=0), device=self.dev) for n in nc])
        self.FA = _ewald_tensor(self) if self.name == "dipolar" else None

    def bonds(self, S):
        g = torch.zeros_like(S)
        for row, J in zip(self.nbr, self.J):
            g += J * S[row]
        return g

    def grad(self, S, J=None, D=-0.1):
        """dE/dS at every site."""
        g = self.bonds(S) if J is None else J * sum(S[row] for row in self.nbr)
        if self.name == "cubic":  # D Sz^2 for s = 1: renormalised by 1 - 1/(2s)
            e = torch.zeros(3, device=self.dev, dtype=S.dtype)
            e[2] = 1
            g = g + (2 * D * 0.5) * S * e
        elif self.name == "pyro":  # -0.05 (S.n)^2 for s = 3/2
            g = g + (2 * -0.05 * (2.0 / 3.0)) * (S * self.axes).sum(1, keepdim=True) * self.axes
        elif self.name == "dipolar":
            g = g + _ewald_field(self, S)
        return g


def _ewald_tensor(m):
    """Transformed dipole-dipole tensor of the supercell, [k][3 na][3 na]."""
    L, dev = m.dims[0], m.dev
    sup = torch.tensor(m.lv @ np.diag(L).astype(float), device=dev)
    rec = 2 * math.pi * torch.linalg.inv(sup).T
    V = float(torch.abs(torch.linalg.det(sup)))
    len_s = torch.linalg.norm(sup, dim=0)
    sig = float(len_s.min()) / 4
    c = torch.stack(torch.meshgrid(*[torch.arange(x, device=dev, dtype=torch.float64) for x in L], indexing="ij"), -1)
    cells = c.reshape(-1, 3)
    lv = torch.tensor(m.lv, device=dev)
    pos = torch.tensor(np.array(m.pos), device=dev)
    nmax = [int(math.ceil(8.3 * sig / float(x) + 1)) for x in len_s]
    kcut = 8.3 / sig
    mmax = [int(math.ceil(kcut * float(x) / (2 * math.pi))) for x in len_s]
    ks = []
    for q in itertools.product(*[range(-x, x + 1) for x in mmax]):
        if q > (0, 0, 0):
            k = rec @ torch.tensor(q, device=dev, dtype=torch.float64)
            ks.append(k)
    ks = torch.stack(ks)
    k2 = (ks * ks).sum(1)
    ks, k2 = ks[k2 < kcut * kcut], k2[k2 < kcut * kcut]
    kw = 2 * torch.exp(-sig * sig * k2 / 2) / k2 / V
    kk = (ks[:, :, None] * ks[:, None, :] * kw[:, None, None]).reshape(-1, 9)
    eye = torch.eye(3, device=dev, dtype=torch.float64)
    images = torch.tensor(list(itertools.product(*[range(-x, x + 1) for x in nmax])), device=dev, dtype=torch.float64)
    na, nc = m.na, cells.shape[0]
    FA = None
    for j in range(na):
        col = torch.zeros((na, nc, 3, 3), device=dev, dtype=torch.float64)
        for i in range(na):
            # A(off; i, j) couples mu at (c - off, j) to the potential at (c, i)
            base = (cells + pos[i] - pos[j]) @ lv.T
            A = (torch.cos(base @ ks.T) @ kk).reshape(nc, 3, 3) + eye / (3 * V)
            for im in images:
                d = base + (sup @ im)
                r = torch.linalg.norm(d, dim=1)
                self_ = r < 1e-9
                r = torch.where(self_, torch.ones_like(r), r)
                ok = (r < 8.3 * sig) & ~self_
                x = r / sig
                e = math.sqrt(2 / math.pi) * x * torch.exp(-x * x / 2)
                f = torch.special.erfc(x / math.sqrt(2.0))
                a = torch.where(ok, (f + e) / r ** 3, torch.zeros_like(r)) / (4 * math.pi)
                b = torch.where(ok, (f + e * (1 + x * x / 3)) / r ** 5, torch.zeros_like(r)) * 3 / (4 * math.pi)
                A += a[:, None, None] * eye - b[:, None, None] * d[:, :, None] * d[:, None, :]
                if bool(self_.any()):
                    A[self_] -= eye / (3 * (2 * math.pi) ** 1.5 * sig ** 3)
            col[i] = A
        f = torch.fft.rfftn(MU0_MUB2 * col.reshape(na, *L, 3, 3), dim=(3, 2, 1))
        if FA is None:
            FA = torch.zeros((f[0, :, :, :, 0, 0].numel(), na, 3, na, 3), device=dev, dtype=torch.complex128)
        FA[:, :, :, j, :] = f.reshape(na, -1, 3, 3).permute(1, 0, 2, 3)
    return FA.reshape(FA.shape[0], 3 * na, 3 * na).contiguous()


def _ewald_field(m, S):
    """-g' phi with phi = A * mu, mu = -g S and g = 2."""
    L, R = m.dims[0], len(m.dims)
    mu = -2.0 * S.reshape(R, m.na, L[2], L[1], L[0], 3).permute(0, 1, 5, 4, 3, 2)  # [R][na][3][c1][c2][c3]
    F = torch.fft.rfftn(mu, dim=(5, 4, 3))
    sh_k = F.shape[3:]
    X = F.reshape(R, 3 * m.na, -1).permute(2, 1, 0).contiguous()
    Y = torch.matmul(m.FA, X).permute(2, 1, 0).reshape(R, m.na, 3, *sh_k)
    phi = torch.fft.irfftn(Y, s=(L[2], L[1], L[0]), dim=(5, 4, 3))
    return -2.0 * phi.permute(0, 1, 5, 4, 3, 2).reshape(-1, 3)


def _philox(c, key):
    """Philox4x32-10 of the counters c (four tensors or numbers) under 64-bit keys."""
    k0, k1 = key & MASK32, (key >> 32) & MASK32
    for _ in range(10):
        p0, p1 = 0xD2511F53 * c[0], 0xCD9E8D57 * c[2]
        c = [((p1 >> 32) & MASK32) ^ c[1] ^ k0, p1 & MASK32, ((p0 >> 32) & MASK32) ^ c[3] ^ k1, p0 & MASK32]
        k0, k1 = (k0 + 0x9E3779B9) & MASK32, (k1 + 0xBB67AE85) & MASK32
    return c


def _normals(m, noise_seed, step, n):
    """n standard normals a site: [total][n]."""
    keys = torch.tensor([_signed(noise_seed + r * GOLDEN) for r in range(len(m.dims))], device=m.dev)[m.rep]
    out = []
    for blk in range((n + 3) // 4):
        z = torch.zeros_like(m.site)
        c = _philox([m.site, z + blk, z + (step & MASK32), z + (step >> 32)], keys)
        for a, b in ((c[0], c[1]), (c[2], c[3])):
            r = torch.sqrt(-2 * torch.log((a.double() + 1) / 4294967296.0))
            t = 2 * math.pi * (b.double() / 4294967296.0)
            out += [r * torch.cos(t), r * torch.sin(t)]
    return torch.stack(out[:n], 1)


def _signed(x):
    x &= (1 << 64) - 1
    return x - (1 << 64) if x >> 63 else x


def _unit(S, kappa):
    return S * (kappa / torch.linalg.norm(S, dim=1, keepdim=True))


def _rhs(S, g, dt, lam):
    v = dt * g if lam == 0 else dt * g - dt * lam * torch.linalg.cross(S, g)
    return -torch.linalg.cross(S, v)


def _heun(m, S, xi, dt, lam):
    """One stochastic Heun step of classical dipoles."""
    d1 = _rhs(S, m.grad(S), dt, lam) - torch.linalg.cross(S, xi)
    Sp = _unit(S + d1, m.kappa)
    d2 = _rhs(Sp, m.grad(Sp), dt, lam) - torch.linalg.cross(Sp, xi)
    return _unit(S + (d1 + d2) / 2, m.kappa)


def _midpoint(m, S, dt, iters, **couplings):
    """One spherical midpoint step, iterated to convergence."""
    S2 = S
    for _ in range(iters):
        h = _unit((S + S2) / 2, m.kappa)
        new = S + _rhs(h, m.grad(h, **couplings), dt, 0.0)
        done = not new.requires_grad and bool(torch.linalg.norm(new - S2) <= 3e-15 * math.sqrt(m.total))
        S2 = new
        if done:
            break
    return _unit(S2, m.kappa)


SPIN1 = (np.array([[0, 1, 0], [1, 0, 1], [0, 1, 0]]) / math.sqrt(2.0),
         np.array([[0, -1j, 0], [1j, 0, -1j], [0, 1j, 0]]) / math.sqrt(2.0), np.diag([1.0, 0.0, -1.0]))


def _sun_heun(m, Z, zeta, dt, lam):
    """One stochastic Heun step of SU(3) coherent states (D Sz^2, D = 2.2)."""
    ops = [torch.tensor(np.array(o, complex), device=m.dev) for o in SPIN1]
    lam_on = 2.2 * (ops[2] @ ops[2])

    def rhs(Z):
        SZ = [Z @ o.T for o in ops]
        g = m.bonds(torch.stack([(Z.conj() * x).sum(1).real for x in SZ], 1))
        v = zeta + dt * (1j + lam) * (Z @ lam_on.T + sum(g[:, a:a + 1] * SZ[a] for a in range(3)))
        return -(v - Z * ((Z.conj() * v).sum(1, keepdim=True) / (Z.conj() * Z).sum(1, keepdim=True)))

    def unit(Z):
        return Z / torch.sqrt((Z.abs() ** 2).sum(1, keepdim=True))

    d1 = rhs(Z)
    d2 = rhs(unit(Z + d1))
    return unit(Z + (d1 + d2) / 2)


def _start(m, case, seed):
    """A thermalised state: random spins (the cubic antiferromagnet: its
    ordered state, tilted at random) relaxed by strongly damped Langevin steps."""
    gen = torch.Generator(device=m.dev)
    gen.manual_seed(int(seed))

    def randn(*shape):
        return torch.randn(*shape, generator=gen, device=m.dev, dtype=torch.float64)

    kT = torch.tensor(_kTs(case), device=m.dev)[m.rep][:, None]
    if m.name == "sun3":
        Z = torch.complex(randn(m.total, 3), randn(m.total, 3))
        Z = Z / torch.sqrt((Z.abs() ** 2).sum(1, keepdim=True))
        for _ in range(20):
            zeta = torch.sqrt(2 * 0.02 * 0.5 * kT) * torch.complex(randn(m.total, 3), randn(m.total, 3)) / math.sqrt(2.0)
            Z = _sun_heun(m, Z, zeta, 0.02, 0.5)
        return Z
    S = randn(m.total, 3)
    if m.name == "cubic":
        L = m.dims[0]
        c = m.site
        sign = 1 - 2.0 * (((c % L[0]) + (c // L[0]) % L[1] + c // (L[0] * L[1])) % 2)
        S = 0.4 * S + sign[:, None] * randn(1, 3)
    S = _unit(S, m.kappa)
    dt, relax = 0.05 / m.kappa, 60 if m.total < 200000 else 20
    if m.name == "dipolar":  # dipolar fields change this state little
        return S
    for _ in range(relax):
        S = _heun(m, S, torch.sqrt(2 * dt * 1.0 * kT) * randn(m.total, 3), dt, 1.0)
    return S


def _noise_seed(seed):
    return (int(seed) * 0x2545F4914F6CDD1D + 0x123456789) & ((1 << 62) - 1)


def _target(case, seed):
    """Structure factor that the trajectory is fitted to, on the 8^3 grid."""
    return np.random.default_rng(seed + 1).uniform(0.5, 1.5, (8, 8, 8))


# ---------------------------------------------------------------------------
# What a script holds before the call

def _system(case, dims, seed):
    bits = case["bits"]
    if case["model"] == "cubic":
        return sh.workloads.cubic_model(dims=dims, seed=seed, precision=bits, params=case["kind"] == "adjoint", J=1.0,
                                        D=-0.1)
    if case["model"] == "pyro":
        return sh.workloads.pyrochlore_model(dims=dims, seed=seed, precision=bits)
    if case["model"] == "dipolar":
        return sh.workloads.pyrochlore_model(dims=dims, J1=0.05, J2=0.0, A=0.0, s=3.5, seed=seed, precision=bits,
                                             dipolar=True, mu0_muB2=MU0_MUB2, demag=1 / 3)
    return sh.workloads.triangular_sun_model(L1=dims[0], L2=dims[1], seed=seed, precision=bits)


def prepare(case, seed):
    # the starting state needs no long-range field (see _start): no tensor either
    m = _Model(dict(case, model="pyro") if case["model"] == "dipolar" else case)
    m.name, m.kappa = case["model"], KAPPA[case["model"]]
    start = _start(m, case, seed).cpu().numpy()
    first, systems, off = {}, [], 0
    for r, L in enumerate(_dims(case)):
        if L not in first:
            first[L] = _system(case, L, seed)
            s = first[L]
        else:
            s = sh.clone_system(first[L], seed=seed + r)
        n = s.nsites
        x = start[off:off + n]
        s.set_state_flat(**({"coh": x} if case["model"] == "sun3" else {"dip": x}))
        s.noise_seed = _noise_seed(seed)
        systems.append(s)
        off += n
    st = {"case": case, "systems": systems, "sys": systems[0]}
    if case["R"] > 1:
        st["sys"] = sh.ReplicaBatch(systems, precision=case["bits"])
        # where the script gathers the replicas' states, in the precision of the run
        width, dtype = (3, np.complex64) if case["model"] == "sun3" else (3, np.float32)
        st["out"] = np.zeros((off, width), dtype)
        st["kTs"] = _kTs(case)
    if case["kind"] == "langevin":
        st["integrator"] = sh.Langevin(case["dt"], damping=case["damping"], kT=case["kT"])
    elif case["kind"] == "midpoint":
        st["integrator"] = sh.ImplicitMidpoint(case["dt"], tol=case["tol"])
    elif case["kind"] == "adjoint":
        st["integrator"] = sh.ImplicitMidpoint(case["dt"], tol=case["tol"])
        st["start"], st["target"], st["dims"] = start, _target(case, seed), _dims(case)[0]
    elif case["kind"] == "correlations":
        st["sc"] = sh.SampledCorrelations(st["sys"], energies=np.linspace(0.0, case["omega_max"], case["nomega"]),
                                          dt=case["dt"], tol=case["tol"])
    else:
        st["integrator"] = sh.LocalSampler(kT=case["kT"], propose=sh.propose_delta(0.3))
    sh.energy(st["sys"])  # the device copy exists, as after any earlier call
    return st


# ---------------------------------------------------------------------------
# One pass

def run(state):
    case, s = state["case"], state["sys"]
    if case["kind"] == "adjoint":
        s.set_state_flat(dip=state["start"])  # every gradient of a fit starts from the same spins
        L, grad, dLdS0 = sh.midpoint_gradient(
            s, state["integrator"], case["nsteps"], ["J", "D"],
            lambda S: sh.structure_factor_loss(S, state["dims"], state["target"], 8), checkpoint_every=25)
        return {"loss": L, "grad": grad, "dLdS0": dLdS0}
    if case["kind"] == "correlations":
        for _ in range(case["nsteps"]):
            sh.add_sample_(state["sc"], s)
        return {"data": state["sc"].data, "dipoles": s.dipoles_flat()}
    if case["R"] == 1:
        acc = sh.step_(s, state["integrator"], nsteps=case["nsteps"])
        x = s.dipoles_flat()
        if case["kind"] == "metropolis":
            return {"dipoles": x.astype(np.float32), "accepted": acc}
        return x if case["bits"] == 64 else x.astype(np.float32)
    sh.step_(s, state["integrator"], nsteps=case["nsteps"],
             **({"kTs": state["kTs"]} if case["kind"] == "langevin" else {}))
    s.sync_to_systems()
    out, off = state["out"], 0
    for x in state["systems"]:
        out[off:off + x.nsites] = x.coherents_flat() if case["model"] == "sun3" else x.dipoles_flat()
        off += x.nsites
    return out


def _sites(case):
    return sum(L[0] * L[1] * L[2] for L in _dims(case)) * len(LATTICE[case["model"]][0])


def work(case):
    """Each step reads the state and writes the next one (a midpoint step and
    a Metropolis sweep too); the field costs six operations a bond, twice a
    Heun step and about eight times a midpoint step at the default tolerance
    (four at 1e-5)."""
    n, bonds = _sites(case), sum({"cubic": [6], "pyro": [6, 12], "dipolar": [6], "sun3": [6, 6, 6]}[case["model"]])
    width = (6 if case["model"] == "sun3" else 3) * case["bits"] // 8
    evals = 2 if case["kind"] == "langevin" else 1 if case["kind"] == "metropolis" else 4 if case["bits"] == 32 else 8
    steps = case["nsteps"]
    if case["kind"] == "correlations":
        steps *= math.ceil(math.pi / (case["dt"] * case["omega_max"])) * (case["nomega"] - 1)
    nbytes, flops = 2.0 * n * width * steps, n * steps * evals * (6.0 * bonds + 60)
    if case["kind"] == "adjoint":
        nbytes, flops = 3 * nbytes, 4 * flops  # forward, the segments again, the reverse sweep
    if case["model"] == "dipolar":  # per field: the tensor once, the transforms, one complex product a wavevector
        L = _dims(case)[0]
        nc, nk = L[0] * L[1] * L[2], (L[0] // 2 + 1) * L[1] * L[2]
        nbytes += 2.0 * steps * nk * 48 * 48 * 8
        flops += 2.0 * steps * case["R"] * (8.0 * nk * 48 * 48 + 2 * 48 * 2.5 * nc * math.log2(nc))
    if case["kind"] == "correlations":
        nbytes += case["nsteps"] * 16.0 * n * 6 * 2 * (case["nomega"] - 1)
    return {"bytes": nbytes, "flops": flops}


# ---------------------------------------------------------------------------
# The same outputs in 64 bits

def exact(case, seed):
    if case["kind"] == "metropolis":
        return None  # accepted moves, not a computed number
    m = _Model(case)
    m0 = m if case["model"] != "dipolar" else None
    if m0 is None:
        m0 = _Model(dict(case, model="pyro"))
        m0.name, m0.kappa = "dipolar", KAPPA["dipolar"]
    S = _start(m0, case, seed)
    if case["kind"] == "langevin":
        kT = torch.tensor(_kTs(case), device=m.dev)[m.rep][:, None]
        scale = torch.sqrt(2 * case["dt"] * case["damping"] * kT)
        for k in range(case["nsteps"]):
            if m.name == "sun3":
                n = _normals(m, _noise_seed(seed), k, 6) * (scale / math.sqrt(2.0))
                S = _sun_heun(m, S, torch.complex(n[:, 0::2].contiguous(), n[:, 1::2].contiguous()), case["dt"],
                              case["damping"])
            else:
                S = _heun(m, S, scale * _normals(m, _noise_seed(seed), k, 3), case["dt"], case["damping"])
        return S.cpu().numpy()
    if case["kind"] == "midpoint":
        for _ in range(case["nsteps"]):
            S = _midpoint(m, S, case["dt"], 60)
        return S.cpu().numpy()
    if case["kind"] == "adjoint":
        return _exact_gradient(m, case, seed, S)
    return _exact_correlations(m, case, S)


def _exact_gradient(m, case, seed, S0):
    """Reverse-mode derivative of the trajectory, one step at a time: each
    step is iterated to its fixed point and, from there, sixteen more times
    on the tape."""
    J = torch.tensor(1.0, device=m.dev, dtype=torch.float64)
    D = torch.tensor(-0.1, device=m.dev, dtype=torch.float64)
    states = [S0]
    for _ in range(case["nsteps"]):
        states.append(_midpoint(m, states[-1], case["dt"], 60))
    L, dims = None, _dims(case)[0]
    S = states[-1].clone().requires_grad_(True)
    B = S.reshape(dims[2] // 8, 8, dims[1] // 8, 8, dims[0] // 8, 8, 3).sum(dim=(0, 2, 4))
    Sq = (torch.fft.ifftn(B.to(torch.complex128), dim=(0, 1, 2)) * 512).abs().square().sum(-1) / m.total
    L = (Sq - torch.tensor(_target(case, seed), device=m.dev)).square().mean()
    lam = torch.autograd.grad(L, S)[0]
    dJ = dD = 0.0
    for x in reversed(states[:-1]):
        with torch.no_grad():
            S2 = x
            for _ in range(40):
                h = _unit((x + S2) / 2, m.kappa)
                S2 = x + _rhs(h, m.grad(h), case["dt"], 0.0)
        a, j, d = x.clone().requires_grad_(True), J.clone().requires_grad_(True), D.clone().requires_grad_(True)
        for _ in range(16):
            h = _unit((a + S2) / 2, m.kappa)
            S2 = a + _rhs(h, m.grad(h, J=j, D=d), case["dt"], 0.0)
        lam, gj, gd = torch.autograd.grad(_unit(S2, m.kappa), (a, j, d), lam)
        dJ, dD = dJ + float(gj), dD + float(gd)
    return {"loss": float(L.detach()), "grad": np.array([dJ, dD]), "dLdS0": lam.cpu().numpy()}


def _exact_correlations(m, case, S):
    """Trajectory snapshots of g S, transformed over the lattice and time with
    zero padding, windowed by cos^2, averaged over samples."""
    T, pairs = 2 * (case["nomega"] - 1), [(2, 2), (1, 2), (0, 2), (1, 1), (0, 1), (0, 0)]
    period = math.ceil(math.pi / (case["dt"] * case["omega_max"]))
    dt = 2 * math.pi / (case["omega_max"] / (case["nomega"] - 1) * period * T)
    L = m.dims[0]
    lag = np.abs(np.rint(np.fft.fftfreq(T, 1.0 / T)))
    contrib = T // 2 + 1 - lag
    contrib[contrib == 0] = np.inf
    window = torch.tensor(np.cos(np.pi * np.arange(T) / T) ** 2 / contrib, device=m.dev)
    mean = 0
    for n in range(case["nsteps"]):
        buf = torch.zeros((3, *L, T), device=m.dev, dtype=torch.complex128)
        for k in range(T // 2 + 1):
            for _ in range(period if k else 0):
                S = _midpoint(m, S, dt, 60)
            buf[..., k] = 2.0 * S.reshape(L[2], L[1], L[0], 3).permute(3, 2, 1, 0)
        F = torch.fft.fft(torch.fft.ifftn(buf, dim=(1, 2, 3)) * math.sqrt(m.total), dim=4)
        c = torch.stack([F[a].conj() * F[b] for a, b in pairs])
        c = torch.fft.fft(torch.fft.ifft(c, dim=4) * window, dim=4)
        mean = mean + (c - mean) / (n + 1)
    return {"data": mean.reshape(6, 1, 1, *L, T).cpu().numpy(), "dipoles": S.cpu().numpy()}
