"""The framework's work as its users have it done: whole events, long evolutions, observables, ensembles of events,
gauge fixing, gradients and field exchange with the host, each through the public Python entry points.

``listed`` names the cases, ``draw`` gives more of the same ranges, ``prepare`` makes what a program holds before the
call, ``run`` is one pass, ``work`` the bytes and operations a pass cannot do without, and ``exact`` the same outputs
from plain torch in 64 bits (complex128), written from the lattice formulas without the framework's code.

In ``exact`` a matrix field is a tensor [3, 3, z, y, x] (complex128), a colour vector [8, z, y, x] (float64); links
are a list over the three directions.
"""
from __future__ import annotations

import math

import numpy as np
import torch

LAMBDA, M_EFF = 1.65, 0.1  # regulators of the MV charge, in lattice units
S2 = math.sqrt(2.0)


def listed():
    return [
        # a parameter scan over many tiny events: each call is bound by launches and latency
        {"name": "event_16x16x32", "kind": "event", "nx": 16, "ny": 16, "nz": 32, "driver": 1, "sigma": 4.0, "qs": 0.5,
         "az": 1.0, "bc": 0, "steps": 20},
        # the reference's CPU-sized case in full: a left-moving nucleus, 100 steps, bulk sums every 20
        {"name": "event_32x32x64", "kind": "event", "nx": 32, "ny": 32, "nz": 64, "driver": 1, "sigma": 4.0, "qs": 0.5,
         "az": 1.0, "bc": 0, "steps": 100},
        # an odd lattice with other spacings and periodic z, as a discretisation study has it
        {"name": "event_81x75x125", "kind": "event", "nx": 81, "ny": 75, "nz": 125, "driver": 0, "sigma": 5.0,
         "qs": 0.4, "az": 0.8, "bc": 1, "steps": 40},
        # the collision workload of ordinary size: initial state, 100 steps, bulk sums and the energy-momentum profile
        {"name": "event_64x64x256", "kind": "event", "nx": 64, "ny": 64, "nz": 256, "driver": 0, "sigma": 5.0,
         "qs": 0.8, "az": 1.0, "bc": 0, "steps": 100},
        # the middle of a long evolution between two records, lattice already on the device
        {"name": "evolve_128x128x384", "kind": "evolve", "nx": 128, "ny": 128, "nz": 384, "sigma": 5.0, "qs": 0.8,
         "steps": 8},
        # the same for a production lattice (the largest that three programs can hold at once)
        {"name": "evolve_256x256x512", "kind": "evolve", "nx": 256, "ny": 256, "nz": 512, "sigma": 5.0, "qs": 0.8,
         "steps": 4},
        # every observable of a given configuration, as an analysis of stored fields records them
        {"name": "measure_64x56x96", "kind": "measure", "nx": 64, "ny": 56, "nz": 96, "bc": 0},
        # an ensemble of uneven events advanced together between two records
        {"name": "ensemble_24", "kind": "ensemble", "events": 24, "nmax": 96, "zmax": 384, "steps": 10, "mix": 12345},
        # gauge fixing of a large evolved lattice, ten iterations of the converging update
        {"name": "gauge_128x128x256", "kind": "gauge", "nx": 128, "ny": 128, "nz": 256, "algorithm": "consistent",
         "tol": 0.0, "maxit": 10, "evolved": 10, "fields": False},
        # gauge fixing to a tolerance with the gauge-fixed fields taken to the host
        {"name": "gauge_32x40x64", "kind": "gauge", "nx": 32, "ny": 40, "nz": 64, "algorithm": "consistent",
         "tol": 1e-7, "maxit": 100, "evolved": 20, "fields": True},
        # one optimisation step over the charge density: energy and gradient through 100 steps
        {"name": "gradient_48x48x128", "kind": "gradient", "nx": 48, "ny": 48, "nz": 128, "steps": 100, "ckpt": 20,
         "qs": 0.5, "sigma": 4.0},
        # a host program that owns the fields: in, a few steps, and out again
        {"name": "exchange_48x48x96", "kind": "exchange", "nx": 48, "ny": 48, "nz": 96, "bc": 0, "steps": 10},
    ]


def _smooth(n: int) -> bool:
    """Whether the transforms take this length (factors up to 13)."""
    for p in (2, 3, 5, 7, 11, 13):
        while n % p == 0:
            n //= p
    return n == 1


def _length(rng, lo, hi):
    """A transform length, spread evenly over its logarithm."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    while not _smooth(n):
        n -= 1
    return n


def draw(rng):
    """One more case: the kinds and sizes of ``listed``, odd sizes among them, none larger than its largest."""
    kind = rng.choice(["event", "event", "event", "evolve", "measure", "ensemble", "gauge", "gauge", "gradient", "exchange"])
    if kind == "event":
        nx, ny, nz = _length(rng, 12, 96), _length(rng, 12, 96), _length(rng, 28, 300)
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "driver": rng.choice([0, 1, 2]),
                "sigma": round(rng.uniform(4.0, 6.0), 3), "qs": round(rng.uniform(0.5, 0.8), 4),
                "az": rng.choice([1.0, 1.0, 0.8]), "bc": rng.choice([0, 0, 1]), "steps": rng.choice([20, 40, 60])}
    if kind == "evolve":
        n = rng.choice([96, 128, 160, 192, 200, 225, 256])
        return {"kind": kind, "nx": n, "ny": rng.choice([96, 128, 160, 192, 250]), "nz": _length(rng, 300, 480),
                "sigma": 5.0, "qs": round(rng.uniform(0.7, 0.9), 4), "steps": 4}
    if kind == "measure":
        return {"kind": kind, "nx": rng.randint(5, 72), "ny": rng.randint(5, 72), "nz": rng.randint(8, 96),
                "bc": rng.choice([0, 1])}
    if kind == "ensemble":
        return {"kind": kind, "events": rng.randint(4, 24), "nmax": rng.choice([32, 64, 96]),
                "zmax": rng.choice([128, 256, 384]), "steps": rng.choice([5, 10]), "mix": rng.randint(1, 10 ** 6)}
    if kind == "gauge":
        fields = rng.choice([False, False, True])
        top = 48 if fields else 128
        return {"kind": kind, "nx": _length(rng, 16, top), "ny": _length(rng, 16, top),
                "nz": _length(rng, 24, 72 if fields else 256), "algorithm": rng.choice(["consistent", "consistent", "jacobi"]),
                "tol": 0.0, "maxit": rng.randint(5, 10), "evolved": 10, "fields": fields}
    if kind == "gradient":
        return {"kind": kind, "nx": _length(rng, 16, 48), "ny": _length(rng, 16, 48), "nz": _length(rng, 40, 128),
                "steps": rng.choice([20, 50, 70]), "ckpt": rng.choice([10, 20]), "qs": round(rng.uniform(0.3, 0.8), 4),
                "sigma": 4.0}
    return {"kind": kind, "nx": rng.randint(8, 56), "ny": rng.randint(8, 56), "nz": rng.randint(16, 96),
            "bc": rng.choice([0, 1]), "steps": rng.randint(1, 20)}


# ---- inputs ---------------------------------------------------------------------------------------------------------
def _shape(case):
    return (case["nx"], case["ny"], case["nz"])


def _spacing(case):
    return (1.0, 1.0, case.get("az", 1.0))


def _dt(a):
    return 0.25 * min(a)


def _charges(seed, nx, ny, qs):
    """Gaussian charges of both nuclei on the transverse plane."""
    r = np.random.RandomState(seed % (1 << 31))
    return qs * r.standard_normal((ny, nx, 8)), qs * r.standard_normal((ny, nx, 8))


def _centers(nz):
    return int(0.85 * nz / 2 - 1), int(1.15 * nz / 2 - 1)


def _density(case, seed):
    """The density of a left-moving sheet on the whole lattice (Nz, Ny, Nx, 8)."""
    nx, ny, nz = _shape(case)
    xi, _ = _charges(seed, nx, ny, case["qs"])
    z, s = np.arange(nz), case["sigma"]
    prof = np.exp(-0.5 * ((z - _centers(nz)[0]) / s) ** 2) / math.sqrt(2 * math.pi * s * s)
    return prof[:, None, None, None] * xi[None]


def _events(case, seed):
    """The ensemble's lattices and charges: transverse sizes and lengths up to the case's largest."""
    r = np.random.RandomState(case["mix"])
    got = []
    for k in range(case["events"]):
        n = int(r.choice([m for m in (32, 48, 64, 96) if m <= case["nmax"]]))
        nz = int(r.choice([m for m in (128, 192, 256, 384) if m <= case["zmax"]]))
        got.append(((n, n, nz), float(r.uniform(0.3, 0.8)), seed + 1000 * (k + 1)))
    return got


def _host_fields(case, seed):
    """A random configuration as a host program stores it: links (Nz, Ny, Nx, 3, j, i), E and currents."""
    nx, ny, nz = _shape(case)
    r = np.random.RandomState(seed % (1 << 31))
    al = torch.from_numpy(0.4 * r.standard_normal((8, 3 * nz, ny, nx)))
    U = _exp(al.to(_device()), 1.0).reshape(3, 3, 3, nz, ny, nx).permute(3, 4, 5, 2, 1, 0)
    U = U.contiguous().cpu().numpy()
    E = 0.3 * r.standard_normal((nz, ny, nx, 3, 8))
    J = [0.2 * r.standard_normal((nz, ny, nx, 8)) for _ in range(4)]
    return U, E, J


def _ghosts(f, bc):
    """A host array with the two z ghost layers of the reference layout."""
    lo, hi = (f[-1:], f[:1]) if bc else (f[:1], f[-1:])
    return np.concatenate([lo, f, hi])


class State:
    pass


def _mv(g, case, nz):
    cl, cr = _centers(nz)
    return g.mv_params(LAMBDA, M_EFF, case.get("sigma", 4.0), case.get("sigma", 4.0), cl, cr)


def prepare(case, seed):
    from soerenpragya3dglasma_amd import Glasma, GlasmaBatch
    s, kind = State(), case["kind"]
    s.case = case
    if kind == "ensemble":
        ev = _events(case, seed)
        s.batch = GlasmaBatch([(n, (1.0, 1.0, 1.0), 0.25) for n, _, _ in ev])
        for g, (n, qs, sd) in zip(s.batch.events, ev):
            g.mv_initial_state(0, _mv(g, case, n[2]), *_charges(sd, n[0], n[1], qs))
        return s
    n, a = _shape(case), _spacing(case)
    s.g = g = Glasma(n, a, _dt(a), case.get("bc", 0))
    if kind in ("measure", "exchange"):
        U, E, J = _host_fields(case, seed)
        s.fields = [_ghosts(v, case["bc"]) for v in (U, E, *J)]
        if kind == "measure":
            g.set_fields(*s.fields)
            g.Update(1)  # the records need the half-step links of one step
            del s.fields
    elif kind == "gradient":
        s.mv = _mv(g, case, n[2])
        s.rho = _density(case, seed)
    else:
        s.mv = _mv(g, case, n[2])
        s.xi = _charges(seed, n[0], n[1], case.get("qs", 0.5))
        if kind != "event":
            g.mv_initial_state(0, s.mv, *s.xi)
            if kind == "gauge":
                g.Update(case["evolved"])
    return s


# ---- one pass -------------------------------------------------------------------------------------------------------
def run(s):
    c, kind = s.case, s.case["kind"]
    if kind == "ensemble":
        s.batch.update(c["steps"])
        return {"bulk": [g.bulk_raw() for g in s.batch.events]}
    g = s.g
    if kind == "event":
        g.mv_initial_state(c["driver"], s.mv, *s.xi)
        bulk = []
        for _ in range(c["steps"] // 20):
            g.Update(20)
            bulk.append(g.bulk_raw())
        return {"bulk": bulk, "emt": g.emt_profile(), "energy_map": g.transverse_energy_map()}
    if kind == "evolve":
        g.Update(c["steps"])
        return {"bulk": g.bulk_raw(), "emt": g.emt_profile(), "energy_map": g.transverse_energy_map()}
    if kind == "measure":
        per_z, gmax, grms = g.gauss()
        return {"bulk": g.bulk_raw(), "emt": g.emt_profile(), "gauss": per_z, "gauss_max": gmax, "gauss_rms": grms,
                "fields": g.field_profile(), "currents": g.current_profile(), "energy_map": g.transverse_energy_map()}
    if kind == "gauge":
        g.gauge_reset()
        stats = g.coulomb_gauge_algorithm(c["algorithm"], c["tol"], c["maxit"])
        return {"stats": stats, "fixed": list(g.get_gauge_fixed()) if c["fields"] else []}
    if kind == "gradient":
        e, grad = g.slab_energy_gradient(s.mv, s.rho, c["steps"], c["ckpt"], c["nz"] // 2, 8)
        return {"energy": e, "gradient": grad}
    g.set_fields(*s.fields)
    g.Update(c["steps"])
    return g.get_fields()


def work(case):
    """Bytes and operations of one pass: each field read once and written once per step (U 432, E 192 and four currents
    256 bytes a site), the inputs of each record, and for gauge fixing the links, the transformation and the four
    complex arrays of the Poisson step; operations of the matrix products."""
    kind = case["kind"]
    if kind == "ensemble":
        S = sum(n[0] * n[1] * n[2] for n, _, _ in _events(case, 0))
        return {"bytes": S * (case["steps"] * 1760 + 752), "flops": S * (14e3 * case["steps"] + 2e3)}
    S = case["nx"] * case["ny"] * case["nz"]
    emt, emap, bulk, step = 1056, 624, 752, 1760  # bytes per site
    if kind == "event":
        n = case["steps"]
        return {"bytes": S * (1312 + step * n + bulk * (n // 20) + emt + emap), "flops": S * (14e3 * n + 3e4)}
    if kind == "evolve":
        return {"bytes": S * (step * case["steps"] + bulk + emt + emap), "flops": S * (14e3 * case["steps"] + 1.5e4)}
    if kind == "measure":
        return {"bytes": S * (2 * bulk + emt + emap + 752 + 256), "flops": S * 2e4}
    if kind == "gauge":
        it = case["maxit"] if case["tol"] == 0.0 else 20
        b = it * (432 + 288 + 256) + 1392 + (768 if case["fields"] else 0)
        return {"bytes": S * b, "flops": S * (it * 4e3 + 3e3)}
    if kind == "gradient":
        return {"bytes": S * case["steps"] * (1760 + 880 + 1760), "flops": S * case["steps"] * 4.5e4}
    return {"bytes": S * (1760 + step * case["steps"]), "flops": S * 14e3 * case["steps"]}


# ---- the same in plain torch ----------------------------------------------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _mul(A, B):
    return A[:, 0, None] * B[None, 0] + A[:, 1, None] * B[None, 1] + A[:, 2, None] * B[None, 2]


def _dag(A):
    return A.transpose(0, 1).conj()


def _herm(al):
    """alpha^a t^a with t^a half the Gell-Mann matrices."""
    z, r3 = torch.zeros_like(al[0]), 1.0 / math.sqrt(3.0)

    def c(re, im):
        return 0.5 * torch.complex(re, im)

    rows = [[c(al[2] + r3 * al[7], z), c(al[0], -al[1]), c(al[3], -al[4])],
            [c(al[0], al[1]), c(-al[2] + r3 * al[7], z), c(al[5], -al[6])],
            [c(al[3], al[4]), c(al[5], al[6]), c(-2 * r3 * al[7], z)]]
    return torch.stack([torch.stack(r) for r in rows])


def _components(H):
    """2 tr(t^a H) of a Hermitian H."""
    r3 = 1.0 / math.sqrt(3.0)
    return torch.stack([H[0, 1].real + H[1, 0].real, H[1, 0].imag - H[0, 1].imag, H[0, 0].real - H[1, 1].real,
                        H[0, 2].real + H[2, 0].real, H[2, 0].imag - H[0, 2].imag, H[1, 2].real + H[2, 1].real,
                        H[2, 1].imag - H[1, 2].imag, r3 * (H[0, 0].real + H[1, 1].real - 2 * H[2, 2].real)])


def _proj(V):
    """Re tr(i t^a V)."""
    r3 = 1.0 / math.sqrt(3.0)
    return -0.5 * torch.stack([V[0, 1].imag + V[1, 0].imag, V[0, 1].real - V[1, 0].real, V[0, 0].imag - V[1, 1].imag,
                               V[0, 2].imag + V[2, 0].imag, V[0, 2].real - V[2, 0].real, V[1, 2].imag + V[2, 1].imag,
                               V[1, 2].real - V[2, 1].real, r3 * (V[0, 0].imag + V[1, 1].imag - 2 * V[2, 2].imag)])


def _one(like):
    e = torch.zeros_like(like)
    e[0, 0] = e[1, 1] = e[2, 2] = 1.0
    return e


def _exp(al, c):
    """exp(i c alpha t): the Taylor series of the matrix scaled to a norm below 1/2, squared back."""
    top = abs(c) * float(al.detach().abs().amax()) * math.sqrt(8.0) if al.numel() else 0.0
    k = max(0, math.ceil(math.log2(max(top, 1e-30) / 0.5)))
    Q = _herm(al * (c / 2 ** k)) * 1j
    one = _one(Q)
    X = one
    for n in range(15, 0, -1):
        X = one + _mul(Q, X) / n
    for _ in range(k):
        X = _mul(X, X)
    return X


def _log(X, c):
    """alpha of X = exp(i c alpha t), X near 1: log X = 2 artanh Y with Y = (X - 1)(X + 1)^-1."""
    one = _one(X)
    P = X + one
    cof = [[P[(j + 1) % 3, (i + 1) % 3] * P[(j + 2) % 3, (i + 2) % 3]
            - P[(j + 1) % 3, (i + 2) % 3] * P[(j + 2) % 3, (i + 1) % 3] for j in range(3)] for i in range(3)]
    inv = torch.stack([torch.stack(r) for r in cof])
    inv = inv / (P[0, 0] * inv[0, 0] + P[0, 1] * inv[1, 0] + P[0, 2] * inv[2, 0])
    Y = _mul(X - one, inv)
    Y2 = _mul(Y, Y)
    L = one / 41.0
    for n in range(39, 0, -2):
        L = one / n + _mul(Y2, L)
    return _components(-2j * _mul(Y, L)) / c


def _shift(f, mu, s, bc):
    """f at x + s mu: x and y periodic, z periodic or with the edge layer repeated."""
    if mu < 2 or bc:
        return torch.roll(f, -s, -1 - mu)
    return torch.cat([f[..., 1:, :, :], f[..., -1:, :, :]], -3) if s > 0 else torch.cat(
        [f[..., :1, :, :], f[..., :-1, :, :]], -3)


def _adj(V, al):
    return _components(_mul(_mul(V, _herm(al)), _dag(V)))


def _inv_adj(V, al):
    return _components(_mul(_mul(_dag(V), _herm(al)), V))


class Fields:
    """Links U, half-step links W, electric fields E, currents J = (J+, J-, J+stat, J-stat)."""

    def __init__(self, U, W, E, J, a, dt, bc):
        self.U, self.W, self.E, self.J, self.a, self.dt, self.bc = U, W, E, J, a, dt, bc

    def at(self, mu, d, s, f=None):
        return _shift((self.U if f is None else f)[mu], d, s, self.bc)

    def step(self):
        """One leapfrog step from t to t + dt."""
        U, a, dt, bc = self.U, self.a, self.dt, self.bc
        vol, dz = a[0] * a[1] * a[2], self.dt / a[2]
        jp, jm, jps, jms = self.J
        E, W, N = [], [], []
        for mu in range(3):
            F = 0.0
            for nu in range(3):
                if nu == mu:
                    continue
                fwd = _mul(_mul(self.at(nu, mu, 1), _dag(self.at(mu, nu, 1))), _dag(U[nu]))
                low = _shift(_mul(_dag(_mul(U[mu], self.at(nu, mu, 1))), U[nu]), nu, -1, bc)
                F = F + (fwd + low) / a[nu] ** 2
            e = self.E[mu] - 2 * dt * vol / a[mu] ** 2 * _proj(_mul(U[mu], F))
            if mu == 2:
                e = e - dz * (jp - jm) / S2
            X = _exp(e, -0.5 * dt * a[mu] ** 2 / vol)
            h = _mul(X, U[mu])
            E.append(e)
            W.append(h)
            N.append(_mul(X, h))
        jps = jps - dz * (jp - _shift(_inv_adj(U[2], jp), 2, -1, bc))
        jms = jms + dz * (jm - _shift(_inv_adj(U[2], jm), 2, -1, bc))
        jp = jp - dz * (_adj(W[2], _shift(jps, 2, 1, bc)) - jps)
        jm = jm + dz * (_adj(W[2], _shift(jms, 2, 1, bc)) - jms)
        return Fields(N, W, E, (jp, jm, jps, jms), a, dt, bc)

    def steps(self, n):
        f = self
        for _ in range(n):
            f = f.step()
        return f

    # records
    def squares(self):
        """E_mu^2 and B_mu^2 of each site, from elementary plaquettes."""
        B = []
        for mu in range(3):
            m, n = (mu + 1) % 3, (mu + 2) % 3
            P = _mul(_mul(self.U[m], self.at(n, m, 1)), _dag(_mul(self.U[n], self.at(m, n, 1))))
            B.append(4.0 * (3.0 - (P[0, 0] + P[1, 1] + P[2, 2]).real))
        return [(e * e).sum(0) for e in self.E], B

    def weights(self):
        vol = self.a[0] * self.a[1] * self.a[2]
        return [(x / vol) ** 2 for x in self.a]

    def bulk(self):
        e, b = self.squares()
        src = (self.E[2] * (self.J[0] - self.J[1])).sum() / S2
        return torch.stack([v.sum() for v in e + b] + [torch.zeros_like(src)] * 2 + [src]).cpu().numpy()

    def field_profile(self):
        e, b = ([v.mean((-1, -2)) for v in q] for q in self.squares())
        return 0.5 * torch.stack([b[0] + b[1], b[2], e[0] + e[1], e[2]], -1).cpu().numpy()

    def current_profile(self):
        p = 0.5 * torch.stack([(self.J[w] ** 2).sum(0).mean((-1, -2)) for w in (1, 3, 0, 2)], -1).cpu().numpy()
        return _ghosts(p, self.bc)

    def energy_map(self):
        e, b = self.squares()
        nz = e[0].shape[0]
        t = sum(c * (x + y) for c, x, y in zip(self.weights(), e, b)) * (0.5 / nz)
        cut = (nz - 2) // 2 + 1
        return torch.stack([t[:cut].sum(0), t[cut:].sum(0)], -1).cpu().numpy()

    def slab(self, zc, half):
        e, b = self.squares()
        t = sum(0.5 * c * (x + y) for c, x, y in zip(self.weights(), e, b))
        return t[max(0, zc - half + 1):zc + half].sum()

    def gauss(self):
        vol = self.a[0] * self.a[1] * self.a[2]
        G = -(self.J[2] + self.J[3]) / S2
        for mu in range(3):
            G = G + self.E[mu] - _shift(_inv_adj(self.U[mu], self.E[mu]), mu, -1, self.bc)
        G = G / vol
        return (G * G).sum(0).mean((-1, -2)).cpu().numpy(), float(G.abs().max()), math.sqrt(float((G * G).mean()))

    def emt(self):
        """Transverse averages of the energy-momentum tensor: clover B of the half-step links, E averaged over x and
        x - mu (transported by the current links)."""
        bc, W = self.bc, self.W
        q = [x / (self.a[0] * self.a[1] * self.a[2]) for x in self.a]
        B, b2, E, e2 = [], [], [], []
        for mu in range(3):
            m, n = (mu + 1) % 3, (mu + 2) % 3
            U, V = W[m], W[n]
            um, vn = _shift(U, m, -1, bc), _shift(V, n, -1, bc)
            umn, vmn = (_shift(_shift(f, m, -1, bc), n, -1, bc) for f in (U, V))
            A = _mul(_mul(U, _shift(V, m, 1, bc)), _dag(_mul(V, _shift(U, n, 1, bc))))
            A = A + _mul(_mul(V, _dag(_shift(_shift(U, m, -1, bc), n, 1, bc))), _mul(_dag(_shift(V, m, -1, bc)), um))
            A = A + _mul(_mul(_dag(vn), _shift(U, n, -1, bc)), _mul(_shift(_shift(V, n, -1, bc), m, 1, bc), _dag(U)))
            A = 0.25 * (A + _mul(_dag(_mul(vmn, um)), _mul(umn, vn)))
            B.append(2.0 * _proj(A))
            b2.append(4.0 * (3.0 - (A[0, 0] + A[1, 1] + A[2, 2]).real))
            low = _shift(self.E[mu], mu, -1, bc)
            E.append(0.5 * (self.E[mu] + _shift(_inv_adj(self.U[mu], self.E[mu]), mu, -1, bc)))
            e2.append(0.5 * ((self.E[mu] ** 2).sum(0) + (low ** 2).sum(0)))
        t = [q[k] ** 2 * (e2[k] + b2[k]) for k in range(3)]

        def dot(x, y):
            return (x * y).sum(0)

        rows = [0.5 * (t[0] + t[1] + t[2]), 0.5 * (t[1] + t[2] - t[0]), 0.5 * (t[0] + t[2] - t[1]),
                0.5 * (t[0] + t[1] - t[2])]
        for k in range(3):
            i, j = (k + 1) % 3, (k + 2) % 3
            rows.append(q[i] * q[j] * (dot(E[i], B[j]) - dot(E[j], B[i])))
        for i, j in ((0, 1), (1, 2), (2, 0)):
            rows.append(q[i] * q[j] * (dot(E[i], E[j]) + dot(B[i], B[j])))
        return torch.stack([r.mean((-1, -2)) for r in rows], -1).cpu().numpy()


def _k2(n, a, dev):
    return (2.0 - 2.0 * torch.cos(2.0 * math.pi * torch.arange(n, device=dev, dtype=torch.float64) / n)) / a ** 2


def _wilson_lines(A, right):
    """Path-ordered products of exp(+-i A / sqrt 2) over z: upwards for a right mover, downwards for a left mover."""
    X = _exp(A, (1.0 if right else -1.0) / S2)
    V, order = [], range(A.shape[1])
    for z in order if right else reversed(order):
        V.append(_mul(X[:, :, z], V[-1]) if V else X[:, :, z])
    return torch.stack(V if right else V[::-1], 2)


def _sheet(rho, a, dt, right, zlo, zhi):
    """The sheet of one nucleus from its charge density (8, z, y, x): half-step and current links, E, J and Jstat."""
    dev, nz = rho.device, rho.shape[1]
    k2 = _k2(rho.shape[2], a[1], dev)[:, None] + _k2(rho.shape[3], a[0], dev)[None, :]
    safe = torch.where(k2 > 0, k2, torch.ones_like(k2))

    def transverse(f, w):
        return torch.fft.ifft2(torch.fft.fft2(f.to(torch.complex128)) * w).real

    poisson = torch.where(k2 > 0, 1.0 / safe, torch.zeros_like(k2))
    rho = transverse(rho, torch.exp(-k2 / (2 * LAMBDA ** 2)) * k2 / (k2 + M_EFF ** 2))
    om = torch.sqrt(_k2(nz, a[2], dev))
    pz = torch.arange(nz, device=dev, dtype=torch.float64)
    sg = 1.0 if right else -1.0
    half = torch.where(pz < nz // 2, sg * torch.ones_like(pz), -sg * torch.ones_like(pz))
    phase = torch.exp(1j * half * om * dt)[None, :, None, None]
    later = torch.fft.ifft(torch.fft.fft(rho.to(torch.complex128), dim=1) * phase, dim=1).real
    links = []
    for r in (rho, later):
        V = _wilson_lines(transverse(r, poisson), right)
        links.append([_mul(_dag(V), torch.roll(V, -1, -1)), _mul(_dag(V), torch.roll(V, -1, -2))])
    W, U = links
    vol = a[0] * a[1] * a[2]
    E = [_log(_mul(U[m], _dag(W[m])), -dt * a[m] ** 2 / vol) for m in range(2)]
    js = S2 * sum(E[m] - _shift(_inv_adj(U[m], E[m]), m, -1, 0) for m in range(2))
    z = torch.arange(nz, device=dev)
    js = js * ((z >= zlo) & (z <= zhi)).to(js.dtype)[None, :, None, None]
    # the moving current from the static one by continuity along z
    grad = sg * (1.0 - torch.exp(-2j * math.pi * pz / nz)) / a[2]
    f = (torch.exp(1j * half * om * dt) - 1.0) / (dt * torch.where(pz == 0, torch.ones_like(grad), grad))
    f = torch.where(pz == 0, torch.ones_like(f), torch.where(pz == nz // 2, torch.zeros_like(f), f))
    J = torch.fft.ifft(torch.fft.fft(js.to(torch.complex128), dim=1) * f[None, :, None, None], dim=1).real
    return U, W, E, J, js


def _mv_fields(n, a, dt, bc, driver, sigma, xi):
    """Initial state of a collision (driver 0), a left (1) or a right mover (2)."""
    nx, ny, nz = n
    dev = _device()
    z = torch.arange(nz, device=dev, dtype=torch.float64)
    zero = torch.zeros((8, nz, ny, nx), dtype=torch.float64, device=dev)
    J, parts = [zero] * 4, []
    for right in (False, True):
        if driver == (1 if right else 2):
            continue
        zlo, zhi = (0, nz - 1) if driver else ((nz // 2, nz - 1) if right else (0, (nz - 2) // 2))
        prof = torch.exp(-0.5 * ((z - _centers(nz)[int(right)]) / sigma) ** 2) / math.sqrt(2 * math.pi * sigma ** 2)
        x = torch.from_numpy(xi[int(right)]).to(dev).permute(2, 0, 1)
        rho = math.sqrt(a[0] * a[1]) * prof[None, :, None, None] * x[:, None]
        U, W, E, j, js = _sheet(rho, a, dt, right, zlo, zhi)
        J[int(right)], J[2 + int(right)] = j, js
        parts.append((zlo, zhi + 1, U, W, E))
    out = []
    for k in (2, 3, 4):
        out.append([torch.cat([p[k][m][..., p[0]:p[1], :, :] for p in parts], -3) for m in range(2)])
    U, W, E = out
    return Fields(U + [_one(U[0])], W + [_one(U[0])], E + [zero], tuple(J), a, dt, bc)


def _gauge(f, algorithm, tol, maxit):
    """Coulomb gauge fixing from g = 1: the Fourier-accelerated update consistent with the z boundary, or the local
    (Jacobi) update, whose links carry the top layer's transformation one iteration late."""
    own, a, bc = algorithm == "consistent", f.a, f.bc
    U, G = f.U, _one(f.U[0])
    dev, (nz, ny, nx) = G.device, G.shape[2:]
    top = G[:, :, -1:].clone()

    def edge():
        return (G[:, :, :1] if bc else G[:, :, -1:]).clone()

    def fixed():
        up = torch.cat([G[:, :, 1:], edge() if own else top], 2)
        ahead = [torch.roll(G, -1, -1), torch.roll(G, -1, -2), up]
        return [_mul(_mul(G, U[m]), _dag(ahead[m])) for m in range(3)]

    mirror = not bc and nz > 1
    mz = 2 * nz if mirror else nz
    k2 = (_k2(nx, a[0], dev)[None, None] + _k2(ny, a[1], dev)[None, :, None] + _k2(mz, a[2], dev)[:, None, None])
    scale = torch.where(k2 > 0, 1.0 / torch.where(k2 > 0, k2, torch.ones_like(k2)), torch.zeros_like(k2))
    V = fixed()
    top = edge()
    stats, n, gmax = np.zeros(7), 0, 1.0
    while n < maxit and gmax > tol:
        below = _one(V[2][:, :, :1]) if not own else V[2][:, :, -1:]
        down = torch.cat([below, V[2][:, :, :-1]], 2)
        up = V[2]
        if own and not bc:
            down = torch.cat([torch.zeros_like(below), down[:, :, 1:]], 2)
            up = torch.cat([up[:, :, :-1], torch.zeros_like(below)], 2)
        w = (V[0] + _dag(torch.roll(V[0], 1, -1))) / a[0] ** 2 + (V[1] + _dag(torch.roll(V[1], 1, -2))) / a[1] ** 2
        w = w + (up + _dag(down)) / a[2] ** 2
        d, tr = _proj(w), (w[0, 0] + w[1, 1] + w[2, 2]).real
        if own:
            g = torch.cat([d, d.flip(1)], 1) if mirror else d
            g = torch.fft.ifftn(torch.fft.fftn(g.to(torch.complex128), dim=(1, 2, 3)) * scale, dim=(1, 2, 3))
            X = _exp(g.real[:, :nz], -2.0)
        else:
            X = _exp(d, -0.3)
        st = (3.0 - X[0, 0] - X[1, 1] - X[2, 2]).abs()
        G = _mul(_dag(X), G)
        V = fixed()
        top = edge()
        gmax, n = float(d.abs().max()), n + 1
        cells = 8.0 * nx * ny * nz
        low = min(float(tr.min()), 6.0 * sum(1.0 / x ** 2 for x in a))
        stats = np.array([n, gmax, math.sqrt(float((d * d).sum()) / cells), float(st.max()),
                          math.sqrt(float((st * st).sum()) / cells), low, float(tr.mean())])
    return stats, fixed(), [_adj(G, e) for e in f.E], G


def _host_matrix(M, bc):
    """A matrix field, or three of them, in the host layout with ghost layers (z, y, x, [mu,] j, i)."""
    M = torch.stack(M).permute(3, 4, 5, 0, 2, 1) if isinstance(M, list) else M.permute(2, 3, 4, 1, 0)
    return _ghosts(M.contiguous().cpu().numpy(), bc)


def _host_vector(E, bc):
    E = torch.stack(E).permute(2, 3, 4, 0, 1) if isinstance(E, list) else E.permute(1, 2, 3, 0)
    return _ghosts(E.contiguous().cpu().numpy(), bc)


def _gradient(case, seed):
    from torch.utils.checkpoint import checkpoint
    a, dt = _spacing(case), _dt(_spacing(case))
    rho = torch.from_numpy(_density(case, seed)).to(_device()).permute(3, 0, 1, 2).contiguous().requires_grad_(True)
    nz = case["nz"]
    U, W, E, J, js = _sheet(rho, a, dt, False, 0, nz - 1)
    zero = torch.zeros_like(js)

    def advance(*t):
        n = Fields(list(t[:3]), None, list(t[3:6]), t[6:], a, dt, 0).step()
        return (*n.U, *n.E, *n.J)

    t = (*U, _one(U[0]), *E, zero, J, zero, js, zero)
    for _ in range(case["steps"]):
        t = checkpoint(advance, *t, use_reentrant=False)
    e = Fields(list(t[:3]), None, list(t[3:6]), t[6:], a, dt, 0).slab(nz // 2, 8)
    (g,) = torch.autograd.grad(e, rho)
    return {"energy": float(e.detach()), "gradient": g.permute(1, 2, 3, 0).contiguous().cpu().numpy()}


def exact(case, seed):
    kind = case["kind"]
    if kind == "gradient":
        return _gradient(case, seed)
    with torch.no_grad():
        if kind == "ensemble":
            out = []
            for n, qs, sd in _events(case, seed):
                a = (1.0, 1.0, 1.0)
                f = _mv_fields(n, a, 0.25, 0, 0, case.get("sigma", 4.0), _charges(sd, n[0], n[1], qs))
                out.append(f.steps(case["steps"]).bulk())
            return {"bulk": out}
        n, a, bc = _shape(case), _spacing(case), case.get("bc", 0)
        dt = _dt(a)
        if kind in ("measure", "exchange"):
            U, E, J = (_host_fields(case, seed))
            dev = _device()
            U = torch.from_numpy(U).to(dev).permute(5, 4, 3, 0, 1, 2)
            E = torch.from_numpy(E).to(dev).permute(4, 3, 0, 1, 2)
            f = Fields([U[:, :, m].contiguous() for m in range(3)], None, [E[:, m].contiguous() for m in range(3)],
                       tuple(torch.from_numpy(j).to(dev).permute(3, 0, 1, 2).contiguous() for j in J), a, dt, bc)
            if kind == "exchange":
                f = f.steps(case["steps"])
                out = {"U": _host_matrix(f.U, bc), "E": _host_vector(f.E, bc)}
                out.update((k, _host_vector(j, bc)) for k, j in zip(("Jp", "Jm", "JpS", "JmS"), f.J))
                return out
            f = f.step()
            per_z, gmax, grms = f.gauss()
            return {"bulk": f.bulk(), "emt": f.emt(), "gauss": per_z, "gauss_max": gmax, "gauss_rms": grms,
                    "fields": f.field_profile(), "currents": f.current_profile(), "energy_map": f.energy_map()}
        xi = _charges(seed, n[0], n[1], case.get("qs", 0.5))
        f = _mv_fields(n, a, dt, bc, case.get("driver", 0), case.get("sigma", 4.0), xi)
        if kind == "gauge":
            stats, V, E, G = _gauge(f.steps(case["evolved"]), case["algorithm"], case["tol"], case["maxit"])
            fixed = [_host_matrix(V, bc), _host_vector(E, bc), _host_matrix(G, bc)] if case["fields"] else []
            return {"stats": stats, "fixed": fixed}
        bulk = []
        if kind == "event":
            for _ in range(case["steps"] // 20):
                f = f.steps(20)
                bulk.append(f.bulk())
        else:
            f = f.steps(case["steps"])
            bulk = f.bulk()
        return {"bulk": bulk, "emt": f.emt(), "energy_map": f.energy_map()}
