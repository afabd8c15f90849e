"""Performance cases of the SCFT inner loop.

Each case is work that a program of this framework has it do through the
Python entry points: density() and scf_stress() of one system (the two calls
of every iteration of any SCFT solver), the grouped density() calls of a
Newton-Raphson Jacobian, the reverse-mode gradient, and whole Anderson solves
of one system and of a batch.

    listed()             the cases, each a dict of plain values
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  systems on the device and seeded fields
    run(state)           one pass: its outputs
    work(case)           bytes and operations that the pass cannot do without
    exact(case, seed)    the outputs in plain torch, 64 bits

All arithmetic of the path is FP64.
"""
import functools
import math

import numpy as np
import torch

from pscf_amd import adjoint, batch, iterate, scf
from pscf_amd.system import System

# ------------------------------------------------------------------- phases
# Space groups by generators: (3x3 integer matrix, translation) in the
# conventional (Bravais) basis, acting on fractional coordinates.
_INV = ((-1, 0, 0, 0, -1, 0, 0, 0, -1), (0, 0, 0))
_BODY = ((1, 0, 0, 0, 1, 0, 0, 0, 1), (.5, .5, .5))
_R3 = ((0, 0, 1, 1, 0, 0, 0, 1, 0), (0, 0, 0))                     # z,x,y
PHASES = {
    # 1D lamellae and 2D cylinders: the cells in which most sweeps are run
    "lam1d": (1, "lamellar", (1.5,), "-1", [((-1,), (0,))]),
    "hex2d": (2, "hexagonal", (1.8,), "p 6 m m",
              [((1, -1, 1, 0), (0, 0)), ((0, 1, 1, 0), (0, 0))]),
    # 3D cells
    "lam": (3, "tetragonal", (1.6, 1.6), "P 4/m m m",
            [((0, -1, 0, 1, 0, 0, 0, 0, 1), (0, 0, 0)),
             ((-1, 0, 0, 0, 1, 0, 0, 0, -1), (0, 0, 0)), _INV]),
    "hex": (3, "hexagonal", (1.9, 1.9), "P 6/m m m",
            [((1, -1, 0, 1, 0, 0, 0, 0, 1), (0, 0, 0)),
             ((0, 1, 0, 1, 0, 0, 0, 0, -1), (0, 0, 0)), _INV]),
    "bcc": (3, "cubic", (1.8,), "I m -3 m",
            [((-1, 0, 0, 0, -1, 0, 0, 0, 1), (0, 0, 0)), _R3,
             ((0, 1, 0, 1, 0, 0, 0, 0, -1), (0, 0, 0)), _INV, _BODY]),
    "gyr": (3, "cubic", (3.4,), "I a -3 d",
            [((-1, 0, 0, 0, -1, 0, 0, 0, 1), (.5, 0, .5)), _R3,
             ((0, 1, 0, 1, 0, 0, 0, 0, -1), (.75, .25, .25)), _INV, _BODY]),
    "fddd": (3, "orthorhombic", (0.95, 1.6, 3.2), "F d d d : 2",
             [((-1, 0, 0, 0, -1, 0, 0, 0, 1), (.75, .75, 0)),
              ((-1, 0, 0, 0, 1, 0, 0, 0, -1), (.75, 0, .75)), _INV,
              ((1, 0, 0, 0, 1, 0, 0, 0, 1), (0, .5, .5)),
              ((1, 0, 0, 0, 1, 0, 0, 0, 1), (.5, 0, .5))]),
    # a chiral group, without inversion (star_invert = +-1 pairs)
    "p213": (3, "cubic", (2.0,), "P 21 3",
             [((-1, 0, 0, 0, -1, 0, 0, 0, 1), (.5, 0, .5)),
              ((-1, 0, 0, 0, 1, 0, 0, 0, -1), (0, .5, .5)), _R3]),
}


def _group(phase):
    """Every element of the phase's group: m (order, 9) in Fortran order, v (order, 3)."""
    dim, _, _, _, gens = PHASES[phase]
    one = (tuple(int(i == j) for i in range(dim) for j in range(dim)), (0.0,) * dim)

    def mul(a, b):
        A, B = np.array(a[0]).reshape(dim, dim), np.array(b[0]).reshape(dim, dim)
        t = (A @ np.array(b[1], float) + np.array(a[1], float)) % 1.0
        return tuple(int(x) for x in (A @ B).ravel()), tuple(float(round(x * 24) % 24) / 24 for x in t)

    els, todo = {one: None}, [one]
    while todo:
        e = todo.pop()
        for g in gens:
            p = mul(g, e)
            if p not in els:
                els[p] = None
                todo.append(p)
    m = np.zeros((len(els), 9))
    v = np.zeros((len(els), 3))
    for i, (a, t) in enumerate(els):
        full = np.zeros((3, 3))
        full[:dim, :dim] = np.array(a).reshape(dim, dim)
        m[i] = full.ravel(order="F")
        v[i, :dim] = t
    return m, v


def _lib():
    from pscf_amd._lib import lib
    return lib()


@functools.lru_cache(maxsize=4)
def _tables(phase, grid):
    """Star tables of the phase on the grid (a program builds or reads them once)."""
    dim, cs, cell, _, _ = PHASES[phase]
    _, G, _ = iterate.unit_cell(_lib(), dim, cs, np.array(cell))
    m, v = _group(phase)
    t = scf.Basis.build_tables(dim, grid, G, m, v, lib=_lib())
    return t, scf.Basis.from_tables(t)


def _grid(case):
    return tuple(int(case[k]) for k in ("n1", "n2", "n3") if k in case)


# Chemistries, N = 100 (1 for the 1D/2D cells, which count lengths in chains):
# "ab": AB diblock; "aba": ABA triblock + A homopolymer; "abas": the same with
# a B solvent.
def _system(case, rng, phase=None, grid=None):
    phase = phase or case["phase"]
    dim, cs, cell, name, _ = PHASES[phase]
    N = 100.0 if dim == 3 else 1.0
    chi = float(rng.uniform(15.0, 22.0)) / N
    f = {"lam1d": .5, "lam": .45, "hex2d": .3, "hex": .3, "bcc": .25, "gyr": .36, "fddd": .42,
         "p213": .4}[phase] + float(rng.uniform(-.02, .02))
    kind = case.get("chem", "ab")
    if kind == "ab":
        chains, phi, solv, phis = [[(1, f * N), (2, (1 - f) * N)]], [1.0], [], []
    else:
        ph = float(rng.uniform(.05, .2))
        chains = [[(1, .2 * N), (2, .6 * N), (1, .2 * N)], [(1, .5 * N)]]
        ps = .05 if kind == "abas" else 0.0
        phi = [1.0 - ph - ps, ph]
        solv, phis = ([(2, .01 * N)], [ps]) if ps else ([], [])
    scale = (10.0 if dim == 3 else 1.0) * float(rng.uniform(.97, 1.03))
    return System(kuhn=[1.0, 1.0], chains=chains, phi_chain=phi,
                  chi=np.array([[0.0, chi], [chi, 0.0]]), dim=dim, crystal_system=cs,
                  cell_param=[c * scale for c in cell], ngrid=list(grid or _grid(case)),
                  chain_step=N / case["steps"], group_name=name, solvents=solv, phi_solvent=phis)


def _omega(sysm, nstar, rng):
    """A field on the way to convergence: an ordered first harmonic, chi phi_B
    and chi phi_A in opposite phase, and decaying noise on the next stars."""
    chi = float(sysm.chi[0, 1])
    om = np.zeros((2, nstar))
    om[:, 0] = sysm.chi @ sysm.phi_monomer()
    n = min(24, nstar)
    om[:, 1:n] = rng.normal(0.0, .1 * chi, (2, n - 1)) / np.sqrt(np.arange(1, n))
    a = .35 * chi * float(rng.uniform(.8, 1.2))
    om[0, 1] += a
    om[1, 1] -= a
    return om


def _make(case, rng, phase=None, grid=None):
    sysm = _system(case, rng, phase, grid)
    t, B = _tables(phase or case["phase"], tuple(sysm.ngrid))
    _, G, dGG = iterate.unit_cell(_lib(), sysm.dim, sysm.crystal_system, np.array(sysm.cell_param))
    S = scf.SCFSystem(sysm, B, G)
    dgsq = iterate.make_dgsq(_lib(), B, dGG, len(sysm.cell_param))
    return S, _omega(sysm, B.N_star, rng), dgsq, G


# -------------------------------------------------------------------- cases
def listed():
    return [
        # an iteration of a lamellar solve: the smallest call, all latency
        {"name": "lam1d-32", "do": "iter", "phase": "lam1d", "n1": 32, "steps": 100},
        # an iteration of a 2D cylinder solve
        {"name": "hex2d-48", "do": "iter", "phase": "hex2d", "n1": 48, "n2": 48, "steps": 100},
        # an iteration of the BCC 32^3 solve (N = 100, ds = 1)
        {"name": "bcc-32", "do": "iter", "phase": "bcc", "n1": 32, "n2": 32, "n3": 32, "steps": 100},
        # an anisotropic grid: the O70 network in its orthorhombic cell
        {"name": "fddd-32x48x64", "do": "iter", "phase": "fddd", "n1": 32, "n2": 48, "n3": 64, "steps": 100},
        # a blend of two chain species with a solvent in a chiral group
        {"name": "p213-blend-40", "do": "iter", "phase": "p213", "chem": "abas", "n1": 40, "n2": 40, "n3": 40, "steps": 100},
        # an iteration of the headline solve: gyroid 64^3, ds = 0.5, with its stress
        {"name": "gyr-64", "do": "iter", "phase": "gyr", "n1": 64, "n2": 64, "n3": 64, "steps": 200},
        # the finest 3D grid in ordinary use
        {"name": "gyr-96", "do": "iter", "phase": "gyr", "n1": 96, "n2": 96, "n3": 96, "steps": 200},
        # columns of a Newton-Raphson Jacobian: 32 perturbed density() calls
        {"name": "jac-bcc-32", "do": "many", "phase": "bcc", "n1": 32, "n2": 32, "n3": 32, "steps": 100, "fields": 32},
        # whole calls: Anderson iterations of one gyroid with its cell relaxed,
        # and of a mixed batch (lamellar 32^3, hexagonal 48^3, cubic 64^3)
        {"name": "solve-gyr-64", "do": "solve", "phase": "gyr", "n1": 64, "n2": 64, "n3": 64, "steps": 200, "iters": 5},
        {"name": "batch-16", "do": "batch", "steps": 100, "iters": 4, "lam": 4, "hex": 4, "bcc": 4, "gyr": 4, "n_cubic": 64},
        # gradients: sum (phi_A - target)^2 at the gyroid by omega(r), cell and block
        # lengths; and of a checkpointed blend on the largest grid
        {"name": "grad-gyr-64", "do": "grad", "phase": "gyr", "n1": 64, "n2": 64, "n3": 64, "steps": 200, "stride": 0},
        {"name": "grad-aba-96", "do": "grad", "phase": "bcc", "chem": "aba", "n1": 96, "n2": 96, "n3": 96, "steps": 200, "stride": 14},
    ]


_CUBE = (12, 16, 20, 24, 28, 32, 40, 48, 56, 64)
_BOX = ((16, 12, 24), (24, 16, 12), (32, 48, 64), (32, 32, 48), (48, 40, 32), (64, 48, 40))


def draw(rng):
    do = rng.choice(["iter"] * 7 + ["many", "solve", "grad"])
    steps = 2 * int(round(math.exp(rng.uniform(math.log(25), math.log(100)))))
    if do == "iter" and rng.random() < .3:
        if rng.random() < .5:
            return {"do": do, "phase": "lam1d", "n1": rng.choice(_CUBE + (96, 128)), "steps": steps}
        n = rng.choice(_CUBE + (96,))
        return {"do": do, "phase": "hex2d", "n1": n, "n2": n, "steps": steps,
                "chem": rng.choice(["ab", "aba"])}
    ph = rng.choice(["lam", "hex", "bcc", "gyr", "fddd", "p213"])
    if ph == "fddd":
        g = rng.choice(_BOX)
    else:
        sizes = [n for n in _CUBE if ph != "gyr" or n % 4 == 0]
        n = rng.choice(sizes[:6] if do in ("many", "solve") else sizes)
        g = (n, n, n)
    case = {"do": do, "phase": ph, "n1": g[0], "n2": g[1], "n3": g[2], "steps": steps,
            "chem": rng.choice(["ab", "ab", "aba", "abas"])}
    if do == "many":
        case["fields"] = rng.randint(2, 32)
    elif do == "solve":
        case["iters"] = rng.randint(2, 5)
    elif do == "grad":
        case["chem"] = rng.choice(["ab", "aba"])
        case["stride"] = rng.choice([0, 0, 7, 14])
    return case


_BATCH = (("lam", 32), ("hex", 48), ("bcc", 0), ("gyr", 0))      # edge 0: n_cubic


def _batch_instances(case, rng):
    out = []
    for phase, n in _BATCH:
        n = n or case["n_cubic"]
        out += [_make(case, rng, phase, (n, n, n)) for _ in range(case[phase])]
    return out


def prepare(case, seed):
    rng = np.random.default_rng([seed, 7])
    do = case["do"]
    if do == "batch":
        return {"case": case, "inst": _batch_instances(case, rng)}
    S, om, dgsq, G = _make(case, rng)
    st = {"case": case, "S": S, "omega": om, "dgsq": dgsq, "G": G}
    if do == "many":                     # one star coefficient moved by 1e-8 each
        oms = np.repeat(om[None], case["fields"], axis=0)
        for i in range(case["fields"]):
            oms[i, i % 2, (1 + i // 2) % S.N_star] += 1e-8
        st["omegas"] = oms
    elif do == "grad":
        if case["stride"]:
            S.set_checkpoint(case["stride"])
        dev = torch.device("cuda")
        tgt = np.zeros((1, S.N_star))
        n = min(20, S.N_star)
        tgt[0, 0] = float(S.system.phi_monomer()[0])
        tgt[0, 1:n] = .05 * rng.normal(size=n - 1)
        st["omega_grid"] = adjoint.stars_to_grid(S, torch.tensor(om, device=dev)).detach()
        st["target"] = adjoint.stars_to_grid(S, torch.tensor(tgt, device=dev))[0].detach()
        st["cell"] = torch.tensor(S.system.cell_param, dtype=torch.float64)
        st["lengths"] = adjoint.block_lengths(S.system)
    return st


# Anderson mixing to a fixed count of iterations: the residual bound is never met
_TOL = 1e-13


def run(st):
    case = st["case"]
    do = case["do"]
    if do == "batch":
        for S, _, _, G in st["inst"]:
            S.set_cell(G)
        B = batch.BatchSolver(n_hist=20, domain=True, error_max=_TOL, max_itr=case["iters"])
        for S, om, _, _ in st["inst"]:
            B.add(S, om)
        B.solve()
        res = [B.result(i) for i in range(len(st["inst"]))]
        return {"omega": [r.omega for r in res],
                "cell": np.concatenate([r.cell_param for r in res]),
                "rho": [r.rho for r in res],
                "f": np.array([r.f_helmholtz for r in res])}
    S = st["S"]
    if do == "iter":
        rho, q, qs = S.density(st["omega"])
        return {"rho": rho, "q": q, "qs": qs, "stress": S.scf_stress(st["dgsq"])}
    if do == "many":
        rho, q, qs = S.density_many(st["omegas"])
        return {"rho": rho, "q": q, "qs": qs}
    if do == "solve":
        S.set_cell(st["G"])
        r = iterate.AndersonMixing(S, 20, True).run(st["omega"], _TOL, case["iters"])
        return {"omega": r.omega, "rho": r.rho, "cell": r.cell_param, "stress": r.stress,
                "f": r.f_helmholtz, "p": r.pressure}
    om = st["omega_grid"].requires_grad_(True)
    om.grad = None
    cell = st["cell"].clone().requires_grad_(True)
    lengths = st["lengths"].clone().requires_grad_(True)
    rho, Q = adjoint.density(S, om, cell, lengths)
    loss = ((rho[0] - st["target"]) ** 2).sum() / rho[0].numel()
    loss.backward()
    return {"rho": rho.detach(), "Q": Q.detach(), "omega": om.grad, "cell": cell.grad,
            "lengths": lengths.grad}


# --------------------------------------------------------------------- work
def _steps(case):
    """Contour steps of all sweeps of one density()."""
    chain = 2 * case["steps"]                        # both directions
    return chain + (chain // 2 if case.get("chem", "ab") != "ab" else 0)


def work(case):
    """Bytes: the fields in and out on the grid (two monomers; of a gradient
    also the target and the gradient), each once.  Operations: the transforms,
    six real 3D transforms of 2.5 M log2 M each per contour step; the backward
    of a gradient sweeps twice what its forward does."""
    if case["do"] == "batch":
        ws = []
        for ph, n in _BATCH:
            n = n or case["n_cubic"]
            w = work({"do": "iter", "phase": ph, "n1": n, "n2": n, "n3": n, "steps": case["steps"]})
            ws.append({k: case[ph] * (case["iters"] + 1) * v for k, v in w.items()})
        return {k: sum(w[k] for w in ws) for k in ("bytes", "flops")}
    M = float(np.prod(_grid(case)))
    fl = _steps(case) * 6 * 2.5 * M * math.log2(M)
    times = {"many": case.get("fields", 1), "solve": case.get("iters", 0) + 1}.get(case["do"], 1)
    if case["do"] == "grad":
        return {"bytes": 56 * M, "flops": 3 * fl}
    return {"bytes": times * 32 * M, "flops": times * fl}


# -------------------------------------------------------------------- exact
def _ksq(grid, dim, G, dev):
    """|G|^2 of the minimum images on the half grid (kz, ky, kx)."""
    n = list(grid) + [1] * (3 - dim)
    ax = [torch.arange(n[2], device=dev), torch.arange(n[1], device=dev),
          torch.arange(n[0] // 2 + 1, device=dev)]
    kz, ky, kx = torch.meshgrid(*ax, indexing="ij")
    best = None
    rng3 = [(0, -1, 1) if d < dim else (0,) for d in range(3)]
    for a in rng3[0]:
        for b in rng3[1]:
            for c in rng3[2]:
                v = [kx + a * n[0], ky + b * n[1], kz + c * n[2]]
                g2 = 0.0
                for j in range(dim):
                    g2 = g2 + sum(v[i].double() * G[i, j] for i in range(dim)) ** 2
                if best is None:
                    best, at = g2, torch.stack(v)
                else:
                    less = g2 < best - 1e-8
                    best = torch.where(less, g2, best)
                    at = torch.where(less, torch.stack(v), at)
    return best, at


class _Plain:
    """density() and scf_stress() of one system in plain torch."""

    def __init__(self, sysm, t, G, dev):
        self.s, self.dev, self.G = sysm, dev, torch.tensor(G, device=dev)
        n = list(sysm.ngrid) + [1] * (3 - sysm.dim)
        self.shape, self.n = (n[2], n[1], n[0]), n
        self.M = n[0] * n[1] * n[2]
        self.k2, _ = _ksq(sysm.ngrid, sysm.dim, self.G, dev)
        w = np.zeros((len(t["coeff"]), 3), dtype=np.int64)
        w[:, :sysm.dim] = t["wave"]
        w %= np.array(n)
        keep = w[:, 0] <= n[0] // 2
        self.at = torch.tensor(((w[:, 2] * n[1] + w[:, 1]) * (n[0] // 2 + 1) + w[:, 0])[keep], device=dev)
        self.co = torch.tensor(t["coeff"][keep], device=dev)
        self.star = torch.tensor(t["star_of_wave"][keep].astype(np.int64) - 1, device=dev)
        self.inv = torch.tensor(t["star_invert"].astype(np.int64), device=dev)
        # the star's own wave, at -k where k is in the upper half
        r = np.zeros((len(t["star_invert"]), 3), dtype=np.int64)
        r[:, :sysm.dim] = t["wave_of_star"]
        full = {tuple(x): c for x, c in zip(w.tolist(), t["coeff"])}
        r %= np.array(n)
        self.cr = torch.tensor(np.array([full[tuple(x)] for x in r.tolist()]), device=dev)
        up = r[:, 0] > n[0] // 2
        r[up] = (-r[up]) % np.array(n)
        self.ar = torch.tensor((r[:, 2] * n[1] + r[:, 1]) * (n[0] // 2 + 1) + r[:, 0], device=dev)
        self.up = torch.tensor(up, device=dev)

    def fwd(self, x):
        return torch.fft.fftn(torch.fft.rfft(x, dim=-1), dim=(-3, -2))

    def back(self, k):
        """Inverse of fwd; the two real columns' imaginary parts are dropped."""
        k = torch.fft.ifftn(k, dim=(-3, -2))
        im = torch.ones(k.shape[-1], dtype=torch.float64, device=self.dev)
        im[0] = 0.0
        im[-1] = 0.0
        return torch.fft.irfft(torch.complex(k.real, k.imag * im), n=self.n[0], dim=-1)

    def grid(self, stars):
        """(nf, N_star) -> (nf, N3, N2, N1)."""
        a = torch.as_tensor(stars, dtype=torch.float64, device=self.dev)
        nxt, prv = torch.roll(a, -1, 1), torch.roll(a, 1, 1)
        h = math.sqrt(.5)
        amp = torch.where(self.inv == 0, torch.complex(a, 0 * a),
                          torch.where(self.inv == 1, torch.complex(h * a, -h * nxt),
                                      torch.complex(h * prv, h * a)))
        k = torch.zeros((len(a), self.n[2] * self.n[1] * (self.n[0] // 2 + 1)),
                        dtype=torch.complex128, device=self.dev)
        k[:, self.at] = amp[:, self.star] * self.co
        return self.back(k.reshape(len(a), self.n[2], self.n[1], -1)) * self.M

    def stars(self, x):
        """(nf, N3, N2, N1) -> (nf, N_star), unnormalised."""
        z = self.fwd(x).reshape(len(x), -1)[:, self.ar]
        z = torch.where(self.up, z.conj(), z) / self.cr
        return torch.where(self.inv == 0, z.real,
                           math.sqrt(2.0) * torch.where(self.inv == 1, z.real, z.imag))

    def blocks(self, chain):
        """(monomer, steps, ds of length 1) of each block: make_chain_grid's rule."""
        out = []
        for m, L in chain:
            h = max(1, int(L / self.s.chain_step / 2.0 + .5))
            out.append((m - 1, 2 * h))
        return out

    def sweep(self, w, blocks, ds, k2, back):
        """q (first to last in the sweep's own order) along one chain."""
        order = list(zip(blocks, ds))
        q = torch.ones(self.shape, dtype=torch.float64, device=self.dev)
        out = [q]
        for (m, n), d in (order[::-1] if back else order):
            e1, e2 = torch.exp(-d / 2 * w[m]), torch.exp(-d / 4 * w[m])
            b2 = self.s.kuhn[m] ** 2
            f1, f2 = torch.exp(-d * b2 / 6 * k2), torch.exp(-d * b2 / 12 * k2)
            for _ in range(n):
                one = e1 * self.back(f1 * self.fwd(e1 * q))
                half = e1 * self.back(f2 * self.fwd(e2 * q))
                q = (4.0 * e2 * self.back(f2 * self.fwd(half)) - one) / 3.0
                out.append(q)
        return out[::-1] if back else out

    def density(self, w, k2=None, lengths=None):
        """rho grids, Q, and per chain (qf, qr, blocks, ds, N)."""
        k2 = self.k2 if k2 is None else k2
        rho = [torch.zeros(self.shape, dtype=torch.float64, device=self.dev) for _ in self.s.kuhn]
        Q, kept, at = [], [], 0
        qs = []
        for (m, size), p in zip(self.s.solvents, self.s.phi_solvent):
            b = torch.exp(-size * w[m - 1])
            qs.append(b.mean())
            rho[m - 1] = rho[m - 1] + p * b / qs[-1]
        for c, chain in enumerate(self.s.chains):
            bl = self.blocks(chain)
            L = [torch.tensor(x, dtype=torch.float64, device=self.dev) for _, x in chain] \
                if lengths is None else list(lengths[at:at + len(chain)])
            at += len(chain)
            ds = [x / n for x, (_, n) in zip(L, bl)]
            N = sum(L)
            qf, qr = self.sweep(w, bl, ds, k2, False), self.sweep(w, bl, ds, k2, True)
            q = qf[-1].mean()
            lo = 0
            for (m, n), d in zip(bl, ds):
                acc = qf[lo] * qr[lo] + qf[lo + n] * qr[lo + n]
                for i in range(1, n):
                    acc = acc + (4.0 if i % 2 else 2.0) * qf[lo + i] * qr[lo + i]
                rho[m] = rho[m] + self.s.phi_chain[c] / (N * q) * (d / 3.0) * acc
                lo += n
            Q.append(q)
            kept.append((qf, qr, bl, ds, N))
        return torch.stack(rho), torch.stack(Q), qs, kept

    def stress(self, Q, kept, dgsq):
        dg = torch.tensor(dgsq, device=self.dev)
        out = torch.zeros(dg.shape[1], dtype=torch.float64, device=self.dev)
        for c, (qf, qr, bl, ds, N) in enumerate(kept):
            lo = 0
            for (m, n), d in zip(bl, ds):
                for i in range(n + 1):
                    x = self.stars(torch.stack([qf[lo + i], qr[lo + i]]))
                    wt = 1.0 if i in (0, n) else (4.0 if i % 2 else 2.0)
                    out += self.s.phi_chain[c] / (N * Q[c]) * wt * d * self.s.kuhn[m] ** 2 \
                        / (18.0 * float(self.M) ** 2) * ((x[0] * x[1]) @ dg)
                lo += n
        return out


def exact(case, seed):
    do = case["do"]
    # iterates of Anderson mixing hang on all that came before, and the rounding
    # of its least-squares problems with them
    if do in ("batch", "solve"):
        return None
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    rng = np.random.default_rng([seed, 7])
    sysm = _system(case, rng)
    t, B = _tables(case["phase"], tuple(sysm.ngrid))
    _, G, dGG = iterate.unit_cell(_lib(), sysm.dim, sysm.crystal_system, np.array(sysm.cell_param))
    om = _omega(sysm, B.N_star, rng)
    P = _Plain(sysm, t, G, dev)
    if do == "many":
        # the fields differ by 1e-8 in one coefficient: computed one by one
        rho, q, qs = [], [], []
        for i in range(case["fields"]):
            o = om.copy()
            o[i % 2, (1 + i // 2) % B.N_star] += 1e-8
            r, Q, s, _ = P.density(P.grid(o))
            rho.append(P.stars(r) / P.M)
            q.append(Q)
            qs.append(torch.stack(s) if s else Q[:0])
        return {"rho": torch.stack(rho), "q": torch.stack(q), "qs": torch.stack(qs)}
    if do == "iter":
        dgsq = iterate.make_dgsq(_lib(), B, dGG, len(sysm.cell_param))
        rho, Q, qs, kept = P.density(P.grid(om))
        return {"rho": P.stars(rho) / P.M, "q": Q, "qs": torch.stack(qs) if qs else Q[:0],
                "stress": P.stress(Q, kept, dgsq)}
    if case["stride"]:
        return None        # the plain form keeps every contour point of every sweep
    n = min(20, B.N_star)
    tgt = np.zeros((1, B.N_star))
    tgt[0, 0] = float(sysm.phi_monomer()[0])
    tgt[0, 1:n] = .05 * rng.normal(size=n - 1)
    tgt = P.grid(tgt)[0]
    w = P.grid(om).requires_grad_(True)
    dk2 = []
    _, at = _ksq(sysm.ngrid, sysm.dim, P.G, dev)
    for k in range(len(sysm.cell_param)):
        g = 0.0
        for i in range(sysm.dim):
            for j in range(sysm.dim):
                g = g + at[i].double() * at[j].double() * float(dGG[i, j, k])
        dk2.append(g)
    cell = torch.zeros(len(dk2), dtype=torch.float64, device=dev, requires_grad=True)
    lengths = torch.tensor([L for c in sysm.chains for _, L in c], dtype=torch.float64, device=dev,
                           requires_grad=True)
    rho, Q, _, _ = P.density(w, P.k2 + sum(cell[k] * dk2[k] for k in range(len(dk2))), lengths)
    loss = ((rho[0] - tgt) ** 2).sum() / P.M
    loss.backward()
    return {"rho": rho.detach(), "Q": Q.detach(), "omega": w.grad, "cell": cell.grad,
            "lengths": lengths.grad}
