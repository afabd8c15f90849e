"""Sweeps on symmetric planes against sweeps that store every plane.

density() on star coefficients keeps only the planes from which the space
group makes the others (kernels.hpp, sym_planes); density() on grids keeps
every plane.  Both are FP64 evaluations of the same map, so Q, the densities,
the contour points and the gradients agree to rounding: 1e-12 of the largest
value (fields of order one, some hundred roundings per point).  The groups
cover each kind of operation: z -> -z by inversion and by a mirror plane,
z -> z + N3/2 by centring and by a screw axis, with and without shifts in the
plane, and grids whose edges give odd and even numbers of planes.
"""
import numpy as np
import pytest
import torch

from conftest import get_lib

from pscf_amd import adjoint, iterate, scf
from pscf_amd.system import System

I3 = (1, 0, 0, 0, 1, 0, 0, 0, 1)
INV = ((-1, 0, 0, 0, -1, 0, 0, 0, -1), (0, 0, 0))
C2Z = (-1, 0, 0, 0, -1, 0, 0, 0, 1)
MZ = (1, 0, 0, 0, 1, 0, 0, 0, -1)
TET = ("tetragonal", [2.0, 2.3])
ORTH = ("orthorhombic", [2.0, 2.4, 2.2])
# name -> (cell, generators, grid)
GROUPS = {
    "P -1": (ORTH, [INV], (8, 8, 12)),
    "body centred": (ORTH, [INV, (I3, (.5, .5, .5))], (12, 16, 8)),
    "A centred": (ORTH, [INV, (I3, (0, .5, .5))], (8, 12, 12)),
    "mirror": (ORTH, [(MZ, (0, 0, 0))], (8, 8, 16)),
    "glide": (ORTH, [(MZ, (.5, 0, 0))], (12, 8, 8)),
    "screw": (ORTH, [(C2Z, (.5, 0, .5))], (8, 12, 8)),
    "screw, inversion": (TET, [(C2Z, (0, .5, .5)), INV], (16, 16, 20)),
    "no operation": (ORTH, [(C2Z, (0, 0, 0))], (8, 8, 8)),
}


def group(gens):
    one = (I3, (0.0, 0.0, 0.0))

    def mul(a, b):
        A, B = np.array(a[0]).reshape(3, 3), np.array(b[0]).reshape(3, 3)
        t = (A @ np.array(b[1], float) + np.array(a[1], float)) % 1.0
        return tuple(int(v) for v in (A @ B).ravel()), tuple(float(round(v * 24) % 24) / 24 for v in t)

    els, todo = {one}, [one]
    while todo:
        e = todo.pop()
        for g in gens:
            p = mul((g[0], tuple(float(v) for v in g[1])), e)
            if p not in els:
                els.add(p)
                todo.append(p)
    els = sorted(els, key=lambda e: (e != one, e))
    m = np.array([np.array(a).reshape(3, 3).ravel(order="F") for a, _ in els], float)
    return m, np.array([t for _, t in els])


def system(name, lib):
    (cs, cell), gens, grid = GROUPS[name]
    s = System(kuhn=[1.0, 1.2], chains=[[(1, 0.4), (2, 0.6)], [(2, 0.3)]], phi_chain=[0.8, 0.2],
               chi=np.array([[0.0, 15.0], [15.0, 0.0]]), dim=3, crystal_system=cs, cell_param=cell,
               ngrid=list(grid), chain_step=0.05, group_name=name)
    _, G, dGG = iterate.unit_cell(lib, 3, cs, np.array(cell))
    m, v = group(gens)
    B = scf.Basis.from_tables(scf.Basis.build_tables(3, grid, G, m, v, lib=lib))
    S = scf.SCFSystem(s, B, G, lib=lib)
    rng = np.random.default_rng(11)
    om = np.zeros((2, B.N_star))
    n = min(14, B.N_star)
    om[:, :n] = rng.normal(0.0, 1.5, (2, n))
    return S, om, iterate.make_dgsq(lib, B, dGG, len(cell))


def on_grid(S, om, lib):
    dev = torch.device(lib.tensor_device)
    w = adjoint.stars_to_grid(S, torch.tensor(om, device=dev)).detach()
    rho, Q = adjoint.density(S, w)
    return w, rho.cpu().numpy(), Q.cpu().numpy()


def close(a, b, tol=1e-12):
    a, b = np.asarray(a), np.asarray(b)
    assert np.abs(a - b).max() <= tol * max(np.abs(b).max(), 1e-30), np.abs(a - b).max() / np.abs(b).max()


@pytest.mark.parametrize("name", list(GROUPS))
def test_symmetric_planes_match_full_storage(name, backend):
    lib = get_lib(backend)
    S, om, dgsq = system(name, lib)
    rho, q, _ = S.density(om)
    st = S.scf_stress(dgsq)
    _, rg = S.grids()
    pts = [(c, d, s) for c in (0, 1) for d in (1, -1) for s in (1, 3)]
    qs = [S.q(*p) for p in pts]
    w, rho_f, q_f = on_grid(S, om, lib)
    close(q, q_f)
    close(rg, rho_f)
    close(st, S.scf_stress(dgsq), 1e-10)          # a sum of terms of both signs
    for p, v in zip(pts, qs):
        close(v, S.q(*p))
    rho2, q2, _ = S.density(om)                   # and back
    assert np.array_equal(rho, rho2) and np.array_equal(q, q2)


@pytest.mark.parametrize("stride", [0, 5])
@pytest.mark.parametrize("name", ["body centred", "screw"])
def test_gradient_after_density_on_symmetric_planes(name, stride, backend):
    """The reverse mode of a star-coefficient density() reads the same contour
    points as that of the density() on grids."""
    import ctypes
    from pscf_amd._lib import dptr
    lib = get_lib(backend)
    S, om, _ = system(name, lib)
    S.set_checkpoint(stride)
    rng = np.random.default_rng(5)
    dev = torch.device(lib.tensor_device)
    lam = torch.tensor(rng.normal(size=(2,) + S.shape), device=dev)
    got = []
    for star in (True, False):
        if star:
            S.density(om)
        else:
            on_grid(S, om, lib)
        g = torch.empty_like(lam)
        dlen = np.zeros(3)
        if dev.type == "cuda":
            torch.cuda.synchronize()
        lib.call("pscf_density_adjoint_dev", S.h, ctypes.c_void_p(lam.data_ptr()), dptr(np.zeros(2)),
                 ctypes.c_void_p(g.data_ptr()), 0, None, None, dptr(dlen), None)
        got.append((g.cpu().numpy(), dlen))
    close(got[0][0], got[1][0], 1e-11)
    close(got[0][1], got[1][1], 1e-11)


@pytest.mark.parametrize("name", ["mirror", "screw"])
def test_cell_without_the_operation_stores_every_plane(name, backend):
    """A cell in which the operation changes |k| (third axis oblique) runs on
    every plane; so do the grouped calls."""
    lib = get_lib(backend)
    S, om, dgsq = system(name, lib)
    S.density(om)
    G = np.array(S.G_basis)
    G[2, 0] += 0.31 * G[0, 0]
    S.set_cell(G)
    rho, q, _ = S.density(om)
    _, rg = S.grids()
    many = S.density_many(np.stack([om, 0.9 * om]))
    w = adjoint.stars_to_grid(S, torch.tensor(om, device=lib.tensor_device)).detach()
    rho_f = torch.empty_like(w)
    import ctypes
    from pscf_amd._lib import dptr
    q_f = np.zeros(2)
    if w.device.type == "cuda":
        torch.cuda.synchronize()
    lib.call("pscf_density_grid_dev", S.h, ctypes.c_void_p(w.data_ptr()), ctypes.c_void_p(rho_f.data_ptr()),
             dptr(q_f), dptr(np.zeros(1)), dptr(S.phi_chain), dptr(S.mu_chain), dptr(S.phi_solvent),
             dptr(S.mu_solvent))
    close(q, q_f)
    close(rg, rho_f.cpu().numpy())
    close(many[0][0], rho)
    close(many[1][0], q)
