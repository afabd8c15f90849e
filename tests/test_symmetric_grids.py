"""density() on grids and its reverse mode, on symmetric planes and off them.

Grid fields with the symmetry of the basis run on the stored planes, others on
every plane.  The reference is the same cell and grid in the group P 1, which
stores every plane: Q, densities and gradients agree to rounding, 1e-12 of the
largest value forward and 1e-11 in the gradients (as between symmetric planes
and full storage of one basis).
"""
import numpy as np
import pytest
import torch

from conftest import get_lib
from test_symmetric_planes import GROUPS, close, group

from pscf_amd import adjoint, iterate, scf
from pscf_amd.system import System


def make(cell, gens, grid, lib, stride):
    cs, par = cell
    s = System(kuhn=[1.0, 1.2], chains=[[(1, 0.4), (2, 0.6)], [(2, 0.3)]], phi_chain=[0.8, 0.2],
               chi=np.array([[0.0, 15.0], [15.0, 0.0]]), dim=3, crystal_system=cs, cell_param=par,
               ngrid=list(grid), chain_step=0.05, group_name="g")
    _, G, _ = iterate.unit_cell(lib, 3, cs, np.array(par))
    m, v = group(gens)
    S = scf.SCFSystem(s, scf.Basis.from_tables(scf.Basis.build_tables(3, grid, G, m, v, lib=lib)), G, lib=lib)
    S.set_checkpoint(stride)
    return S


def gradient(S, w, lam):
    """rho, Q and the gradients of sum lam rho + sum Q by field, cell and lengths."""
    w = w.clone().requires_grad_(True)
    cell = torch.tensor(S.system.cell_param, dtype=torch.float64, requires_grad=True)
    lengths = adjoint.block_lengths(S.system).clone().requires_grad_(True)
    rho, Q = adjoint.density(S, w, cell, lengths)
    ((lam * rho).sum() + Q.sum()).backward()
    return [x.detach().cpu().numpy() for x in (rho, Q, w.grad, cell.grad, lengths.grad)]


@pytest.mark.parametrize("stride", [0, 5])
@pytest.mark.parametrize("name", ["P -1", "body centred", "glide", "screw, inversion"])
def test_grid_fields(name, stride, backend):
    lib = get_lib(backend)
    cell, gens, grid = GROUPS[name]
    S, P = make(cell, gens, grid, lib, stride), make(cell, [], grid, lib, stride)
    rng = np.random.default_rng(23)
    stars = np.zeros((2, S.N_star))
    n = min(14, S.N_star)
    stars[:, :n] = rng.normal(0.0, 1.0, (2, n))
    dev = torch.device(lib.tensor_device)
    w = adjoint.stars_to_grid(S, torch.tensor(stars, device=dev)).detach()
    lam = adjoint.stars_to_grid(S, torch.tensor(stars[::-1].copy(), device=dev)).detach() / w[0].numel()
    off = torch.tensor(rng.normal(size=tuple(w.shape)), device=dev)
    one = torch.zeros_like(w)
    one.view(-1)[7] = 1e-9                   # one grid point off the symmetry
    calls = [(w, lam), (w, lam + 1e-3 * off), (w + 0.1 * off, lam), (w + one, lam), (w, lam + one), (w, lam)]
    if backend == "emu":                     # a gradient takes half a minute there
        if (name, stride) not in (("P -1", 0), ("screw, inversion", 5)):
            pytest.skip("on the GPU")
        calls = calls[1::4] if stride else calls[:1]
    for field, weight in calls:
        got, want = gradient(S, field, weight), gradient(P, field, weight)
        for a, b, tol in zip(got, want, (1e-12, 1e-12, 1e-11, 1e-11, 1e-11)):
            close(a, b, tol)
    if name == "P -1" and calls[-1][1] is lam:                       # the last ran on symmetric planes: r and -r are one value
        r = got[0].reshape((2,) + S.shape)
        k = S.shape[0] // 2 + 1
        assert np.array_equal(r[:, k:, 1:, 1:], r[:, S.shape[0] - k:0:-1, :0:-1, :0:-1])


def test_grouped_gradients(backend):
    """A group whose members are not all symmetric runs on every plane; either
    way each equals its single call."""
    if backend == "emu":
        pytest.skip("on the GPU")
    lib = get_lib(backend)
    cell, gens, grid = GROUPS["body centred"]
    dev = torch.device(lib.tensor_device)
    rng = np.random.default_rng(29)
    for asym in (False, True):
        single, grads, members, fields = [], [], [], []
        for i in range(2):
            S = make(cell, gens, grid, lib, 0)
            stars = np.zeros((2, S.N_star))
            stars[:, :10] = rng.normal(0.0, 1.0, (2, 10))
            w = adjoint.stars_to_grid(S, torch.tensor(stars, device=dev)).detach()
            if asym and i:
                w = w + 0.1 * torch.tensor(rng.normal(size=tuple(w.shape)), device=dev)
            single.append(gradient(S, w, w / w[0].numel())[2])
            members.append(S)
            fields.append(w)
        G = adjoint.Group(members)
        ws = [w.clone().requires_grad_(True) for w in fields]
        out = G.density(ws)
        sum((w.detach() / w[0].numel() * rho).sum() + Q.sum() for w, (rho, Q) in zip(ws, out)).backward()
        for w, ref in zip(ws, single):
            close(w.grad.cpu().numpy(), ref, 1e-11)


I3 = (1, 0, 0, 0, 1, 0, 0, 0, 1)
INV = ((-1, 0, 0, 0, -1, 0, 0, 0, -1), (0, 0, 0))
CENTRED = {"body": [INV, (I3, (.5, .5, .5))], "A": [(I3, (0, .5, .5))], "B": [INV, (I3, (.5, 0, .5))],
           "half edge": [(I3, (0, 0, .5))]}


@pytest.mark.parametrize("grid", [(12, 16, 16), (16, 12, 24), (16, 24, 32)], ids=lambda g: "%dx%dx%d" % g)
@pytest.mark.parametrize("name", list(CENTRED))
def test_centred_planes(name, grid, backend):
    """Translations along z: the z lines of half the edge, with even or odd kz."""
    lib = get_lib(backend)
    cell = ("orthorhombic", [2.0, 2.4, 2.2])
    S, P = make(cell, CENTRED[name], grid, lib, 0), make(cell, [], grid, lib, 0)
    rng = np.random.default_rng(31)
    stars = np.zeros((2, S.N_star))
    stars[:, :14] = rng.normal(0.0, 1.0, (2, 14))
    rho, q, _ = S.density(stars)
    got = S.grids()[1]
    points = [(c, d, p) for c in (0, 1) for d in (1, -1) for p in (1, 4)]
    qs = [S.q(*p) for p in points]
    w = adjoint.stars_to_grid(S, torch.tensor(stars, device=lib.tensor_device)).detach()
    want, Q = adjoint.density(P, w)
    close(got, want.cpu().numpy())
    close(q, Q.cpu().numpy())
    for p, v in zip(points, qs):
        close(v, P.q(*p))
    many = S.density_many(np.stack([stars, 0.5 * stars]))
    assert np.array_equal(many[0][0], rho)
