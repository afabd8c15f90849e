"""Sweeps of 1D and 2D grids (N3 = 1) against contour steps in numpy.

The edges cover each line length in one and two dimensions, rectangular
planes, lines of one thread, and the edges (96, 128) that take the step
kernels instead of the one-launch sweep.  Fields are random, without any
symmetry.  One contour step of FP64 transforms agrees to 1e-13 of the largest
value (the bound of the reference's own steps); a sweep of n steps to n times
that.
"""
import numpy as np
import pytest
import torch

from conftest import get_lib

from pscf_amd import adjoint, iterate, scf
from pscf_amd.system import System

GRIDS = [(8, 1), (12, 1), (20, 1), (56, 1), (96, 1), (128, 1), (8, 8), (8, 16), (12, 20), (16, 8),
         (24, 12), (28, 28), (40, 24), (48, 48), (64, 64), (28, 56), (96, 96)]


def step(q, w, ds, b, ksq):
    def conv(x, f):
        return np.fft.irfftn(f * np.fft.rfftn(x), s=x.shape, axes=(0, 1, 2))
    e1, e2 = np.exp(-ds / 2 * w), np.exp(-ds / 4 * w)
    k1, k2 = np.exp(-ds * b * b / 6 * ksq), np.exp(-ds * b * b / 12 * ksq)
    q1 = e1 * conv(e1 * q, k1)
    q2 = e2 * conv(e1 * conv(e2 * q, k2), k2)
    return (4.0 * q2 - q1) / 3.0


@pytest.mark.parametrize("grid", GRIDS, ids=lambda g: "%dx%d" % g)
def test_one_step(grid, backend):
    lib = get_lib(backend)
    ng = [grid[0], grid[1], 1]
    rng = np.random.default_rng(grid[0] * 200 + grid[1])
    St = scf.Step(ng, lib=lib)
    w, q = rng.normal(size=St.shape), rng.uniform(0.1, 1.5, St.shape)
    k = [np.minimum(np.arange(n), n - np.arange(n)) * g for n, g in zip(grid, (2.1, 2.9))]
    ksq = (k[0][None, :grid[0] // 2 + 1] ** 2 + k[1][:, None] ** 2)[None]
    St.make_propg(0.02, 1.2, ksq, w)
    got, want = St.step_exp(q), step(q, w, 0.02, 1.2, ksq)
    assert np.abs(got - want).max() <= 1e-13 * np.abs(want).max()


@pytest.mark.parametrize("stride", [0, 3])
@pytest.mark.parametrize("grid", [(12, 1), (64, 1), (8, 8), (24, 16), (40, 40)], ids=lambda g: "%dx%d" % g)
def test_sweeps(grid, stride, backend):
    """Two chains of several blocks, both directions, stored whole or recomputed
    from checkpoints, alone and grouped."""
    lib = get_lib(backend)
    dim = 2 if grid[1] > 1 else 1
    ng = list(grid[:dim])
    s = System(kuhn=[1.0, 1.2], chains=[[(1, 0.3), (2, 0.5), (1, 0.2)], [(2, 0.3)]], phi_chain=[0.8, 0.2],
               chi=np.array([[0.0, 15.0], [15.0, 0.0]]), dim=dim,
               crystal_system="rectangular" if dim == 2 else "lamellar",
               cell_param=[1.7, 2.2][:dim], ngrid=ng, chain_step=0.05, group_name="1")
    _, G, _ = iterate.unit_cell(lib, dim, s.crystal_system, np.array(s.cell_param))
    one = np.zeros((3, 3))
    one[:dim, :dim] = np.eye(dim)
    B = scf.Basis.from_tables(scf.Basis.build_tables(dim, ng, G, one.ravel()[None], np.zeros((1, 3)), lib=lib))
    S = scf.SCFSystem(s, B, G, lib=lib)
    S.set_checkpoint(stride)
    rng = np.random.default_rng(17)
    om = np.zeros((2, B.N_star))
    om[:, :12] = rng.normal(0.0, 1.5, (2, 12))
    w = adjoint.stars_to_grid(S, torch.tensor(om, device=lib.tensor_device)).detach().cpu().numpy()
    w = w.reshape((2,) + S.shape)
    ksq = S.ksq().reshape(S.shape[0], S.shape[1], -1)
    rho, Q, _ = S.density(om)
    want = np.zeros((2,) + S.shape)
    for c, chain in enumerate(s.chains):
        bgn, ds = scf.chain_discretize([L for _, L in chain], s.chain_step, lib=lib)
        steps = [(m - 1, d) for (m, _), d, a, b in zip(chain, ds, bgn, bgn[1:]) for _ in range(b - a)]
        qf, qr = [np.ones(S.shape)], [np.ones(S.shape)]
        for m, d in steps:
            qf.append(step(qf[-1], w[m], d, s.kuhn[m], ksq))
        for m, d in steps[::-1]:
            qr.append(step(qr[-1], w[m], d, s.kuhn[m], ksq))
        qr = qr[::-1]
        n = len(steps)
        q0 = qf[-1].mean()
        assert abs(Q[c] / q0 - 1.0) <= 1e-13 * n
        if stride == 0:
            for p in (0, 1, n // 2, n):
                for d, ref in ((1, qf), (-1, qr)):
                    got = S.q(c, d, p)
                    assert np.abs(got.reshape(S.shape) - ref[p]).max() <= 1e-13 * n * np.abs(ref[p]).max()
        N = sum(L for _, L in chain)
        for (m, _), d, a, b in zip(chain, ds, bgn - 1, bgn[1:] - 1):
            for p in range(a, b + 1):
                wt = 1.0 if p in (a, b) else (4.0 if (p - a) % 2 else 2.0)
                want[m - 1] += s.phi_chain[c] / (N * q0) * wt * d / 3.0 * qf[p] * qr[p]
    _, rg = S.grids()
    n = 2 * 20
    assert np.abs(rg.reshape(want.shape) - want).max() <= 1e-13 * n * np.abs(want).max()
    many = S.density_many(np.stack([om, 0.5 * om, om]))
    assert np.array_equal(many[0][0], rho) and np.array_equal(many[0][2], rho)
    assert np.array_equal(many[1][0], Q)
