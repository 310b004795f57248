"""Adjoint RGF on the GPU: gradients of sum_i w_i T_LR(i) with respect to the
device blocks against the dense formula (itself pinned to finite differences
of the oracle in test_adjoint_cpu.py), and dG/dbeta of the interface-film
conductance against central finite differences of the oracle's FP64 T
(h = 1e-4 N/m, 32 seeded bonds, agreement to 1e-5 relative)."""
import numpy as np
import pytest

import oracle as O
from adjoint_ref import T_and_grad
from phinfortran_amd import lattice as lt

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("both_paths")]


def oparams(p):
    return O.OrParams(p.eta, p.eta0, p.convergence, p.device_eta_factor, p.eta_mode, p.max_iter)


@pytest.fixture(scope="module")
def T():
    from phinfortran_amd import transport
    return transport


@pytest.mark.parametrize("nl,b,L,lo,hi,nk", [(4, 4, 5, 1, 3, 1), (12, 12, 6, 2, 3, 2), (24, 24, 4, 0, 3, 2),
                                             (20, 20, 3, 2, 2, 1)])
def test_adjoint_blocks_vs_dense(engine, T, nl, b, L, lo, hi, nk):
    blocks = [lt.random_blocks(nl, b, L, seed=40 + i) for i in range(nk)]
    p = T.params("phonon", eta=1e-3, eta0=1e-4, convergence=1e-13)
    op = oparams(p)
    rng = np.random.default_rng(5)
    npts = 11
    E = rng.uniform(0.05, 0.9, npts)
    kidx = rng.integers(0, nk, npts).astype(np.int32)
    w = rng.uniform(0.5, 2.0, npts)
    mask = np.zeros(npts, np.int32)
    mask[3] = 1
    print(f"adjoint nl={nl} b={b} L={L} window=[{lo},{hi}] nk={nk}", flush=True)
    d = engine.upload_blocks(blocks)
    r = engine.solve_tdb_adjoint(d, E, p, w, lo, hi, kidx=kidx if nk > 1 else None, first_point_mask=mask)
    r0 = engine.solve_tdb(d, E, p, kidx=kidx if nk > 1 else None, first_point_mask=mask)
    assert (r["status"].cpu().numpy() == 0).all()
    assert np.abs(r["T_LR"].cpu().numpy() - r0["T_LR"].cpu().numpy()).max() < 1e-12
    nc = min(hi, L - 2) - lo + 1
    ref_d = np.zeros((nk, hi - lo + 1, b, b), complex)
    ref_v = np.zeros((nk, max(nc, 0), b, b), complex)
    for i in range(npts):
        if mask[i]:
            continue
        k = kidx[i] if nk > 1 else 0
        _, gd, gv = T_and_grad(blocks[k], E[i], op, lo, hi)
        ref_d[k] += w[i] * gd
        if nc > 0:
            ref_v[k] += w[i] * gv
    gd = r["dHamd"].cpu().numpy()
    gv = r["dHamdv"].cpu().numpy()
    assert np.abs(gd - ref_d).max() < 1e-8 * np.abs(ref_d).max()
    if nc > 0:
        assert np.abs(gv - ref_v).max() < 1e-8 * np.abs(ref_v).max()


def _film(engine, T, nx=1, ny=1, L=6, nf=12):
    from phinfortran_amd.adjoint import InterfaceFilm
    p = T.params("phonon", eta=1e-4, eta0=1e-5, convergence=1e-12, max_iter=400)
    f = np.linspace(0.4, 15.5, nf)
    return InterfaceFilm(engine, nx, ny, L, [(0.0, 0.0), (0.25, 0.125)], f, n_iface=2, params=p)


def test_film_gradient_vs_oracle_fd(engine, T):
    """dG/dbeta (adjoint, GPU) against central differences of G computed with
    the oracle's FP64 solve on the CPU, h = 1e-4 N/m, 32 seeded bonds."""
    import torch
    film = _film(engine, T)
    rng = np.random.default_rng(7)
    beta = 13.8 + 0.5 * rng.standard_normal(film.nparam)
    G, g, _ = film.conductance(torch.as_tensor(beta, device=film.dev))
    g = g.cpu().numpy()
    op = oparams(film.p)
    w = film.weight.cpu().numpy().reshape(film.nk, film.nf)
    E = film.f ** 2

    def G_oracle(bv):
        tot = 0.0
        for k in range(film.nk):
            blk = film.blocks_numpy(bv, k).as_dict()
            tl, _, st = O.solve_tdb_batch(blk, E, op, nthreads=8)
            assert (np.asarray(st) == 0).all()
            tl = np.asarray(tl).copy()
            tl[0] = 0.0                         # the ie = 1 point
            tot += float(np.dot(w[k], tl))
        return tot
    G_or = G_oracle(beta)
    assert abs(float(G) - G_or) < 1e-9 * abs(G_or)
    h = 1e-4
    bonds = rng.choice(film.nparam, 32, replace=False)
    scale = np.abs(g).max()
    for n in bonds:
        e = np.zeros(film.nparam)
        e[n] = h
        fd = (G_oracle(beta + e) - G_oracle(beta - e)) / (2 * h)
        assert abs(fd - g[n]) < 1e-5 * max(abs(fd), 1e-3 * scale), (n, fd, g[n])


def test_autograd_function_and_adam(engine, T):
    import torch
    from phinfortran_amd.adjoint import conductance, maximize_conductance
    film = _film(engine, T, nf=10)
    beta = torch.full((film.nparam,), 13.8, dtype=torch.float64, device=film.dev)
    x = beta.clone().requires_grad_(True)
    G = conductance(x, film)
    G.backward()
    _, g, _ = film.conductance(beta)
    assert torch.allclose(x.grad, g, rtol=1e-12, atol=0)
    _, hist = maximize_conductance(film, beta, steps=6, lr=0.5)
    assert hist[-1] > hist[0]
