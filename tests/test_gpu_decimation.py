"""Decimation of small dense leads in one kernel, at the sizes where its waves
and padding change and on both sides of the rule that selects it."""
import numpy as np
import pytest

import oracle as O
from phinfortran_amd import _native as N
from phinfortran_amd import lattice as lt
from phinfortran_amd import transport as T

pytestmark = pytest.mark.gpu


def planes_launches(engine, f):
    engine.profile_reset()
    engine.profile(True)
    try:
        r = f()
    finally:
        engine.profile(False)
    return r, engine.profile_get(N.NT_K_PLANES)["launches"]


@pytest.mark.parametrize("n,one", [(1, False), (12, False), (13, True), (15, True), (16, True), (17, False),
                                   (26, True), (32, True), (33, False), (38, True), (47, True), (48, True),
                                   (49, False), (51, True), (63, True), (64, True), (65, False)])
def test_surface_green_one_kernel(engine, n, one):
    """Every lead Green's function satisfies its Dyson fixed point as tightly
    as the oracle's, steps within one of the oracle's (max|alpha| may cross the
    convergence limit one step apart by rounding), and the size rule sends n
    where it says."""
    blk = lt.random_blocks(n, n, 1, seed=n)
    p = T.params("phonon", eta=1e-3, eta0=1e-4, convergence=1e-13)
    E = 0.37
    eta = E * p.eta + p.eta0
    print(f"decimation n={n}", flush=True)
    g, launches = planes_launches(
        engine, lambda: engine.surface_green_tdb(blk.Haml, blk.Hamr, blk.Hamlv, blk.Hamrv, E, p))
    assert (launches > 0) == one
    o = O.surface_green(blk.Haml, blk.Hamlv, blk.Hamr, blk.Hamrv, E,
                        O.OrParams(p.eta, p.eta0, p.convergence, p.device_eta_factor, p.eta_mode, p.max_iter))
    for k, H, V, z in (("gl_adv", blk.Haml, blk.Hamlv, E - 1j * eta), ("gr_ret", blk.Hamr, blk.Hamrv, E + 1j * eta)):
        def residual(x):
            return np.abs(x - np.linalg.inv(z * np.eye(n) - H - V.conj().T @ x @ V)).max() / np.abs(x).max()
        assert residual(g[k]) < 10 * residual(o[k]) + 1e-12
    assert all(abs(a - b) <= 1 for a, b in zip(g["iters"], o["iters"]))


@pytest.mark.parametrize("n", [16, 38, 48, 64])
def test_batched_against_launches(engine, n):
    """A batch on one kernel and, with a panel width of the caller's, as
    launches: statuses and step counts are equal; a NaN in a lead and an
    iteration limit end both the same way.  The steps of a dense random lead
    pass through matrices far worse conditioned than the result, by how much
    depends on the point, so T is held to the oracle's and the one kernel's
    largest difference to ten times that of the launches, itself the distance
    of two correct FP64 algorithms on these inputs."""
    blk = lt.random_blocks(n, n, 3, seed=n + 1)
    E = np.linspace(0.05, 0.9, 9)
    bad = lt.random_blocks(n, n, 3, seed=n + 1)
    bad.Haml[1, 1] = np.nan
    for b, kw in ((blk, {}), (blk, dict(max_iter=3)), (blk, dict(max_iter=1)), (bad, dict(max_iter=50))):
        p = T.params("phonon", eta=1e-3, eta0=1e-4, convergence=1e-13, **kw)
        out = []
        for width in (0, 8):
            engine.set_inverse_panel(n, width)
            try:
                r = engine.solve_tdb(engine.upload_blocks(b), E, p)
                out.append({k: r[k].cpu().numpy() for k in ("T_LR", "T_RL", "status", "iters")})
            finally:
                engine.set_inverse_panel(n, 0)
        assert np.array_equal(out[0]["status"], out[1]["status"])
        assert np.abs(out[0]["iters"] - out[1]["iters"]).max() <= 1
        if kw:
            assert np.array_equal(out[0]["iters"], out[1]["iters"])
        for k in ("T_LR", "T_RL"):
            assert np.array_equal(np.isnan(out[0][k]), np.isnan(out[1][k]))
        if not kw:
            op = O.OrParams(p.eta, p.eta0, p.convergence, p.device_eta_factor, p.eta_mode, p.max_iter)
            for k, t in zip(("T_LR", "T_RL"), O.solve_tdb_batch(blk.as_dict(), E, op)[:2]):
                one, launched = (np.abs(o[k] - t).max() for o in out)
                print(f"n={n} {kw} {k}: one kernel {one:.2e}, launches {launched:.2e}", flush=True)
                assert one <= 10 * launched + 1e-10 * max(1.0, np.abs(t).max())
