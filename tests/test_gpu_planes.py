"""Batched solves on the planes of the principal layers (nt_planes.hip).

Systems whose layers are made of planes of given sizes (couplings only inside
a plane and to the next one), with the degrees of freedom of every layer in
random order, so that the planes have to be found: sizes at the edges of the
kernels' 16-column tiles and classes (16, 32, 48, 64, 96), planes of different
sizes, leads of other sizes than the device, several k-points whose patterns
differ.  T against the C oracle per point to max(1e-10, 256 eps kappa) (kappa
the largest condition number the oracle inverts), gradients and left-out
points against the layer path, which the planes replace."""
import dataclasses

import numpy as np
import pytest

import oracle as O
from phinfortran_amd import _native as N
from phinfortran_amd import lattice as lt

pytestmark = pytest.mark.gpu

EPS = 2.220446049250313e-16


@pytest.fixture(scope="module")
def T():
    from phinfortran_amd import transport
    return transport


@pytest.fixture
def planes_on(engine):
    yield
    engine.set_planes(True)


def oparams(p):
    return O.OrParams(p.eta, p.eta0, p.convergence, p.device_eta_factor, p.eta_mode, p.max_iter)


def plane_blocks(lead, dev, L, seed, lead_r=None, density=1.0, order_seed=0, flat_lead=None, flat_dev=None):
    """Block set whose lead cells and device layers consist of planes of the
    sizes lead (lead_r on the right) and dev, each layer's degrees of freedom
    in a random order (of order_seed: the same for all k-points of a system).
    The leads are periodic; density thins the couplings.  flat_lead, flat_dev:
    energy of the sites of every cell's or layer's second plane, which then are
    not coupled to one another."""
    rng = np.random.default_rng(seed)
    lead_r = lead if lead_r is None else lead_r

    def c(m, n):
        x = (rng.standard_normal((m, n)) + 1j * rng.standard_normal((m, n))) / np.sqrt(max(m, n))
        return x * (rng.random((m, n)) < density)

    def herm(n):
        x = c(n, n)
        return 0.5 * (x + x.conj().T)

    def layer(sizes, flat=None):
        off = np.concatenate([[0], np.cumsum(sizes)])
        H = np.zeros((off[-1], off[-1]), np.complex128)
        for i, n in enumerate(sizes):
            H[off[i]:off[i + 1], off[i]:off[i + 1]] = herm(n) if flat is None or i != 1 else flat * np.eye(n)
            if i + 1 < len(sizes):
                u = c(n, sizes[i + 1])
                H[off[i]:off[i + 1], off[i + 1]:off[i + 2]] = u
                H[off[i + 1]:off[i + 2], off[i]:off[i + 1]] = u.conj().T
        return H, off

    def couple(a, oa, b, ob):
        """last plane of a to first plane of b"""
        V = np.zeros((oa[-1], ob[-1]), np.complex128)
        V[oa[-2]:oa[-1], ob[0]:ob[1]] = c(a[-1], b[0])
        return V
    Hl, ol = layer(lead, flat_lead)
    Hr, orr = layer(lead_r, flat_lead)
    Vl = couple(lead, ol, lead, ol)                     # V_{-1,0}
    Vr = couple(lead_r, orr, lead_r, orr).conj().T      # V_{N+2,N+1}
    Hd = [layer(dev, flat_dev) for _ in range(L)]
    od = Hd[0][1]
    order = np.random.default_rng(order_seed)
    perm = [order.permutation(od[-1]) for _ in range(L)]
    pl, pr = order.permutation(ol[-1]), order.permutation(orr[-1])
    return lt.Blocks(
        Haml=Hl[np.ix_(pl, pl)], Hamlv=Vl[np.ix_(pl, pl)], Hamr=Hr[np.ix_(pr, pr)], Hamrv=Vr[np.ix_(pr, pr)],
        Hamd=np.stack([Hd[i][0][np.ix_(perm[i], perm[i])] for i in range(L)]),
        Hamdv=np.stack([couple(dev, od, dev, od)[np.ix_(perm[i], perm[i + 1])] for i in range(L - 1)]) if L > 1
        else np.zeros((0, od[-1], od[-1]), np.complex128),
        Hamld=couple(lead, ol, dev, od)[np.ix_(pl, perm[0])],
        Hamrd=couple(dev, od, lead_r, orr).conj().T[np.ix_(pr, perm[-1])])


def planes_launches(engine, call):
    engine.profile_reset()
    engine.profile(True)
    r = call()
    engine.profile(False)
    return r, engine.profile_get(N.NT_K_PLANES)["launches"], engine.profile_get(N.NT_K_INV)["launches"]


CASES = [((1, 1), (1, 1), 1, None), ((9, 9), (9, 9), 3, None), ((16, 16), (16, 16), 2, None),
         ((17, 16), (16, 17), 2, None), ((5, 7, 6), (7, 5, 6, 4), 3, (8, 7)), ((32, 32), (32, 32), 2, None),
         ((33, 20), (20, 33), 2, None), ((48, 48, 48, 48), (48, 48), 2, None), ((49, 48), (30, 49), 2, None),
         ((64, 64), (64, 64, 64), 1, None), ((63, 40, 50), (64, 33), 2, (40, 64)),
         # planes of 65 to 96: the leads through the layers' decimation
         ((70, 66), (65, 96), 2, None), ((65, 70, 80), (96, 70), 1, (66, 90, 70)),
         ((65, 66, 67, 68), (66, 65), 1, None)]


@pytest.mark.parametrize("lead,dev,L,lead_r", CASES)
def test_planes_vs_oracle(engine, T, planes_on, lead, dev, L, lead_r):
    p = T.params("phonon", eta=1e-3, eta0=1e-4, convergence=1e-13)
    blocks = [plane_blocks(lead, dev, L, 10 * L + i, lead_r) for i in range(2)]
    rng = np.random.default_rng(3)
    E = rng.uniform(0.05, 0.9, 9)
    kidx = rng.integers(0, 2, E.size).astype(np.int32)
    mask = np.zeros(E.size, np.int32)
    mask[2] = 1
    print(f"planes: lead {lead} device {dev} L={L}", flush=True)
    d = engine.upload_blocks(blocks)
    r, used, inverses = planes_launches(engine, lambda: engine.solve_tdb(d, E, p, kidx=kidx, first_point_mask=mask))
    assert used > 0 and (inverses == 0 or max(lead + dev) > 64)
    assert (r["status"].cpu().numpy() == 0).all()
    for i in range(2):
        sel = (kidx == i) & (mask == 0)
        if not sel.any():
            continue
        otl, otr, ost, kap = O.solve_tdb_batch_kappa(blocks[i].as_dict(), E[sel], oparams(p), nthreads=4)
        tol = np.maximum(1e-10, 256 * EPS * kap)
        assert (np.abs(r["T_LR"].cpu().numpy()[sel] - otl) <= tol * np.maximum(1.0, otl)).all()
        assert (np.abs(r["T_RL"].cpu().numpy()[sel] - otr) <= tol * np.maximum(1.0, otr)).all()
    assert float(r["T_LR"][2]) == 0.0
    # the recursion's own counts of steps
    engine.set_planes(False)
    q = engine.solve_tdb(d, E, p, kidx=kidx, first_point_mask=mask)
    assert np.array_equal(r["iters"].cpu().numpy(), q["iters"].cpu().numpy())


@pytest.mark.parametrize("dev,lo,hi", [((9, 9), 0, 2), ((16, 20), 1, 1), ((33, 20, 40), 2, 2), ((64, 30), 0, 1),
                                       ((90, 65), 0, 2)])
def test_planes_gradient(engine, T, planes_on, dev, lo, hi):
    """the gradient of the planes' sweep against the layers', whose own test is
    finite differences; sums over 11 points of two k-points.  Tolerance: dT =
    2 Re Tr[dH G Gamma G^+ Gamma G] has three factors G, each good to 256 eps
    kappa (kappa the largest condition number the oracle inverts)."""
    p = T.params("phonon", eta=1e-3, eta0=1e-4, convergence=1e-13)
    blocks = [plane_blocks((12, 10) if max(dev) <= 64 else (66, 65), dev, 3, 50 + i) for i in range(2)]
    rng = np.random.default_rng(4)
    E = rng.uniform(0.05, 0.9, 11)
    kidx = rng.integers(0, 2, 11).astype(np.int32)
    w = rng.uniform(0.5, 2.0, 11)
    d = engine.upload_blocks(blocks)
    print(f"planes gradient: device {dev} window {lo}..{hi}", flush=True)
    r, used, inverses = planes_launches(engine, lambda: engine.solve_tdb_adjoint(d, E, p, w, lo, hi, kidx=kidx))
    assert used > 0 and (inverses == 0 or max(dev) > 64)
    engine.set_planes(False)
    q = engine.solve_tdb_adjoint(d, E, p, w, lo, hi, kidx=kidx)
    kap = max(O.solve_tdb_batch_kappa(blocks[i].as_dict(), E[kidx == i], oparams(p), nthreads=4)[3].max()
              for i in range(2) if (kidx == i).any())
    tol = max(1e-10, 3 * 256 * EPS * kap)
    print(f"  kappa {kap:.1e}, tolerance {tol:.1e}", flush=True)
    for k in ("T_LR", "T_RL", "dHamd", "dHamdv"):
        x, y = r[k].cpu().numpy(), q[k].cpu().numpy()
        assert x.shape == y.shape and np.abs(x - y).max(initial=0.0) <= tol * max(1.0, np.abs(y).max(initial=0.0)), k


def test_left_out_points_are_the_layers(engine, T, planes_on):
    """A plane of uncoupled sites at their own energy, at no broadening to speak
    of: the plane is singular there though its layer is not.  Those points come
    from the layers, bit for bit, the others from the planes."""
    blk = lt.agnr_blocks(n_dimer=9, L=3, onsite_w=0.0, hop_noise=0.0)
    p = T.params("tb", eta=1e-9, convergence=1e-12)
    E = np.array([0.7, 0.0, -1.3, 1e-14, 0.9])
    d = engine.upload_blocks(blk)
    r, used, inverses = planes_launches(engine, lambda: engine.solve_tdb(d, E, p))
    assert used > 0 and inverses > 0
    engine.set_planes(False)
    engine.set_inverse_panel(18, 16)       # their inverses keep to the panel kernels
    q = engine.solve_tdb(d, E, p)
    engine.set_inverse_panel(18, 0)
    for k in ("T_LR", "T_RL", "status", "iters"):
        x, y = r[k].cpu().numpy(), q[k].cpu().numpy()
        assert np.array_equal(x[[1, 3]], y[[1, 3]], equal_nan=True), (k, x, y)
        assert np.allclose(x, y, rtol=1e-6, atol=1e-9, equal_nan=True), (k, x, y)


@pytest.mark.parametrize("what", ["dense", "nan", "not hermitian"])
def test_what_stays_on_the_layers(engine, T, planes_on, what):
    """dense blocks have no planes; a block with a NaN fails on either path
    with the same status; leads that are not Hermitian are not decimated on
    planes (the adjoint of the advanced function is not the retarded one)"""
    p = T.params("phonon", eta=1e-3, eta0=1e-4, convergence=1e-13)
    blk = plane_blocks((9, 8), (9, 8), 2, 5) if what != "dense" else lt.random_blocks(12, 12, 2, seed=3)
    E = np.array([0.1, 0.4, 0.8])
    if what == "nan":
        H = blk.Hamd.copy()
        i = np.argwhere(np.abs(H[0]) > 0)[0]
        H[0, i[0], i[1]] = np.nan
        blk = dataclasses.replace(blk, Hamd=H)
    if what == "not hermitian":
        H = blk.Haml.copy()
        i = np.argwhere(np.triu(np.abs(H), 1) > 0)[0]
        H[i[0], i[1]] *= 1.001
        blk = dataclasses.replace(blk, Haml=H)
    d = engine.upload_blocks(blk)
    r, used, _ = planes_launches(engine, lambda: engine.solve_tdb(d, E, p))
    assert (used > 0) == (what == "nan")
    engine.set_planes(False)
    q = engine.solve_tdb(d, E, p)
    for k in ("T_LR", "T_RL", "status", "iters"):
        assert np.array_equal(r[k].cpu().numpy(), q[k].cpu().numpy(), equal_nan=True), k


def test_noalloc_and_no_check_agree(engine, T, planes_on):
    """the allocation-free entry and the solve without host synchronisation
    run the same kernels: the same bits"""
    p = T.params("phonon", eta=1e-3, eta0=1e-4, convergence=1e-13, max_iter=48)
    d = engine.upload_blocks(plane_blocks((20, 33), (33, 20), 3, 9))
    E = np.linspace(0.05, 0.9, 21)
    ref = engine.solve_tdb(d, E, p)
    try:
        for every in (4, 0):
            engine.set_decimation_check(every)
            for noalloc in (False, True):
                print(f"check every {every}, noalloc {noalloc}", flush=True)
                r = engine.solve_tdb(d, E, p, noalloc=noalloc)
                for k in ("T_LR", "T_RL", "status", "iters"):
                    assert np.array_equal(ref[k].cpu().numpy(), r[k].cpu().numpy()), (every, noalloc, k)
    finally:
        engine.set_decimation_check(4)


@pytest.mark.parametrize("points", [63, 131, 300])
def test_gradient_parts(engine, points):
    """The window's sums over the points in parts side by side (from 1024 rows
    of a k-point on) with points left over, against the same points in calls
    too small to be split, whose gradients add up: the order of the sums is all
    that differs, so they agree to the number of points times eps of the
    largest sum of moduli."""
    from phinfortran_amd import lattice as lt
    from phinfortran_amd import transport as T
    blk = lt.si_ge_interface_film(nx=2, ny=1, L=6, kfrac=(0.125, 0.25))
    p = T.params("phonon")
    E = np.linspace(2.0, 14.0, points) ** 2
    d = engine.upload_blocks(blk)
    w = np.linspace(0.5, 1.5, points)
    print(f"gradient parts, {points} points", flush=True)
    whole = engine.solve_tdb_adjoint(d, E, p, w, 1, 4)
    parts = [engine.solve_tdb_adjoint(d, E[i:i + 15], p, w[i:i + 15], 1, 4) for i in range(0, points, 15)]
    for k in ("dHamd", "dHamdv"):
        got = whole[k].cpu().numpy()
        each = [r[k].cpu().numpy() for r in parts]
        bound = points * np.finfo(float).eps * sum(np.abs(x) for x in each).max()
        assert np.abs(got - sum(each)).max() <= 16 * bound


@pytest.mark.parametrize("seed,nw,at,res", [(22, 512, 145, 7.5e-6), (21, 1024, 361, 4.7e-6), (17, 1024, 249, 1.2e-7)])
def test_lossy_leads_come_from_the_layers(engine, T, planes_on, seed, nw, at, res):
    """Frequencies at which successive steps of a lead's decimation are nearly
    singular: planes and layers lose different digits there (T to 1e-5, the
    gradient to 6e-5 of its norm).  With the residual res of the self-energy
    over its bound (1e-6, for gradients 1e-7) it comes from the layers, and what
    is left is the sweep's rounding, 5e-16 kappa (kappa <= 1e5, three factors G in
    the gradient).  Below the bound T was seen to move by up to 10 times the
    residual and the gradient by 30."""
    rng = np.random.default_rng(seed)
    kf = tuple(rng.uniform(-0.5, 0.5, 2))
    springs = rng.uniform(0.95, 1.05, (2, lt.DiamondLayer(4, 2, periodic=True).nbond))
    blk = lt.si_ge_interface_film(nx=4, ny=2, L=40, kfrac=kf, iface_springs=springs)
    E = (16.0 * (np.arange(nw) + rng.uniform(0.25, 1.0)) / nw)[at - 2:at + 3] ** 2
    p = T.params("phonon")
    d = engine.upload_blocks(blk)
    print(f"lossy leads: seed {seed}, E = {E[2]:.5f}", flush=True)
    r, used, _ = planes_launches(engine, lambda: engine.solve_tdb(d, E, p))
    g = [engine.solve_tdb_adjoint(d, E[i:i + 1], p, np.ones(1), 12, 28) for i in range(5)]
    engine.set_planes(False)
    q = engine.solve_tdb(d, E, p)
    h = [engine.solve_tdb_adjoint(d, E[i:i + 1], p, np.ones(1), 12, 28) for i in range(5)]
    assert used > 0
    for k in ("T_LR", "T_RL"):
        x, y = r[k].cpu().numpy(), q[k].cpu().numpy()
        tol = np.full(5, 1e-5)
        if res > 1e-6:
            tol[2] = 1e-10
        assert (np.abs(x - y) <= tol * np.maximum(1.0, y)).all(), k
    for i in range(5):
        for k in ("dHamd", "dHamdv"):
            x, y = g[i][k].cpu().numpy(), h[i][k].cpu().numpy()
            rel = np.linalg.norm(x - y) / np.linalg.norm(y)
            print(f"  {k} point {i}: {rel:.1e}", flush=True)
            assert rel <= (3e-10 if i == 2 else 3e-6), (i, k)


@pytest.mark.parametrize("lead,dev,flat_lead,flat_dev,L", [
    ((20, 20), (13, 14, 13), None, 0.3, 3), ((20, 20), (13, 14, 13), None, 0.3, 1),
    ((30, 31, 30), (30, 30), 0.3, None, 2), ((30, 31, 30, 29), (30, 30), 0.3, None, 2),
    ((30, 30), (30, 31, 30), None, 0.3, 2),
    ((66, 65), (65, 70, 65), None, 0.3, 1), ((66, 70, 66), (66, 65), 0.3, None, 1),
    ((66, 70, 66, 65), (66, 65), 0.3, None, 1)])
def test_nearly_singular_planes(engine, T, planes_on, lead, dev, flat_lead, flat_dev, L):
    """Planes of uncoupled sites next to planes of fewer, at E near the sites'
    energy and at a small broadening: the plane is nearly singular where its
    layer is not.  T against the oracle to max(1e-10, 256 eps kappa), as
    everywhere (on the planes alone it is off by 1e-16 scale / |E - site|)."""
    blk = plane_blocks(lead, dev, L, 7, flat_lead=flat_lead, flat_dev=flat_dev)
    p = T.params("phonon", eta=1e-8, eta0=1e-9, convergence=1e-13)
    E = 0.3 + np.array([0.0, 1e-8, -1e-7, 1e-6, -1e-5, 1e-4, 1e-3, -1e-2])
    print(f"nearly singular planes: lead {lead} device {dev} L={L}", flush=True)
    d = engine.upload_blocks(blk)
    r, used, _ = planes_launches(engine, lambda: engine.solve_tdb(d, E, p))
    assert used > 0 and (r["status"].cpu().numpy() == 0).all()
    otl, otr, ost, kap = O.solve_tdb_batch_kappa(blk.as_dict(), E, oparams(p), nthreads=4)
    tol = np.maximum(1e-10, 256 * EPS * kap)
    for k, o in (("T_LR", otl), ("T_RL", otr)):
        err = np.abs(r[k].cpu().numpy() - o) / np.maximum(1.0, o)
        print(f"  {k}: " + " ".join(f"{e:.1e}/{t:.1e}" for e, t in zip(err, tol)), flush=True)
        assert (err <= tol).all(), k


@pytest.mark.parametrize("lead,dev", [((9, 8), (9, 8)), ((13, 14, 13), (13, 14, 13)), ((66, 70, 66), (66, 65))])
def test_planes_in_other_units(engine, T, planes_on, lead, dev):
    """energies in units 2^80 times as large or small: the same T to the bit
    (powers of two), all points on the planes"""
    E = np.array([0.1, 0.4, 0.8])
    blk = plane_blocks(lead, dev, 2, 5)
    ref = None
    for u in (1.0, 2.0 ** 80, 2.0 ** -80):
        p = T.params("phonon", eta=1e-3, eta0=1e-4 * u, convergence=1e-13 * u)
        b = lt.Blocks(**{k: v * u for k, v in blk.as_dict().items()})
        print(f"planes {lead} {dev} in units of {u:.1e}", flush=True)
        d = engine.upload_blocks(b)
        r, used, inverses = planes_launches(engine, lambda: engine.solve_tdb(d, E * u, p))
        assert used > 0 and (inverses == 0 or max(lead) > 64)
        t = np.stack([r[k].cpu().numpy() for k in ("T_LR", "T_RL", "iters", "status")])
        ref = t if ref is None else ref
        assert np.array_equal(t, ref)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_some_points_left_without_waiting(engine, T, planes_on, prec):
    """The allocation-free entry and the solve without host synchronisation with
    some points left to the layers and some not (the ribbon's uncoupled sites at
    E, and two energies beside them): the former by the layers' launches under a
    mask, in FP64 whatever the precision, the latter keep what the planes gave."""
    blk = lt.agnr_blocks(n_dimer=9, L=3, onsite_w=0.0, hop_noise=0.0)
    E = np.array([0.7, 0.0, -1.3, 1e-14, 0.9, 0.31, 0.0, 1.1])
    left = np.abs(E) < 0.1
    d = engine.upload_blocks(blk)
    par = {k: T.params("tb", eta=1e-9, convergence=1e-12, precision=k, max_iter=60) for k in ("fp64", prec)}
    ref, used, _ = planes_launches(engine, lambda: engine.solve_tdb(d, E, par["fp64"]))
    assert used > 0
    engine.set_planes(False)
    engine.set_inverse_panel(18, 16)
    lay = engine.solve_tdb(d, E, par["fp64"])
    engine.set_inverse_panel(18, 0)
    engine.set_planes(True)
    want = {k: np.where(left, lay[k].cpu().numpy(), ref[k].cpu().numpy()) for k in ("T_LR", "T_RL", "status", "iters")}
    try:
        for every, noalloc in ((4, True), (0, False), (0, True)):
            print(f"left points {prec}: check every {every}, noalloc {noalloc}", flush=True)
            engine.set_decimation_check(every)
            r, used, _ = planes_launches(engine, lambda: engine.solve_tdb(d, E, par[prec], noalloc=noalloc))
            assert used > 0
            for k, v in want.items():
                assert np.array_equal(r[k].cpu().numpy(), v, equal_nan=True), (every, noalloc, k, r[k], v)
    finally:
        engine.set_decimation_check(4)


@pytest.mark.parametrize("noalloc", [False, True])
def test_mixed_counts_all_points(engine, T, planes_on, noalloc):
    """every point of a mixed-precision call is counted in that call, those
    solved on the layers by a worker context too (the energy of the uncoupled
    sites of a lead's plane, without broadening)"""
    d = engine.upload_blocks(plane_blocks((30, 31, 30), (30, 30), 2, 7, flat_lead=0.3))
    E = np.array([0.1, 0.3, 0.5])
    p = T.params("tb", eta=0.0, convergence=1e-12, precision="mixed", max_iter=60)
    for _ in range(2):
        engine.profile_reset()
        _, used, _ = planes_launches(engine, lambda: engine.solve_tdb(d, E, p, noalloc=noalloc))
        assert used > 0 and engine.mixed_counts()[0] == E.size


@pytest.mark.parametrize("limit", [1, 8, 21])
def test_batch_limit_holds_on_planes(engine, T, planes_on, limit):
    """at most that many points per chunk, a decimation and a sweep each"""
    p = T.params("phonon", eta=1e-3, eta0=1e-4, convergence=1e-13)
    blk = plane_blocks((20, 33), (33, 20), 3, 9)
    E = np.linspace(0.05, 0.9, 21)
    ref = engine.solve_tdb(engine.upload_blocks(blk), E, p)
    eng = T.Engine(0, batch_limit=limit)
    try:
        d = eng.upload_blocks(blk)
        r, used, _ = planes_launches(eng, lambda: eng.solve_tdb(d, E, p))
        assert used == 2 * -(-E.size // limit)
        for k in ("T_LR", "T_RL", "status", "iters"):
            assert np.array_equal(ref[k].cpu().numpy(), r[k].cpu().numpy()), k
    finally:
        eng.close()


def test_no_check_reserves_no_more_than_its_budget(engine, T, planes_on):
    """Without host waits the planes' blocks are reserved by their bound, the
    largest class for every plane and k-point: where that takes gigabytes (here
    9 of them for 130 MB of blocks) the layers solve the call."""
    import torch
    blk = plane_blocks((16, 16), (16, 16), 30, 5)
    nk = 256
    E = np.full(nk, 0.4)
    kidx = np.arange(nk, dtype=np.int32)
    p = T.params("phonon", eta=1e-3, eta0=1e-4, convergence=1e-13, max_iter=32)
    eng = T.Engine(0, batch_limit=64)
    try:
        d = eng.upload_blocks([blk] * nk)
        ref = eng.solve_tdb(d, E, p, kidx=kidx)
        eng.close()
        eng = T.Engine(0, batch_limit=64)
        eng.set_decimation_check(0)
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        r = eng.solve_tdb(d, E, p, kidx=kidx)
        torch.cuda.synchronize()
        took = before - torch.cuda.mem_get_info()[0]
        print(f"took {took / 2 ** 30:.2f} GiB", flush=True)
        assert took < 6 * 2 ** 30
        assert np.abs(r["T_LR"].cpu().numpy() - ref["T_LR"].cpu().numpy()).max() < 1e-8
    finally:
        eng.close()
