"""Several devices of uneven block size and length in one call
(nt_solve_tdb_multi_dev) give exactly the per-device batched results, which
the oracle checks on a few points."""
import numpy as np
import pytest

import oracle as O
from phinfortran_amd import lattice as lt

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("both_paths")]


@pytest.fixture(scope="module")
def T():
    from phinfortran_amd import transport
    return transport


def test_multi_device_equals_single(engine, T):
    p = T.params("phonon", eta=1e-5, eta0=1e-6)
    op = O.OrParams(p.eta, p.eta0, p.convergence, p.device_eta_factor, p.eta_mode, p.max_iter)
    ks = lt.mp_grid(2, 2)
    specs = [dict(n=1, period=2, L=7), dict(n=2, period=3, L=4), dict(n=1, period=1, L=12)]
    devices, blocks = [], []
    rng = np.random.default_rng(0)
    for i, sp in enumerate(specs):
        blk = [lt.si_ge_superlattice_film(sp["n"], sp["period"], sp["L"], kf, seed=i) for kf in ks]
        blocks.append(blk)
        npts = 9
        E = (rng.uniform(0.5, 14.0, npts)) ** 2
        kidx = rng.integers(0, len(ks), npts).astype(np.int32)
        devices.append(dict(blocks=engine.upload_blocks(blk), E=E, kidx=kidx))
    print("multi-device", flush=True)
    outs = engine.solve_tdb_multi(devices, p)
    for i, (d, o) in enumerate(zip(devices, outs)):
        r = engine.solve_tdb(d["blocks"], d["E"], p, kidx=d["kidx"])
        assert (o["status"].cpu().numpy() == 0).all()
        assert np.abs(o["T_LR"].cpu().numpy() - r["T_LR"].cpu().numpy()).max() < 1e-12
        assert np.abs(o["T_RL"].cpu().numpy() - r["T_RL"].cpu().numpy()).max() < 1e-12
        for j in (0, 4):
            tl, tr, _ = O.solve_tdb(blocks[i][d["kidx"][j]].as_dict(), d["E"][j], op)
            assert abs(o["T_LR"][j].item() - tl) < 1e-9 * max(1, tl)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_multi_device_workers(engine, T, precision):
    """Twelve devices of four block sizes (groups sharing leads among them):
    the groups solved side by side by four worker contexts give bitwise the
    results of one after the other on the context itself, the caller's
    stream sees them without a further synchronisation, and the profile
    counts the workers' launches."""
    import torch
    from phinfortran_amd import _native as N
    p = T.params("phonon", precision=precision)
    ks = lt.mp_grid(2, 2)
    f = 16.0 * np.arange(1, 17) / 16
    devices = []
    for i, n in enumerate([1, 2, 3, 1, 2, 3, 1, 2, 1, 4, 1, 2]):
        blk = [lt.si_ge_superlattice_film(n, 2 + i % 3, 6 + 2 * i, kf, seed=40 + i) for kf in ks]
        devices.append(dict(blocks=engine.upload_blocks(blk), E=np.tile(f ** 2, 4),
                            kidx=np.repeat(np.arange(4, dtype=np.int32), f.size)))
    print(f"multi-device workers, {precision}", flush=True)
    try:
        engine.set_multi_workers(1)
        ref = engine.solve_tdb_multi(devices, p)
        engine.set_multi_workers(4)
        engine.profile_reset()
        engine.profile(True)
        got = engine.solve_tdb_multi(devices, p, stream_sync=False)
        # read on the caller's stream: ordered after the workers by the call
        tl = [o["T_LR"].clone() for o in got]
        torch.cuda.synchronize()
        engine.profile(False)
        prof = engine.profile_get(N.NT_K_GEMM)
    finally:
        engine.set_multi_workers(4)
        engine.profile(False)
    assert prof["launches"] > 0 and prof["ms"] > 0
    for i, (a, b, t) in enumerate(zip(ref, got, tl)):
        assert (b["status"].cpu().numpy() == 0).all(), i
        for k in ("T_LR", "T_RL"):
            assert torch.equal(a[k], b[k]), (i, k)
        assert torch.equal(t, a["T_LR"]), i


@pytest.mark.parametrize("with_extras", [True, False])
@pytest.mark.parametrize("parts,npts", [(2, 600), (3, 800)])
def test_point_split_equals_one_stream(engine, T, parts, npts, with_extras):
    """A batched FP64 solve of at least parts x 256 points runs as parts
    solved side by side by worker contexts (nt_set_point_split): bitwise the
    T, statuses, iteration counts and extras of the solve on one stream, and
    the caller's stream sees them without a further synchronisation.  Part q
    takes every parts-th point from q (inputs, results and extras gathered
    and scattered back)."""
    import torch
    ks = lt.mp_grid(2, 2)
    blocks = [lt.si_ge_superlattice_film(2, 2, 6, kf, seed=7) for kf in ks]
    d = engine.upload_blocks(blocks)
    f = 16.0 * (np.arange(npts) + 0.5) / npts
    E = f ** 2
    kidx = (np.arange(npts) % len(ks)).astype(np.int32)
    mask = np.zeros(npts, np.int32)
    mask[0] = 1
    p = T.params("phonon")
    ex = ("G_D_RL", "gl_adv", "G_L", "sdos_l", "ldos", "ddos") if with_extras else ()
    print(f"split solve, {parts} parts of {npts} points, extras {with_extras}", flush=True)
    try:
        engine.set_point_split(1)
        ref = engine.solve_tdb(d, E, p, kidx=kidx, first_point_mask=mask, extras=ex)
        it1 = engine.last_mean_iters()
        engine.set_point_split(parts)
        got = engine.solve_tdb(d, E, p, kidx=kidx, first_point_mask=mask, extras=ex, stream_sync=False)
        snap = {k: v.clone() for k, v in got.items()}       # on the caller's stream
        torch.cuda.synchronize()
        it2 = engine.last_mean_iters()
    finally:
        engine.set_point_split(2)
    assert (ref["status"].cpu().numpy() == 0).all()
    for k in ("T_LR", "T_RL", "status", "iters") + ex:
        assert torch.equal(ref[k], snap[k]), k
    assert abs(it1 - it2) < 1e-9 * max(1.0, it1)


@pytest.mark.parametrize("case", ["unequal_leads", "circular"])
def test_point_split_other_lead_paths(engine, T, case):
    """The two-part solve with leads of different sizes (one decimation batch
    per lead) and with the block-circulant decimation: bitwise the
    one-stream results, with and without extras."""
    import torch
    if case == "unequal_leads":
        blocks = [lt.random_blocks(8, 12, 4, nr=16, seed=40 + i, scale=0.7) for i in range(2)]
        p = T.params("phonon", eta=1e-3, eta0=1e-4)
    else:
        blocks = [lt.circulant_lead_blocks(3, 2, 2, 3, seed=s) for s in (1, 2)]
        p = T.params("phonon", eta=1e-3, eta0=1e-4, convergence=1e-13, circular=1, n_bloch_x=2, n_bloch_y=2)
    d = engine.upload_blocks(blocks)
    npts = 520
    E = np.linspace(0.05, 0.9, npts)
    kidx = (np.arange(npts) % 2).astype(np.int32)
    print(f"split solve, {case}", flush=True)
    for ex in ((), ("G_D_RL", "G_L")):
        try:
            engine.set_point_split(1)
            ref = engine.solve_tdb(d, E, p, kidx=kidx, extras=ex)
            engine.set_point_split(2)
            got = engine.solve_tdb(d, E, p, kidx=kidx, extras=ex)
        finally:
            engine.set_point_split(2)
        assert (ref["status"].cpu().numpy() == 0).all(), (case, ex)
        for k in ("T_LR", "T_RL", "status", "iters") + ex:
            assert torch.equal(ref[k], got[k]), (case, ex, k)


def test_point_split_adjoint(engine, T):
    """The adjoint solve of at least 2 x 256 points runs as two interleaved
    parts on worker contexts, the second part's gradients summed into the
    caller's at the end: T, statuses and iteration counts bitwise the
    one-stream solve's, the gradients to the rounding of the summation order
    (1e-12 of their largest element)."""
    import torch
    blocks = [lt.random_blocks(12, 12, 5, seed=60 + i, scale=0.7) for i in range(2)]
    d = engine.upload_blocks(blocks)
    p = T.params("phonon", eta=1e-3, eta0=1e-4, convergence=1e-13)
    npts = 530
    E = np.linspace(0.05, 0.9, npts)
    kidx = (np.arange(npts) % 2).astype(np.int32)
    w = np.random.default_rng(8).uniform(0.5, 2.0, npts)
    mask = np.zeros(npts, np.int32)
    mask[7] = 1
    print("split adjoint solve, 2 parts of 530 points", flush=True)
    try:
        engine.set_point_split(1)
        ref = engine.solve_tdb_adjoint(d, E, p, w, 1, 3, kidx=kidx, first_point_mask=mask)
        engine.set_point_split(2)
        got = engine.solve_tdb_adjoint(d, E, p, w, 1, 3, kidx=kidx, first_point_mask=mask)
    finally:
        engine.set_point_split(2)
    assert (ref["status"].cpu().numpy() == 0).all()
    for k in ("T_LR", "T_RL", "status", "iters"):
        assert torch.equal(ref[k], got[k]), k
    for k in ("dHamd", "dHamdv"):
        a, b = ref[k].cpu().numpy(), got[k].cpu().numpy()
        assert np.abs(a).max() > 0
        assert np.abs(a - b).max() < 1e-12 * np.abs(a).max(), k



def test_point_split_mixed(engine, T):
    """The mixed-precision solve split in two interleaved parts: T, statuses,
    iteration counts bitwise those of one stream, and the refinement counters
    (second steps, FP64 recomputes) summed over the parts equal."""
    import torch
    ks = lt.mp_grid(2, 2)
    blocks = [lt.si_ge_superlattice_film(2, 2, 6, kf, seed=7) for kf in ks]
    d = engine.upload_blocks(blocks)
    npts = 600
    f = 16.0 * (np.arange(npts) + 0.5) / npts
    E = f ** 2
    kidx = (np.arange(npts) % len(ks)).astype(np.int32)
    p = T.params("phonon", precision="mixed")
    print("split mixed solve, 2 parts of 600 points", flush=True)
    try:
        engine.set_point_split(1)
        c0 = np.array(engine.mixed_counts())
        ref = engine.solve_tdb(d, E, p, kidx=kidx)
        c1 = np.array(engine.mixed_counts())
        engine.set_point_split(2)
        got = engine.solve_tdb(d, E, p, kidx=kidx)
        c2 = np.array(engine.mixed_counts())
    finally:
        engine.set_point_split(2)
    assert (ref["status"].cpu().numpy() == 0).all()
    for k in ("T_LR", "T_RL", "status", "iters"):
        assert torch.equal(ref[k], got[k]), k
    assert np.array_equal(c1 - c0, c2 - c1), (c1 - c0, c2 - c1)
