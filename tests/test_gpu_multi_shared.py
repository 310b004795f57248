"""Devices with the same leads and points in one multi-device call: the
engine computes their lead Green's functions once and runs each device's
sweep on them.  Results equal the per-device solves (which the oracle pins)
and the oracle on sampled points."""
import numpy as np
import pytest

import oracle as O
from phinfortran_amd import lattice as lt

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("both_paths")]


def test_shared_leads_equal_single_solves(engine):
    from phinfortran_amd import transport as T
    p = T.params("phonon")
    op = O.OrParams(p.eta, p.eta0, p.convergence, p.device_eta_factor, p.eta_mode, p.max_iter)
    ks = lt.mp_grid(2, 2)
    f = 16.0 * np.arange(1, 33) / 32
    E = np.tile(f ** 2, len(ks))
    kidx = np.repeat(np.arange(len(ks), dtype=np.int32), len(f))
    # three n = 1 superlattice films (same pristine Si leads) and one n = 2
    specs = [dict(n=1, period=2, L=9, seed=1), dict(n=1, period=3, L=14, seed=2), dict(n=2, period=2, L=6, seed=3),
             dict(n=1, period=1, L=5, seed=4)]
    devices, blocks = [], []
    for sp in specs:
        blk = [lt.si_ge_superlattice_film(sp["n"], sp["period"], sp["L"], kf, seed=sp["seed"]) for kf in ks]
        blocks.append(blk)
        devices.append(dict(blocks=engine.upload_blocks(blk), E=E, kidx=kidx))
    print("multi-device, shared leads", flush=True)
    outs = engine.solve_tdb_multi(devices, p)
    for i, (d, o) in enumerate(zip(devices, outs)):
        r = engine.solve_tdb(d["blocks"], E, p, kidx=kidx)
        assert (o["status"].cpu().numpy() == 0).all()
        for key in ("T_LR", "T_RL"):
            a, b = o[key].cpu().numpy(), r[key].cpu().numpy()
            assert np.abs(a - b).max() <= 1e-12 * max(1.0, np.abs(b).max()), (i, key)
        for j in (3, 40, 101):
            tl, tr, _ = O.solve_tdb(blocks[i][kidx[j]].as_dict(), E[j], op)
            assert abs(o["T_LR"][j].item() - tl) < 1e-9 * max(1, tl)
            assert abs(o["T_RL"][j].item() - tr) < 1e-9 * max(1, tr)


def test_shared_leads_on_planes(engine):
    """Devices with the same leads on planes: one decimation for those whose lead
    cells have the same planes, a further one where the coupling to the device
    reaches deeper into the cell; bit for bit the single solves, in chunks of
    different sizes too."""
    import dataclasses

    from phinfortran_amd import _native as N
    from phinfortran_amd import transport as T
    from test_gpu_planes import plane_blocks
    p = T.params("phonon", eta=1e-3, eta0=1e-4, convergence=1e-13)
    base = plane_blocks((12, 12, 12), (12, 11), 3, 4)
    deep = base.Hamld.copy()
    inside = np.flatnonzero(np.any(base.Hamlv != 0, 0))                # the plane that faces the lead
    middle = np.flatnonzero(np.any(base.Haml[inside] != 0, 0) & ~np.any(base.Hamlv != 0, 0))
    deep[middle[0], np.flatnonzero(np.any(deep != 0, 0))[0]] = 0.3
    sets = [base, dataclasses.replace(base, Hamd=1.1 * base.Hamd), dataclasses.replace(base, Hamld=deep),
            dataclasses.replace(base, Hamdv=0.9 * base.Hamdv)]
    E = np.linspace(0.05, 0.9, 33)
    for limit in (512, 10):
        eng = T.Engine(0, batch_limit=limit)
        try:
            devices = [dict(blocks=eng.upload_blocks(b), E=E) for b in sets]
            chunks = -(-E.size // limit)
            print(f"shared leads on planes, {limit} points a chunk", flush=True)
            for workers in (1, 4):
                eng.set_multi_workers(workers)
                eng.profile_reset()
                eng.profile(True)
                outs = eng.solve_tdb_multi(devices, p)
                eng.profile(False)
                assert eng.profile_get(N.NT_K_PLANES)["launches"] == chunks * (2 + 4)
                for d, o in zip(devices, outs):
                    r = eng.solve_tdb(d["blocks"], E, p)
                    for k in ("T_LR", "T_RL", "status"):
                        assert np.array_equal(o[k].cpu().numpy(), r[k].cpu().numpy()), k
        finally:
            eng.close()
