"""The calls whose speed is measured: what a program that uses this engine has
it do, through the public entry points, from one point to thousands.

A case is a dict: "kind" names the call and the sort of system, the other
entries its sizes.  Systems come from phinfortran_amd.lattice (the builders of
the workloads), block sizes and lengths from the workloads, tests and example.

  point          surface_green_tdb + get_G_full_tdb of one (omega, k) on host
                 arrays, the sequence the reference's driver calls per point
  superlattice   batched solve of Si/Ge superlattice films over a k-grid
  film           batched solve of the Si|Ge interface film, one k-point
  mixed          the same film in the mixed-precision mode
  wire           batched solve of the alloyed Si/Ge wire (no transverse k)
  ribbon         batched tight-binding solve of the graphene ribbon
  longrange      a film whose force constants reach over the whole layer (no
                 zero blocks), many k-points, short device: the shape of the
                 first-principles example (b = 48, L = 2, 49 k x 61 omega)
  uneven         films of different block sizes and lengths in one call
  gradient       T and its gradient with respect to the interface layers
  modes          solve plus mode-resolved transmission of the wire
  probes         solve with a Buttiker probe in every layer
"""
import math
import random

import numpy as np
import torch

from phinfortran_amd import lattice as lt
from phinfortran_amd import transport as T

FMAX = 16.0          # THz, top of the phonon frequency grids


def listed():
    return [
        # one point through the per-point entries: every launch and copy counts
        dict(name="point_b48", kind="point", nx=2, ny=1, L=4),
        # a small film on a 2 x 2 k-grid, 16 frequencies each
        dict(name="superlattice_b24", kind="superlattice", n=1, period=2, L=10, nk=4, nw=16),
        # a middle-sized film, odd length and odd number of frequencies
        dict(name="superlattice_b216", kind="superlattice", n=3, period=5, L=31, nk=4, nw=37),
        # the wire of the small phonon workload, 512 frequencies
        dict(name="wire_b96", kind="wire", nx=2, ny=2, L=20, nw=512),
        # the ribbon of the electron workload, 2048 energies
        dict(name="ribbon_b80", kind="ribbon", dimers=40, L=60, nw=2048),
        # the first-principles example's shape, every block dense
        dict(name="longrange_b48", kind="longrange", nx=2, ny=1, L=2, nk=49, nw=61),
        # the headline: one k-point of the interface film, 1024 frequencies
        dict(name="film_b192", kind="film", nx=4, ny=2, L=40, nw=1024),
        # the same film in the mixed-precision mode, a quarter of the grid
        dict(name="film_b192_mixed", kind="mixed", nx=4, ny=2, L=40, nw=256),
        # gradient with respect to the 16 layers around the interface
        dict(name="film_b192_gradient", kind="gradient", nx=4, ny=2, L=40, window=16, nw=512),
        # 8 devices of the uneven-batching draw, two of each block size
        dict(name="uneven_8", kind="uneven", devices=8, nmax=4, nk=1, nw=64),
        # mode-resolved transmission of the wire
        dict(name="modes_b96", kind="modes", nx=2, ny=2, L=20, nw=128),
        # probes in a shorter film: every block of the full G
        dict(name="probes_b96", kind="probes", nx=2, ny=2, L=20, nw=64),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["point", "superlattice", "superlattice", "wire", "ribbon", "longrange", "film", "film",
                       "mixed", "gradient", "uneven", "modes", "probes"])
    if kind == "point":
        return dict(kind=kind, nx=rng.choice([1, 2]), ny=rng.choice([1, 2]), L=rng.randint(2, 9))
    if kind == "superlattice":
        n = rng.choice([1, 2, 3, 4])
        return dict(kind=kind, n=n, period=rng.randint(2, 8), L=_log(rng, 10, 80 if n < 4 else 40),
                    nk=rng.choice([1, 4, 9] if n < 3 else [1, 4] if n < 4 else [1]),
                    nw=_log(rng, 16, {1: 512, 2: 128, 3: 32, 4: 64}[n]))
    if kind == "wire":
        nx, ny = rng.choice([(1, 1), (2, 1), (2, 2), (3, 2)])
        return dict(kind=kind, nx=nx, ny=ny, L=_log(rng, 5, 40), nw=_log(rng, 33, 512))
    if kind == "ribbon":
        return dict(kind=kind, dimers=rng.randint(5, 48), L=_log(rng, 10, 60), nw=_log(rng, 65, 2048))
    if kind == "longrange":
        nx, ny = rng.choice([(1, 1), (2, 1), (2, 2)])
        return dict(kind=kind, nx=nx, ny=ny, L=rng.randint(1, 6), nk=rng.choice([4, 9, 16]), nw=_log(rng, 16, 61))
    if kind in ("film", "mixed", "gradient"):
        nx, ny = rng.choice([(1, 1), (2, 1), (3, 1), (2, 2), (4, 2)])
        c = dict(kind=kind, nx=nx, ny=ny, L=_log(rng, 8, 40), nw=_log(rng, 32, 1024 if kind == "film" else 256))
        if kind == "gradient":
            c["window"] = rng.randint(1, c["L"] // 2)
        return c
    if kind == "uneven":
        nmax = rng.randint(2, 4)
        return dict(kind=kind, devices=rng.randint(3, 8), nmax=nmax, nk=rng.choice([1, 4]) if nmax < 4 else 1,
                    nw=_log(rng, 16, 64))
    if kind == "modes":
        nx, ny = rng.choice([(1, 1), (2, 1), (2, 2)])
        return dict(kind=kind, nx=nx, ny=ny, L=_log(rng, 5, 20), nw=_log(rng, 32, 128))
    nx, ny = rng.choice([(1, 1), (2, 1), (2, 2)])
    return dict(kind=kind, nx=nx, ny=ny, L=_log(rng, 5, 20), nw=_log(rng, 32, 64))


# ------------------------------------------------------------------ systems

def _omega(rng, n):
    """n frequencies over (0, FMAX], the grid shifted by a seeded part of its step"""
    return FMAX * (np.arange(n) + rng.uniform(0.25, 1.0)) / n


def _kpoints(rng, nk):
    """a shifted sqrt(nk) x sqrt(nk) transverse grid"""
    m = int(math.isqrt(nk))
    s = rng.uniform(0.0, 1.0 / m, 2)
    return [(i / m + s[0] - 0.5, j / m + s[1] - 0.5) for i in range(m) for j in range(m)]


def _film(c, rng):
    kf = tuple(rng.uniform(-0.5, 0.5, 2))
    layer = lt.DiamondLayer(c["nx"], c["ny"], periodic=True)
    springs = rng.uniform(0.95, 1.05, (2, layer.nbond))
    return lt.si_ge_interface_film(nx=c["nx"], ny=c["ny"], L=c["L"], kfrac=kf, iface_springs=springs)


def _long_range(c, rng):
    """The film at nk k-points plus couplings between all pairs of atoms of a
    layer and of neighbouring layers, a few per cent of the nearest-neighbour
    ones, Hermitian in the layers; leads and device take the same ones."""
    ks = _kpoints(rng, c["nk"])
    out = []
    for kf in ks:
        b = lt.si_ge_interface_film(
            nx=c["nx"], ny=c["ny"], L=c["L"], kfrac=kf)
        n = b.b
        x = rng.standard_normal((2, n, n)) + 1j * rng.standard_normal((2, n, n))
        s = 0.02 * np.abs(b.Haml).max() / math.sqrt(n)
        h, v = s * 0.5 * (x[0] + x[0].conj().T), 0.5 * s * x[1]
        b.Haml += h
        b.Hamr += h
        b.Hamd += h
        b.Hamlv += v
        b.Hamrv += v.conj().T
        b.Hamdv += v
        b.Hamld += v
        b.Hamrd += v.conj().T
        out.append(b)
    return out


def _devices(c, seed):
    """the first devices of the seeded uneven draw, block sizes in turn"""
    specs = lt.superlattice_set(256, seed=seed, sizes=tuple(range(1, c["nmax"] + 1)), lengths=(10, 40))
    by = {n: [s for s in specs if s["n"] == n] for n in range(1, c["nmax"] + 1)}
    return [by[1 + i % c["nmax"]][i // c["nmax"]] for i in range(c["devices"])]


def _inputs(c, seed):
    """(block sets, energies, k index of each point) of a batched case"""
    rng = np.random.default_rng(seed)
    kind = c["kind"]
    if kind in ("film", "mixed", "gradient"):
        return [_film(c, rng)], _omega(rng, c["nw"]) ** 2, None
    if kind in ("wire", "modes"):
        return [lt.si_ge_wire(nx=c["nx"], ny=c["ny"], L=c["L"], seed=seed)], _omega(rng, c["nw"]) ** 2, None
    if kind == "ribbon":
        E = -3.0 + 6.0 * (np.arange(c["nw"]) + rng.uniform(0.0, 1.0)) / c["nw"]
        return [lt.agnr_blocks(n_dimer=c["dimers"], L=c["L"], seed=seed)], E, None
    if kind == "longrange":
        blocks = _long_range(c, rng)
    elif kind == "superlattice":
        ks = _kpoints(rng, c["nk"])
        blocks = [lt.si_ge_superlattice_film(c["n"], c["period"], c["L"], kf, seed=seed) for kf in ks]
    elif kind == "probes":
        return [lt.si_ge_superlattice_film(2, 3, c["L"], tuple(rng.uniform(-0.5, 0.5, 2)), seed=seed)
                if (c["nx"], c["ny"]) == (2, 2) else _film(c, rng)], _omega(rng, c["nw"]) ** 2, None
    E = np.tile(_omega(rng, c["nw"]) ** 2, len(blocks))
    return blocks, E, np.repeat(np.arange(len(blocks), dtype=np.int32), c["nw"])


def _params(kind):
    if kind == "ribbon":
        return T.params("tb", eta=1e-8)
    if kind in ("wire", "modes"):
        return T.params("phonon", eta=1e-6, eta0=1e-6 * FMAX)
    return T.params("phonon", precision="mixed" if kind == "mixed" else "fp64")


def prepare(case, seed):
    kind = case["kind"]
    st = dict(kind=kind, p=_params(kind), eng=T.Engine(0, batch_limit=2048))
    if kind == "point":
        rng = np.random.default_rng(seed)
        st["blk"], st["E"] = _film(case, rng), float(rng.uniform(1.0, 14.0) ** 2)
        return st
    if kind == "uneven":
        rng = np.random.default_rng(seed)
        ks = _kpoints(rng, case["nk"])
        om = _omega(rng, case["nw"])
        st["devs"] = []
        for s in _devices(case, seed % 1000):
            blocks = [lt.si_ge_superlattice_film(s["n"], s["period"], s["L"], kf, seed=s["seed"]) for kf in ks]
            st["devs"].append(dict(
                blocks=st["eng"].upload_blocks(blocks),
                E=torch.as_tensor(np.tile(om ** 2, len(ks)), dtype=torch.float64, device="cuda"),
                kidx=torch.as_tensor(np.repeat(np.arange(len(ks), dtype=np.int32), case["nw"]), device="cuda")))
        return st
    blocks, E, kidx = _inputs(case, seed)
    st["d"] = st["eng"].upload_blocks(blocks)
    st["E"] = torch.as_tensor(E, dtype=torch.float64, device="cuda")
    st["kidx"] = None if kidx is None else torch.as_tensor(kidx, device="cuda")
    if kind == "gradient":
        # the weights of the thermal conductance at 300 K
        from phinfortran_amd.adjoint import conductance_weights
        w = conductance_weights(np.sqrt(E), 300.0, (case["nx"] * case["ny"]) * (lt.A_SI * 1e-10) ** 2)
        w = np.asarray(w)
        st["w"] = torch.as_tensor(w / np.abs(w).max(), dtype=torch.float64, device="cuda")
        st["lo"] = case["L"] // 2 - case["window"] // 2
        st["hi"] = min(st["lo"] + case["window"], case["L"] - 1)
    if kind == "probes":
        st["temp"] = torch.as_tensor(np.linspace(310.0, 290.0, case["L"]), dtype=torch.float64, device="cuda")
    return st


def run(state):
    eng, p, kind = state["eng"], state["p"], state["kind"]
    if kind == "point":
        b, E = state["blk"], state["E"]
        s = eng.surface_green_tdb(b.Haml, b.Hamr, b.Hamlv, b.Hamrv, E, p, want_plus_minus=False)
        r = eng.get_G_full_tdb(s["gl_adv"].conj().T, s["gr_ret"], -s["gml_adv"], s["gmr_ret"], s["sl_adv"].conj().T,
                               s["sr_ret"], E, b.Hamd, b.Hamdv, b.Hamld, b.Hamrd, b.Haml, b.Hamr, p)
        return {"T_LR": r["transl"], "T_RL": r["transr"], "sl_adv": s["sl_adv"], "sr_ret": s["sr_ret"]}
    if kind == "uneven":
        outs = eng.solve_tdb_multi(state["devs"], p, stream_sync=False)
        return [{k: o[k] for k in ("T_LR", "T_RL", "status")} for o in outs]
    if kind == "gradient":
        r = eng.solve_tdb_adjoint(state["d"], state["E"], p, state["w"], state["lo"], state["hi"], stream_sync=False)
        return {k: r[k] for k in ("T_LR", "T_RL", "status", "dHamd", "dHamdv")}
    if kind == "modes":
        # the totals over the modes: the modes of a degenerate set (the wire's
        # cross-section is symmetric) have no order or basis of their own
        r = eng.solve_modes(state["d"], state["E"], p, lt.A_SI, lt.A_SI)
        return {k: r[k] for k in ("T_LR", "T_RL", "status", "sums", "n_prop")}
    if kind == "probes":
        r = eng.solve_buttiker(state["d"], state["E"], p, state["temp"], 320.0, 280.0, stream_sync=False)
        return {k: r[k] for k in ("T_LR", "T_RL", "status", "flux", "jacobian", "flux_left", "flux_right", "a_sum",
                                  "gn_sum")}
    r = eng.solve_tdb(state["d"], state["E"], p, kidx=state["kidx"], stream_sync=False)
    return {k: r[k] for k in ("T_LR", "T_RL", "status", "iters")}


# ------------------------------------------------------------ needed work

def _shape(c):
    """(b, size of the planes a layer's couplings divide it into, planes per layer)"""
    k = c["kind"]
    if k == "ribbon":
        return 2 * c["dimers"], c["dimers"] / 2, 4
    b = 24 * c["n"] ** 2 if k == "superlattice" else 24 * c["nx"] * c["ny"]
    return (b, b, 1) if k == "longrange" else (b, b / 4, 4)


def _solve_work(b, m, planes, L, npts, nk):
    """Block elimination over the smallest coupled blocks: per point two
    systems of L + 2 layers, five products of m^3 per plane (inverse, two for
    the self-energy, two for the end column), and 2 x 13 decimation steps of
    an inverse and six products (the periodic cell reduced to its two coupled
    planes: 16 m^3, or 7 b^3 with one plane)."""
    dec = 2 * 13 * (16 if planes > 1 else 7) * m ** 3
    return {"bytes": 16.0 * nk * b * b * (2 * L + 6) + 40.0 * npts,
            "flops": 8.0 * npts * (2 * (L + 2) * planes * 5 * m ** 3 + dec)}


def work(case):
    c = case
    if c["kind"] == "uneven":
        out = {"bytes": 0.0, "flops": 0.0}
        for s in _devices(c, 1):
            w = _solve_work(s["b"], s["b"] / 4, 4, s["L"], c["nk"] * c["nw"], c["nk"])
            out = {k: out[k] + w[k] for k in out}
        return out
    b, m, planes = _shape(c)
    nk = c.get("nk", 1)
    npts = c.get("nw", 1) * nk
    w = _solve_work(b, m, planes, c["L"], npts, nk)
    if c["kind"] == "gradient":
        # T_LR only: one system, its column and row back to the window, and the
        # window's dense gradient blocks, three products b x b x m each layer
        lay = c["window"] + 1
        w["flops"] += 8.0 * npts * (4 * planes * c["L"] * m ** 3 + 3 * lay * b * b * m)
        w["bytes"] += 16.0 * b * b * 2 * lay
    if c["kind"] == "modes":
        # four lead eigenproblems of b: about 25 b^3 each, and the t and r chains
        w["flops"] += 8.0 * npts * 4 * (25 + 10) * b ** 3
    if c["kind"] == "probes":
        # every block of the full G enters the probe currents
        w["flops"] += 8.0 * npts * c["L"] * (c["L"] - 1) * b * b * m
        w["bytes"] += 8.0 * npts * c["L"] * (c["L"] + 3)
    return w


def tolerance(case):
    # Near band edges the decimation passes through nearly singular blocks
    # and T amplifies rounding by up to 1e10 at single points: there two
    # correct 64-bit evaluations differ by 1e-6 (at one point of the film,
    # LAPACK against a Newton-refined inverse 5e-8, 80-bit sums in two orders
    # 2e-11).  Seen against exact(): 3e-8 (longrange), 8e-8 (dHamdv).
    return {"rel": 4e-7 if case["kind"] == "gradient" else 1e-7, "max": 1e-5, "differ": 0.01}


# ----------------------------------------------------------- 64-bit values

def _inv(a):
    """Inverse of every matrix, one Newton step after the library's (whose
    residuals reach 1e-8 here; near band edges T amplifies them by 1e8 and
    more); a few matrices at a time, as its workspace grows with the batch."""
    m = max(8, int(1.2e6 / a.shape[-1] ** 2))
    eye = torch.eye(a.shape[-1], dtype=a.dtype, device=a.device)
    out = []
    for x in a.split(m):
        y = torch.linalg.inv(x)
        out.append(y + y @ (eye - x @ y))
    return torch.cat(out)


def _surface(H, V, z, conv, max_iter):
    """Lopez-Sancho surface function of H (n, n per point) coupled by V from
    the next lead cell to this one, and its self-energy V^+ g V."""
    eye = torch.eye(H.shape[-1], dtype=H.dtype, device=H.device)
    zI = z[:, None, None] * eye
    es, e1, al, be = H.clone(), H.clone(), V.mH.contiguous(), V.clone()
    for _ in range(max_iter):
        live = (al.abs().amax((1, 2)) > conv)
        if not bool(live.any()):
            break
        i = live.nonzero()[:, 0]
        a, bt = al[i], be[i]
        g = _inv(zI[i] - e1[i])
        t1, t2 = a @ g, bt @ g
        ab = t1 @ bt
        es[i] = es[i] + ab
        e1[i] = e1[i] + ab + t2 @ a
        al[i], be[i] = t1 @ a, t2 @ bt
    g = _inv(zI - es)
    return g, V.mH @ g @ V


def _exact_solve(blocks, E, kidx, p, dev, grad=None):
    """T_LR and T_RL of every point by the two block sweeps, in complex128;
    grad = (weights, lo, hi): also the gradient blocks of sum w T_LR."""
    E = torch.as_tensor(E, dtype=torch.float64, device=dev)
    k = torch.zeros(E.numel(), dtype=torch.long, device=dev) if kidx is None else \
        torch.as_tensor(kidx, device=dev).long()
    get = lambda n: torch.as_tensor(np.stack([getattr(b, n) for b in blocks]), device=dev)
    Hl, Vl, Hr, Vr, Hd, Hv, Hld, Hrd = (get(n) for n in ("Haml", "Hamlv", "Hamr", "Hamrv", "Hamd", "Hamdv", "Hamld",
                                                         "Hamrd"))
    L, n = Hd.shape[1], Hd.shape[2]
    chunk = max(1, int(4e9 / (16.0 * n * n * (12 + (2 * L if grad else 0)))))
    tl, tr = [], []
    gd = gv = None
    if grad:
        w, lo, hi = grad
        hc = min(hi, L - 2)
        gd = torch.zeros((len(blocks), hi - lo + 1, n, n), dtype=Hd.dtype, device=dev)
        gv = torch.zeros((len(blocks), hc - lo + 1, n, n), dtype=Hd.dtype, device=dev)
    for q in range(0, E.numel(), chunk):
        e, kk = E[q:q + chunk], k[q:q + chunk]
        eta = p.eta * e + p.eta0 if p.eta_mode == 0 else torch.full_like(e, p.eta)
        zl, zd = torch.complex(e, eta), torch.complex(e, eta * p.device_eta_factor)
        gl, sl = _surface(Hl[kk], Vl[kk], zl.conj(), p.convergence, p.max_iter)
        gl, sl = gl.mH, sl.mH
        gr, sr = _surface(Hr[kk], Vr[kk], zl, p.convergence, p.max_iter)
        gamL, gamR = 1j * (sl - sl.mH), 1j * (sr - sr.mH)
        sh = lambda H: zd[:, None, None] * torch.eye(H.shape[-1], dtype=H.dtype, device=dev) - H
        # left to right
        V, G, G0, kept = Hld[kk], gl, gl, []
        for i in range(L):
            G = _inv(sh(Hd[kk, i]) - V.mH @ G @ V)
            G0 = G0 @ V @ G
            if grad:
                kept.append((G, G0))
            V = Hv[kk, i] if i + 1 < L else Hrd[kk].mH
        Gc = _inv(sh(Hr[kk]) - sr - V.mH @ G @ V)
        G0c = G0 @ V @ Gc
        tl.append(((gamL @ G0c @ gamR) * G0c.conj()).sum((1, 2)).real)
        if grad:
            A = w[q:q + chunk, None, None] * (gamR @ G0c.mH @ gamL)
            C, R, cols, rows = Gc, G0c, {}, {}
            for j in range(L - 1, lo - 1, -1):
                g, g0 = kept[j]
                R, C = g0 + R @ V.mH @ g, g @ V @ C
                cols[j], rows[j] = C @ A, R
                V = Hv[kk, j - 1] if j else V
            for j in range(lo, hi + 1):
                gd[:, j - lo].index_add_(0, kk, 2 * (cols[j] @ rows[j]).mH)
            for j in range(lo, hc + 1):
                gv[:, j - lo].index_add_(0, kk, 2 * ((cols[j + 1] @ rows[j]).mH + cols[j] @ rows[j + 1]))
        # right to left
        V, G, G0 = Hrd[kk], gr, gr
        for i in range(L - 1, -1, -1):
            G = _inv(sh(Hd[kk, i]) - V.mH @ G @ V)
            G0 = G0 @ V @ G
            V = Hv[kk, i - 1].mH if i else Hld[kk].mH
        Gc = _inv(sh(Hl[kk]) - sl - V.mH @ G @ V)
        G0c = G0 @ V @ Gc
        tr.append(((gamR @ G0c @ gamL) * G0c.conj()).sum((1, 2)).real)
    clamp = lambda t: torch.where(t < 1e-60, torch.zeros_like(t), t)
    out = {"T_LR": clamp(torch.cat(tl)), "T_RL": clamp(torch.cat(tr))}
    if grad:
        out.update(dHamd=gd, dHamdv=gv)
    return out


def exact(case, seed):
    """T (and the gradient) in 64 bits by plain torch; the counts, the mode
    sums and the probe outputs have no value here."""
    kind = case["kind"]
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    if kind not in ("point", "uneven", "probes"):
        if case["nw"] * case.get("nk", 1) * (2 * case["L"] + 46) * _shape(case)[0] ** 3 > 6e11:
            return None          # over 20 seconds
    if kind == "point":
        rng = np.random.default_rng(seed)
        b, E = _film(case, rng), float(rng.uniform(1.0, 14.0) ** 2)
        r = _exact_solve([b], [E], None, _params(kind), dev)
        return {"T_LR": float(r["T_LR"][0]), "T_RL": float(r["T_RL"][0]), "sl_adv": None, "sr_ret": None}
    if kind == "probes":
        return None
    if kind == "uneven":
        rng = np.random.default_rng(seed)
        ks = _kpoints(rng, case["nk"])
        om = _omega(rng, case["nw"])
        out = []
        for s in _devices(case, seed % 1000):
            blocks = [lt.si_ge_superlattice_film(s["n"], s["period"], s["L"], kf, seed=s["seed"]) for kf in ks]
            r = _exact_solve(blocks, np.tile(om ** 2, len(ks)), np.repeat(np.arange(len(ks)), case["nw"]), _params(kind), dev)
            out.append({**r, "status": None})
        return out
    blocks, E, kidx = _inputs(case, seed)
    p = _params(kind)
    if kind == "gradient":
        st = prepare(case, seed)
        r = _exact_solve(blocks, E, kidx, p, dev, (st["w"].to(dev), st["lo"], st["hi"]))
        return {**r, "status": None}
    r = _exact_solve(blocks, E, kidx, p, dev)
    none = {"modes": ("status", "sums", "n_prop")}.get(kind, ("status", "iters"))
    return {**r, **{k: None for k in none}}
