"""Cases of the docking library's main path, measured through its public calls.

Each case is one call (or one request stream) as a docking program makes it:
re-scoring poses (`DeviceJob.eval`, `gd_energy_eval_noalloc`), docking one
complex (`DeviceJob.dock`, `DeviceJob.dock_stream`), docking many complexes in
shared launches (`gd_batch_dock`) and serving requests (`gd_server_*`).  Inputs
are synthetic complexes (`synth_complex`, `synth_screen`) of the sizes that the
benchmark, the tests and the shipped fixture have.

Case fields: kind; P protein points, L ligand atoms; nl / np / nt ligand
conformers, protein conformers and temperatures (replicas = nl * np * nt);
n poses (evaluations); jobs complexes; steps MC steps; dump steps per dump;
spe steps per exchange point (0: none); axes the exchange axes (comma list);
move the move mode.
"""
import ctypes
import math

import numpy as np
import torch

import geauxdock_amd as g
from geauxdock_amd import abi
from geauxdock_amd.host import ReplicaOut

ALL_AXES = "temp,lig,prt"
_ENE = []


def _ene():
    if not _ENE:
        _ENE.append(g.load_enepara())
    return _ENE[0]


def listed():
    return [
        # a user re-scores one pose of a fixture-sized complex (344 points, 34 atoms,
        # 51 ligand and 11 protein conformers): the smallest call, latency alone
        dict(name="eval one pose", kind="eval", P=344, L=34, nl=51, np=11, nt=1, n=1),
        # re-scoring a pose list of a small complex (the CPU reference configuration's
        # shape), more poses than the job has replicas
        dict(name="eval small complex", kind="eval", P=1200, L=24, nl=5, np=5, nt=1, n=500),
        # re-scoring one pose per replica of the benchmark complex
        dict(name="eval benchmark complex", kind="eval", P=3000, L=40, nl=20, np=11, nt=8, n=1760),
        # the allocation-free evaluation of a ragged complex (odd points, atoms and poses)
        dict(name="eval without allocation", kind="eval_noalloc", P=1617, L=45, nl=5, np=11, nt=4, n=333),
        # the largest complex of the heterogeneous workloads
        dict(name="eval large complex", kind="eval", P=9000, L=80, nl=5, np=11, nt=4, n=880),
        # one small complex docked alone: 25 replicas, bound by the latency of a step
        dict(name="dock small", kind="dock", P=1200, L=24, nl=5, np=5, nt=1, steps=200, dump=200, spe=0,
             axes="temp", move="gaussian"),
        # one complex of the heterogeneous workload's ensemble (220 replicas, ragged sizes),
        # exchange on every axis
        dict(name="dock medium", kind="dock", P=4001, L=46, nl=5, np=11, nt=4, steps=100, dump=100, spe=50,
             axes=ALL_AXES, move="gaussian"),
        # the benchmark job: 1,760 replicas, exchange on every axis each 100 steps
        dict(name="dock benchmark complex", kind="dock", P=3000, L=40, nl=20, np=11, nt=8, steps=100, dump=100,
             spe=100, axes=ALL_AXES, move="gaussian"),
        # docking with every dump's accept records taken to the host, the reference's
        # uniform moves
        dict(name="dock with records", kind="stream", P=3000, L=40, nl=10, np=11, nt=4, steps=100, dump=50,
             spe=50, axes="temp", move="reference"),
        # many small complexes in shared launches
        dict(name="batch of small complexes", kind="batch", P=1200, L=24, nl=5, np=5, nt=1, jobs=64, steps=100,
             spe=0, axes="temp", move="gaussian"),
        # a virtual screen: one protein target, ligands of 12 to 80 atoms
        dict(name="screen", kind="screen", P=4000, L=80, nl=10, np=11, nt=4, jobs=8, steps=40, spe=20,
             axes=ALL_AXES, move="gaussian"),
        # the serving loop on requests of mixed sizes and lengths
        dict(name="serve", kind="serve", P=6000, L=64, nl=8, np=11, nt=4, jobs=8, steps=60, spe=20,
             axes=ALL_AXES, move="gaussian"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["eval", "eval", "eval_noalloc", "dock", "dock", "stream", "batch", "screen", "serve"])
    c = dict(kind=kind, L=rng.randint(12, 80), P=_log_int(rng, 1000, 9000))
    ens = rng.choice([(5, 5, 1), (5, 11, 4), (10, 11, 4), (7, 3, 5), (20, 11, 8), (3, 2, 6)])
    c.update(nl=ens[0], np=ens[1], nt=ens[2])
    if kind == "eval":
        c.update(n=_log_int(rng, 1, 1760))
    elif kind == "eval_noalloc":
        # its static workspace holds one 64-pose block of the complexes below
        c.update(P=_log_int(rng, 1000, 4000), L=rng.randint(12, 48), n=_log_int(rng, 1, 600))
    elif kind in ("dock", "stream"):
        # at most about the work of the benchmark complex's 100 steps
        most = 100.0 * 1760 * 40 * 3000
        steps = int(max(10, min(rng.randint(20, 200), most / (ens[0] * ens[1] * ens[2] * c["L"] * c["P"]))))
        if ens[0] * ens[1] * ens[2] * c["L"] * c["P"] * steps > most:
            c.update(nl=5, np=11, nt=4)
        spe = rng.choice([0, max(2, steps // 2), 10])
        c.update(steps=steps, dump=steps if kind == "dock" else max(1, steps // rng.randint(1, 3)), spe=spe,
                 axes=rng.choice(["temp", ALL_AXES, "lig,prt"]), move=rng.choice(["gaussian", "reference"]))
    else:
        e = rng.choice([(5, 5, 1), (5, 11, 2), (5, 11, 4)])
        c.update(nl=e[0], np=e[1], nt=e[2], P=_log_int(rng, 1000, 4000), jobs=rng.randint(3, 8),
                 steps=rng.randint(20, 40), spe=rng.choice([0, 10, 20]), axes=rng.choice(["temp", ALL_AXES]),
                 move="gaussian")
    return c


# ---- inputs ------------------------------------------------------------------


def _temps(c):
    # the workloads' ladders: one temperature 0.044, several from 0.004 to 0.04
    return (0.044, 0.044) if c["nt"] == 1 else (0.004, 0.04)


def _hosts(c, seed):
    """The complexes of a case on the host."""
    lo, hi = _temps(c)
    s = int(seed) % (1 << 30) + 1
    rng = np.random.default_rng(s)
    kw = dict(floor_temp=lo, ceiling_temp=hi, ene=_ene())
    if c["kind"] == "screen":  # one target, ligands of 12 atoms to L
        return [g.synth_screen(c["P"], s, int(rng.integers(12, c["L"] + 1)), s + 1 + i, c["nl"], c["np"], c["nt"],
                               **kw) for i in range(c["jobs"])]
    if c["kind"] == "serve":  # points from 1,500 to P, atoms from 12 to L, 5 to nl ligand conformers
        return [g.synth_complex(int(math.exp(rng.uniform(math.log(min(1500, c["P"])), math.log(c["P"])))),
                                int(rng.integers(12, c["L"] + 1)), 5 + i % max(1, c["nl"] - 4),
                                c["np"], c["nt"], seed=s + i, **kw) for i in range(c["jobs"])]
    return [g.synth_complex(c["P"], c["L"], c["nl"], c["np"], c["nt"], seed=s + i, **kw)
            for i in range(c.get("jobs", 1))]


def _poses(c, host, seed):
    """Poses around the pocket: the benchmark's displacements, any rotation for a third of them."""
    rng = np.random.default_rng(int(seed) + 77)
    d, n = host.desc, c["n"]
    conf = np.stack([rng.integers(0, d.n_lig, n), rng.integers(0, d.n_prt, n)], 1).astype(np.int32)
    rot = np.where(rng.random((n, 1)) < 1 / 3, rng.uniform(-np.pi, np.pi, (n, 3)), rng.normal(0, 0.1, (n, 3)))
    pose = np.concatenate([rng.normal(0, 1.0, (n, 3)), rot], 1).astype(np.float32)
    return np.ascontiguousarray(conf), np.ascontiguousarray(pose)


def _mc(c, seed, k=0, steps=None):
    return g.make_mc(steps or c["steps"], steps_per_dump=c.get("dump"), steps_per_exchange=c["spe"],
                     move_mode="gaussian" if c["move"] == "gaussian" else "reference", seed=int(seed) + 5, job_id=k,
                     axes=tuple(c["axes"].split(",")))


def prepare(case, seed):
    c = case
    g.check(g.lib().gd_init(0), "gd_init")
    hosts = _hosts(c, seed)
    st = dict(case=c, hosts=hosts)
    kind = c["kind"]
    if kind in ("eval", "eval_noalloc"):
        st["dev"] = g.DeviceJob(hosts[0])
        st["conf"], st["pose"] = _poses(c, hosts[0], seed)
    elif kind in ("dock", "stream"):
        st["dev"] = g.DeviceJob(hosts[0])
        st["mc"] = _mc(c, seed)
    elif kind in ("batch", "screen"):
        devs = [g.DeviceJob(h) for h in hosts]
        st["devs"] = devs
        st["handles"] = (ctypes.c_void_p * len(devs))(*[d.h for d in devs])
        st["mc"] = (abi.gd_mc_param * len(devs))(*[_mc(c, seed, k) for k in range(len(devs))])
    else:
        rng = np.random.default_rng(int(seed) + 3)
        st["mc"] = [_mc(c, seed, k, int(rng.integers(c["steps"] // 2, c["steps"] + 1))) for k in range(len(hosts))]
    return st


# ---- one pass ----------------------------------------------------------------


def _replicas(o):
    return dict(movematrix=o.movematrix, energy=o.energy, idx_tmp=o.idx_tmp, n_accept=o.n_accept,
                n_exchange=o.n_exchange, best=o.best_energy, is_accept=o.is_accept, swap_lig=o.n_swap_lig,
                swap_prt=o.n_swap_prt)


def _gather(outs):
    """The replicas of several jobs, one array per field."""
    d = [_replicas(o) for o in outs]
    return {k: np.concatenate([x[k] for x in d]) for k in d[0]}


def run(state):
    kind = state["case"]["kind"]
    if kind == "eval":
        terms, raw, _ = state["dev"].eval(state["conf"], state["pose"])
        return dict(terms=terms, raw=raw)
    if kind == "eval_noalloc":
        conf, pose = state["conf"], state["pose"]
        n = conf.shape[0]
        terms, raw = np.zeros((n, 10), np.float32), np.zeros((n, 9), np.float32)
        fp, ip = ctypes.POINTER(ctypes.c_float), ctypes.POINTER(ctypes.c_int)
        g.check(g.lib().gd_energy_eval_noalloc(state["dev"].h, n, conf.ctypes.data_as(ip), pose.ctypes.data_as(fp),
                                               terms.ctypes.data_as(fp), raw.ctypes.data_as(fp)),
                "gd_energy_eval_noalloc")
        return dict(terms=terms, raw=raw)
    if kind == "dock":
        out, _ = state["dev"].dock(state["mc"], stats=False)
        return _replicas(out)
    if kind == "stream":
        kept, counts = [], []

        def on_dump(dump, step_begin, rec, count):  # rows beyond a replica's count were not written
            rec[np.arange(rec.shape[1])[None, :] >= count[:, None]] = 0.0
            kept.append(rec)
            counts.append(count)

        out, _ = state["dev"].dock_stream(state["mc"], on_dump, stats=False)
        return dict(_replicas(out), records=np.concatenate([r.reshape(-1) for r in kept]), counts=np.concatenate(counts))
    if kind in ("batch", "screen"):
        outs = [ReplicaOut(d.n_rep) for d in state["devs"]]
        oc = (abi.gd_replica_out * len(outs))(*[o.c for o in outs])
        g.check(g.lib().gd_batch_dock(state["handles"], len(outs), state["mc"], oc, None), "gd_batch_dock")
        return _gather(outs)
    return _serve(state)


def _serve(state):
    """All requests queued at once, swept until each has its result."""
    lib, hosts, mcs = g.lib(), state["hosts"], state["mc"]
    cfg = abi.gd_server_config(hbm_budget=64 << 30, max_active=32, sweep_steps=50)
    s = ctypes.c_void_p()
    g.check(lib.gd_server_create(ctypes.byref(cfg), ctypes.byref(s)), "gd_server_create")
    try:
        outs = [ReplicaOut(h.n_rep) for h in hosts]
        status, tickets = {}, []
        for h, mc, o in zip(hosts, mcs, outs):
            t = ctypes.c_int64()
            g.check(lib.gd_server_submit(s, ctypes.byref(h.desc), ctypes.byref(mc), ctypes.byref(o.c),
                                         ctypes.byref(t)), "gd_server_submit")
            tickets.append(t.value)
        while len(status) < len(hosts):
            g.check(lib.gd_server_step(s, None, None), "gd_server_step")
            res, n = (abi.gd_job_result * 16)(), ctypes.c_int()
            g.check(lib.gd_server_results(s, res, 16, ctypes.byref(n)), "gd_server_results")
            for r in res[:n.value]:
                status[r.ticket] = r.status
    finally:
        lib.gd_server_destroy(s)
    return dict(_gather(outs), status=np.array([status[t] for t in tickets], np.int32))


# ---- what a pass cannot do without ---------------------------------------------


def _pass_counts(c, host):
    """(energy evaluations of the job, per-evaluation flops, table bytes)."""
    d = host.desc
    kt, lt = (np.ctypeslib.as_array(p, (n,)) for p, n in ((d.kde_t, d.kde_npoint), (d.lig_t, d.lig_natom)))
    bins = np.bincount(kt, minlength=abi.GD_NLT)
    mcs = np.ctypeslib.as_array(d.mcs_x, (d.mcs_nrow * d.lig_natom,))
    # 62 flops per (atom, point) pair, 11 per matched KDE anchor, 9 per valid MCS entry
    flops = (62.0 * d.lig_natom * d.prt_npoint + 11.0 * float(bins[lt].sum())
             + 9.0 * float((mcs != np.float32(abi.GD_MCS_INVALID)).sum()))
    tables = 4.0 * (3 * d.n_lig * d.lig_natom + 3 * d.n_prt * d.prt_npoint + 6 * d.prt_npoint + 4 * d.kde_npoint
                    + 3 * d.mcs_nrow * d.lig_natom)
    return flops, tables


def work(case):
    c = case
    b = f = 0.0
    for k, h in enumerate(_hosts(c, 1)):
        flops, tables = _pass_counts(c, h)
        R = h.n_rep
        if c["kind"].startswith("eval"):
            evals, io = c["n"], c["n"] * 4.0 * (8 + 19)
        else:
            steps = c["steps"] if c["kind"] != "serve" else 0.75 * c["steps"]
            on = [a for a, n in (("lig", c["nl"]), ("prt", c["np"])) if a in c["axes"].split(",") and n > 1]
            swaps = (steps // c["spe"]) * len(on) if c["spe"] else 0
            evals, io = R * (steps + 1 + swaps), R * 4.0 * 23
            if c["kind"] == "stream":
                io += R * steps * 17 * 4.0 * 0.3
        f += evals * flops
        b += tables + io
    return {"bytes": b, "flops": f}


# ---- the same values in 64 bits --------------------------------------------------


def exact(case, seed):
    """Energies of an evaluation in FP64 from the job's inputs (the reference's
    energy_prt_v1 / energy_kde_v1 / energy_mcs_v1 formulas, written out in torch);
    None for the docking kinds, whose chains branch on every rounding."""
    c = case
    if not c["kind"].startswith("eval"):
        return None
    host = _hosts(c, seed)[0]
    conf, pose = _poses(c, host, seed)
    a, e = host.arrays(), _ene()
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    t = lambda x: torch.as_tensor(np.array(x), device=dev).to(torch.float64)  # noqa: E731
    ti = lambda x: torch.as_tensor(np.array(x), device=dev).long()  # noqa: E731
    L, M = host.desc.lig_natom, host.desc.mcs_nrow
    lt, pt = ti(a["lig_t"]), ti(a["prt_t"])
    row = lambda x: t(x)[lt][:, pt]  # (L, P) of a [ligand type][point type] table  # noqa: E731
    p1a, p2a, pmf0, pmf1, hdb0, hdb1 = (row(getattr(e, k)) for k in ("p1a", "p2a", "pmf0", "pmf1", "hdb0", "hdb1"))
    hb = hdb0 > np.float32(0.1)
    cdc, cls2 = ti(a["prt_cdc"]) == 1, ti(a["prt_c"]) == 2
    res = ti(a["prt_seq3r"])
    okr = (res >= 0) & (res < a["psp"].shape[1])
    psp = torch.where((okr & cls2)[None, :], t(a["psp"])[lt][:, res.clamp(0, a["psp"].shape[1] - 1)], 0.0)
    q, ele, hpp = t(a["lig_c"]), t(a["prt_ele"]), t(a["prt_hpp"])
    hpl0, hpl1, hpl2 = (t(getattr(e, k))[lt] for k in ("hpl0", "hpl1", "hpl2"))
    kde_t = ti(a["kde_t"])
    kde = torch.stack([t(a["kde_x"]), t(a["kde_y"]), t(a["kde_z"])], 1)
    same = (lt[:, None] == kde_t[None, :]).double()
    n_bin = same.sum(1)
    mcs = torch.stack([t(a["mcs_x"]), t(a["mcs_y"]), t(a["mcs_z"])], 2)
    valid = torch.as_tensor(np.array(a["mcs_x"]) != np.float32(abi.GD_MCS_INVALID), device=dev).double()
    tcc = t(a["mcs_tcc"])
    prt = torch.stack([t(a["prt_x"]), t(a["prt_y"]), t(a["prt_z"])], 2)
    lig = torch.stack([t(a["lig_x"]), t(a["lig_y"]), t(a["lig_z"])], 2)
    center, pocket = t(a["lig_center"]), t(a["pocket_center"])
    ap, bp, w = t(e.a_para), t(e.b_para), t(e.w)
    n = conf.shape[0]
    raw, terms = torch.zeros(n, 9, dtype=torch.float64), torch.zeros(n, 10, dtype=torch.float64)
    at_once = max(1, int((2e7 if dev == "cuda" else 2e6) // (L * host.desc.prt_npoint)))
    for lo in range(0, n, at_once):
        m = t(pose[lo:lo + at_once])
        li, pi = ti(conf[lo:lo + at_once, 0]), ti(conf[lo:lo + at_once, 1])
        s, k = torch.sin(m[:, 3:]), torch.cos(m[:, 3:])
        (s1, s2, s3), (c1, c2, c3) = s.T, k.T
        R = torch.stack([c1 * c2, c1 * s2 * s3 - c3 * s1, s1 * s3 + c1 * c3 * s2,
                         c2 * s1, c1 * c3 + s1 * s2 * s3, c3 * s1 * s2 - c1 * s3,
                         -s2, c2 * s3, c2 * c3], 1).view(-1, 3, 3)
        # the rotation of each atom, coordinate by coordinate (no batched product)
        x = (R[:, None, :, :] * lig[li][:, :, None, :]).sum(3) + (m[:, :3] + center)[:, None, :]
        d = x[:, :, None, :] - prt[pi][:, None, :, :]
        r2 = (d * d).sum(3)
        del d
        r = r2.sqrt()
        e_raw = torch.zeros(m.shape[0], 9, dtype=torch.float64, device=dev)
        r3 = r2 * r
        p1, p2 = p1a / (r3 * r3 * r3), p2a / (r3 * r3)
        e_raw[:, 0] = ((p1 - p2) / (p1 * e.lj0 * (1.0 + e.lj1 * r2) + 1.0)).sum((1, 2))
        del p1, p2, r3
        u = e.el1 * r
        gq = torch.where(u < 1.0, e.el0 + e.a1 * u * u + e.b1 * u * u * u, 1.0 / u)
        e_raw[:, 1] = (gq * q[:, None] * ele[None, :]).sum((1, 2))
        dm = r - pmf0
        e_raw[:, 2] = (pmf1 / (1.0 + torch.exp((6.0 - 0.5 * r) * dm))).sum((1, 2))
        e_raw[:, 3] = torch.where(dm <= 0.0, psp, 0.0).sum((1, 2))
        h = (r - hdb0) * hdb1
        e_raw[:, 4] = torch.where(hb, hdb1 * torch.exp(-0.5 * h * h), 0.0).sum((1, 2)) * (-1.0 / math.sqrt(2.0 * math.pi))
        y = r2 / 81.0
        hp = torch.where((r2 <= 81.0) & cdc, hpp * (1.0 - y * (3.5 - y * (4.5 - y * (2.5 - 0.5 * y)))), 0.0).sum(2)
        e_raw[:, 5] = (0.5 * ((hp - hpl0) / hpl1) ** 2 - hpl2).sum(1)
        del u, gq, dm, h, y, r, r2
        dk = ((x[:, :, None, :] - kde[None, None]) ** 2).sum(3)
        ks = (torch.exp(e.kde2 * dk) * same).sum(2)
        e_raw[:, 6] = torch.where(n_bin > 0, ks / n_bin.clamp(min=1.0), 0.0).sum(1) / e.kde3
        dmcs = (((x[:, None] - mcs[None]) ** 2).sum(3) * valid).sum(2)
        e_raw[:, 7] = torch.log((tcc * torch.sqrt(dmcs / valid.sum(1))).sum(1) / M)
        e_raw[:, 8] = (center + m[:, :3] - pocket).square().sum(1).sqrt()
        norm = e_raw.clone()
        norm[:, :7] /= L
        norm = ap[:9] * norm + bp[:9]
        raw[lo:lo + at_once] = e_raw.cpu()
        terms[lo:lo + at_once, :9] = norm.cpu()
        terms[lo:lo + at_once, 9] = (norm * w[:9]).sum(1).cpu()
    return dict(terms=terms, raw=raw)
