"""What the framework's users have it do, as cases to be timed.

The work is molecular dynamics of one-bead-per-nucleotide RNA through
sis_amd's public entry points, over the range of the benchmark
configurations (sis_amd/configs.py), the tests and bench.py:

  md      Engine.step of one system: a single chain of tens to about a
          thousand nucleotides, or a periodic box of many chains up to 94,000
          beads; one pass is one segment of a run as a workflow's driver does
          it: the restart state in, whole job_md steps (list rebuilds, limit
          MC, noise, update), the state out
  remd    the same for a replica-exchange ladder (Engine mode "auto" takes the
          batched form), with exchanges inside the segment
  serve   a burst of independent jobs through JobPool until the last is done
  eval    forces and energies of one configuration on fresh lists
  dcd     job_dcd: the energies of the frames of a trajectory file

A case's fields: chains x length (to length2 when chains differ), conc (mM of
nucleotides, 0: no box), nrep and its ladder, ff ("sis": triplet base pairs
with the limit MC, or "nht22": base-pair model 1 without it), precision (0:
FP64, 1: FP32 pair arithmetic), mode, margin (list skin, A), tempK, salt (M),
integrator (1 GJF-2GJ Langevin, 2 Brownian), steps, exchange.
"""
import math
import os
import tempfile
import time

import numpy as np
import torch

from sis_amd import forcefield
from sis_amd.abi import MOLT_RNA, NNT_ORDER, SEQT
from sis_amd.configs import box_for_concentration
from sis_amd.engine import Engine, write_dcd_file
from sis_amd.serving import DONE, JobPool

BASE = dict(kind="md", chains=1, length=64, length2=0, seq="random", conc=0.0, nrep=1, ff="sis", precision=0,
            mode="phases", margin=5.0, tempK=310.0, salt=0.15, integrator=1, steps=256, exchange=0)


def _case(**over):
    return dict(BASE, **over)


def listed():
    return [
        # the smallest run: one 64-nt hairpin, the default form and precision (launch-bound)
        _case(name="md_hairpin64", seq="hairpin", length=64, margin=10.0, tempK=300.0, steps=512),
        # a single ragged mid-sized chain, FP32 pair arithmetic
        _case(name="md_chain397_f32", length=397, precision=1, steps=384),
        # the condensate of 200 CAG repeats, FP64
        _case(name="md_cag47x200", seq="cag", chains=200, length=47, conc=1.0, steps=384),
        # the large condensate, FP32 pair arithmetic
        _case(name="md_cag47x2000_f32", seq="cag", chains=2000, length=47, conc=2.0, precision=1, steps=384),
        # the temperature ladder of the headline benchmark
        _case(name="remd_256x128_f32", kind="remd", nrep=256, length=128, precision=1, mode="auto", tempK=290.0,
              steps=1000, exchange=1000),
        # a small ladder, FP64, short exchange period
        _case(name="remd_14x47", kind="remd", seq="cag", nrep=14, length=47, mode="auto", tempK=290.0, steps=500,
              exchange=100),
        # an odd ladder of a longer chain, FP64, exchanges that do not divide the segment
        _case(name="remd_99x211", kind="remd", nrep=99, length=211, mode="auto", tempK=290.0, steps=300, exchange=128),
        # a burst of mixed jobs, half FP64 and half FP32, as the serving benchmark draws them
        _case(name="serve_12", kind="serve", chains=64, length=20, length2=400, conc=5.0, steps=2000, nrep=12),
        # forces and energies of a 9,400-bead configuration, FP32 pair arithmetic, every formed pair counted
        _case(name="eval_cag47x200_f32", kind="eval", seq="cag", chains=200, length=47, conc=1.0, precision=1),
        # energies of a 100-frame trajectory of the 47-nt CAG repeat
        _case(name="dcd_cag47", kind="dcd", seq="cag", length=47, ff="nht22", tempK=295.15, steps=100),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    c = _case(precision=rng.randrange(2), margin=round(rng.uniform(3.0, 10.0), 2), tempK=round(rng.uniform(280.0, 360.0), 2),
              salt=round(rng.uniform(0.05, 0.5), 3), seq=rng.choice(["random", "cag"]))
    kind = rng.choice(["md", "box", "box", "remd", "remd", "serve", "eval", "dcd"])
    if kind == "md":
        c.update(length=_log(rng, 30, 1000), steps=rng.randrange(96, 400), integrator=rng.choice([1, 1, 1, 2]),
                 ff=rng.choice(["sis", "sis", "sis", "nht22"]))
    elif kind in ("box", "eval"):
        lo = rng.randrange(20, 60)
        hi = lo + rng.choice([0, 0, 1, 17, 60])
        beads = _log(rng, 600, 90000 if kind == "box" else 12000)
        c.update(kind="eval" if kind == "eval" else "md", length=lo, length2=hi if hi > lo else 0,
                 chains=max(2, beads // hi), conc=round(rng.uniform(0.5, 3.0), 2), steps=rng.randrange(64, 256))
    elif kind == "remd":
        n = _log(rng, 24, 420)
        c.update(kind="remd", length=n, nrep=min(256, _log(rng, 2, max(3, 32000 // n))), mode="auto", tempK=290.0,
                 steps=rng.randrange(100, 300), exchange=rng.randrange(40, 160), integrator=rng.choice([1, 1, 1, 2]))
    elif kind == "serve":
        c.update(kind="serve", chains=_log(rng, 1, 40), length=20, length2=rng.randrange(60, 400),
                 conc=round(rng.uniform(0.5, 5.0), 2), nrep=rng.randrange(3, 11), steps=rng.randrange(200, 1500))
    else:
        c.update(kind="dcd", length=rng.randrange(30, 150), steps=rng.randrange(20, 120), ff="nht22", precision=0)
    return c


# ---------------------------------------------------------------------
# inputs: seeded self-avoiding random coils, the start of every benchmark
# configuration, grown all chains at once
def _grow(rng, nch, n, clash=9.0, bond=5.9, tries=12):
    """(nch, n, 3) coils: fixed bonds, angles near 120 degrees, free
    dihedrals, beads of a chain at least `clash` apart beyond second
    neighbours.  Each bead takes the first of `tries` random directions that
    keeps clear; a chain that is caught is grown again."""
    dev = torch.device("cuda")
    x = torch.zeros((nch, n, 3), dtype=torch.float64, device=dev)
    left = np.arange(nch)
    for _ in range(200):
        m = len(left)
        th = torch.from_numpy(np.deg2rad(rng.normal(120.0, 5.0, (n, m, tries)))).to(dev)
        ph = torch.from_numpy(rng.uniform(-np.pi, np.pi, (n, m, tries))).to(dev)
        d = rng.normal(size=(m, 2, 3))
        u = d[:, 0] / np.linalg.norm(d[:, 0], axis=1, keepdims=True)
        w = d[:, 1] - (d[:, 1] * u).sum(1, keepdims=True) * u
        w /= np.linalg.norm(w, axis=1, keepdims=True)
        y = torch.zeros((m, n, 3), dtype=torch.float64, device=dev)
        y[:, 1] = bond * torch.from_numpy(u).to(dev)
        if n > 2:
            y[:, 2] = y[:, 1] + bond * torch.from_numpy(0.5 * u + math.sqrt(0.75) * w).to(dev)
        ok = torch.ones(m, dtype=torch.bool, device=dev)
        rows = torch.arange(m, device=dev)
        for i in range(3, n):
            b = y[:, i - 1] - y[:, i - 2]
            b = b / b.norm(dim=1, keepdim=True)
            k = torch.linalg.cross(y[:, i - 2] - y[:, i - 3], b)
            k = k / k.norm(dim=1, keepdim=True)
            f = torch.linalg.cross(k, b)
            t, p = th[i], ph[i]
            cand = y[:, None, i - 1] + bond * ((-torch.cos(t))[..., None] * b[:, None] + (torch.sin(t) * torch.cos(p))[..., None] * f[:, None]
                                               + (torch.sin(t) * torch.sin(p))[..., None] * k[:, None])
            far = (cand[:, :, None] - y[:, None, : i - 2]).square().sum(3).amin(2) >= clash * clash
            pick = far.to(torch.int8).argmax(1)
            ok &= far.any(1)
            y[:, i] = cand[rows, pick]
        done = ok.cpu().numpy()
        x[torch.from_numpy(left[done]).to(dev)] = y[ok]
        left = left[~done]
        if not len(left):
            return x.cpu().numpy()
    raise RuntimeError("chains could not be grown")


def _place(rng, x, lens, box, clash=10.0):
    """Whole chains moved to random places of the periodic box until no two
    beads of different chains are closer than `clash`."""
    dev = torch.device("cuda")
    nch, n, _ = x.shape
    real = np.arange(n)[None, :] < lens[:, None]
    mid = np.stack([x[c, : lens[c]].mean(0) for c in range(nch)])
    rad = np.array([np.linalg.norm(x[c, : lens[c]] - mid[c], axis=1).max() for c in range(nch)])
    x = x - mid[:, None]
    pos = rng.uniform(0.0, box, (nch, 3))
    new = np.ones(nch, bool)
    for _ in range(400):
        bad = np.zeros(nch, bool)
        a = np.nonzero(new)[0]
        d = pos[a][:, None] - pos[None]
        d -= box * np.round(d / box)
        near = np.sqrt((d ** 2).sum(2)) < rad[a][:, None] + rad[None] + clash
        i, j = np.nonzero(near)
        i = a[i]
        keep = (i < j) | (~new[j])
        keep &= i != j
        i, j = i[keep], j[keep]
        for s in range(0, len(i), 256):
            p, q = i[s: s + 256], j[s: s + 256]
            u = torch.from_numpy(x[p] + pos[p][:, None]).to(dev)
            v = torch.from_numpy(x[q] + pos[q][:, None]).to(dev)
            e = u[:, :, None] - v[:, None]
            e = e - box * torch.round(e / box)
            near2 = e.square().sum(3) < clash * clash
            near2 &= torch.from_numpy(real[p][:, :, None] & real[q][:, None]).to(dev)
            hit = near2.any(2).any(1).cpu().numpy()
            bad[np.maximum(p, q)[hit]] = True
        if not bad.any():
            return x + pos[:, None]
        pos[bad] = rng.uniform(0.0, box, (int(bad.sum()), 3))
        new = bad
    raise RuntimeError("chains could not be placed")


def _sequence(rng, how, n):
    if how == "cag":
        return ("CAG" * (n // 3 + 1))[:n]
    if how == "hairpin":    # A/U flanks, a stem of random pairs and an 8-nt loop
        stem = "".join(rng.choice(list("GCAU"), (n - 16) // 2, p=[0.3, 0.3, 0.2, 0.2]))
        back = "".join({"A": "U", "U": "A", "G": "C", "C": "G"}[c] for c in reversed(stem))
        loop = "".join(rng.choice(list("AUGC"), 8))
        rest = n - len(stem) * 2 - 8
        return "".join(rng.choice(list("AU"), rest // 2)) + stem + loop + back + "".join(rng.choice(list("AU"), rest - rest // 2))
    return "".join(rng.choice(list("AUGC"), n))


def _system(case, rng, lens, frames=1):
    """The dict that Engine and JobPool take, with `frames` coordinate sets
    of a single chain (replicas or trajectory frames)."""
    lens = np.asarray(lens, np.int32)
    if case["seq"] == "cag":
        seqs = [_sequence(rng, "cag", int(n)) for n in lens]
    elif case["length2"]:
        seqs = [_sequence(rng, case["seq"], int(n)) for n in lens]
    else:
        seqs = [_sequence(rng, case["seq"], int(lens[0]))] * len(lens)
    make = forcefield.nht22_params if case["ff"] == "nht22" else forcefield.default_params
    p = make(tempK=case["tempK"], ionic_strength=case["salt"], nl_margin=case["margin"], integrator=case["integrator"])
    nmp = int(lens.sum())
    if case["conc"] > 0:
        box = box_for_concentration(nmp, case["conc"])
        x = _place(rng, _grow(rng, len(lens), int(lens.max())), lens, box)
        xyz = np.concatenate([x[c, : lens[c]] for c in range(len(lens))])[None]
        p.update(pbc=1, box=[box] * 3)
    else:
        xyz = _grow(rng, frames, int(lens[0]))
    if case["kind"] in ("eval", "dcd"):
        p.update(nstep_bp_mc=0)
    temps = np.array([case["tempK"]]) if case["nrep"] == 1 or case["kind"] == "serve" else \
        case["tempK"] * (380.0 / case["tempK"]) ** (np.arange(case["nrep"]) / (case["nrep"] - 1))
    return dict(name=case["kind"], nchains=len(lens), nmp_chain=lens, moltype=np.full(len(lens), MOLT_RNA, np.int32),
                seq=np.array([SEQT[c] for s in seqs for c in s], np.int32), seqs=seqs, xyz=np.ascontiguousarray(xyz),
                params=p, nrep=len(temps), temps=temps, nstep=case["steps"])


def _sizes(case):
    """The stream that a case's sizes come from: its own, whatever the seed of its inputs."""
    return np.random.default_rng([case["chains"], case["length"], case["length2"], case["nrep"], case["steps"]])


def _inputs(case, seed):
    lens = np.full(case["chains"], case["length"])
    if case["length2"]:
        lens = _sizes(case).integers(case["length"], case["length2"] + 1, case["chains"])
    frames = {"remd": case["nrep"], "dcd": case["steps"]}.get(case["kind"], 1)
    return _system(case, np.random.default_rng(seed), lens, frames)


def _jobs(case, seed):
    """(system, steps, precision) of each job: 1 to `chains` chains of its
    own, its temperature, salt and box, steps log-uniform over two decades."""
    rng, size = np.random.default_rng(seed), _sizes(case)
    jobs = []
    for k in range(case["nrep"]):
        lens = size.integers(case["length"], case["length2"] + 1, int(size.integers(1, case["chains"] + 1)))
        one = dict(case, tempK=rng.uniform(280.0, 360.0), salt=rng.uniform(0.05, 0.5),
                   conc=size.uniform(min(0.5, case["conc"]), case["conc"]))
        steps = int(round(case["steps"] * 10.0 ** size.uniform(-2.0, 0.0)))
        jobs.append((_system(one, rng, lens), max(1, steps), k % 2))
    return jobs


# ---------------------------------------------------------------------
def prepare(case, seed):
    if case["kind"] == "serve":
        return dict(kind="serve", jobs=_jobs(case, seed), pool=JobPool(), seed=seed)
    s = _inputs(case, seed)
    if case["kind"] == "dcd":
        d = tempfile.TemporaryDirectory(prefix="dcd_")
        path = os.path.join(d.name, "traj.dcd")
        write_dcd_file(path, s["xyz"])
        s["xyz"] = s["xyz"][:1]
        return dict(kind="dcd", eng=Engine(s), path=path, dir=d, frames=case["steps"])
    eng = Engine(s, precision=case["precision"], mode=case["mode"], seed=seed + 1, exchange_every=case["exchange"])
    if case["kind"] == "eval":
        return dict(kind="eval", eng=eng, xyz=s["xyz"])
    eng.init_velocities()
    x, v, a = eng.get_state()
    return dict(kind="step", eng=eng, start=(x, v, a), labels=np.arange(1, s["nrep"] + 1), steps=case["steps"])


def run(state):
    if state["kind"] == "step":
        eng = state["eng"]
        eng.set_step(0)
        if eng.nrep > 1:
            eng.set_labels(state["labels"])
        eng.set_state(*state["start"])
        rebuilds = eng.step(state["steps"])
        x, v, a = eng.get_state()
        out = dict(xyz=x, velos=v, accels=a, rebuilds=rebuilds)
        if eng.nrep > 1:
            out["labels"] = eng.labels()
        return out
    if state["kind"] == "serve":
        pool = state["pool"]
        ids = [pool.submit(s, n, seed=state["seed"] + k, precision=p) for k, (s, n, p) in enumerate(state["jobs"])]
        out, wait = {}, set(ids)
        while wait:
            time.sleep(0.0005)
            for j in list(wait):
                st, tm, x = pool.poll(j, want_xyz=True)
                if st == DONE:
                    out[ids.index(j)] = x
                    pool.forget(j)
                    wait.remove(j)
        return [out[k] for k in range(len(ids))]
    if state["kind"] == "eval":
        eng = state["eng"]
        eng.set_state(state["xyz"])
        eng.neighbor_list(0)
        f = eng.force(1, 0)
        return dict(force=f, energy=eng.energy_sumup(1, -1.0, 0, 1))
    return state["eng"].dcd_energies(state["path"], None, state["frames"])


# Half-list entries per bead within the cutoffs that set what a step must
# touch, as the benchmark counts them: (WCA, Debye-Hueckel, base pairs).
def _entries(case):
    if case["conc"] > 0:
        return 1.4, 17.0, 0.65
    n = case["length"]
    return 2.0, min(0.5 * n, 30.0 + 0.1 * n), 1.5


def work(case):
    """The benchmark's algorithmic bytes and the arithmetic of the terms:
    per bead and step the state read and written (144 B), the bonded indices
    (36 B), 8 B a WCA or Debye-Hueckel pair and 44 B a base-pair candidate;
    about 30 operations a pair, 300 a formed-pair candidate, 250 for the
    bonded terms and 150 for noise and update."""
    w, e, b = _entries(case)
    per_bytes, per_flops = 144 + 36 + 8 * w + 8 * e + 44 * b, 30 * (w + e) + 300 * b + 400
    beads = case["chains"] * (case["length"] + max(case["length"], case["length2"])) / 2
    if case["kind"] == "serve":   # mean chains, and mean steps of a log-uniform draw over two decades
        beads, evals = beads / 2, case["nrep"] * case["steps"] * 0.215
    elif case["kind"] == "eval":
        evals = 1
    else:
        evals = case["steps"] * (case["nrep"] if case["kind"] == "remd" else 1)
    return dict(bytes=per_bytes * beads * evals, flops=per_flops * beads * evals)


# ---------------------------------------------------------------------
# the values of eval and dcd in 64 bits: the energy terms in torch, forces
# as their gradient
def _vec(a, b, box):
    v = a - b
    if box is None:
        return v
    return v - box * torch.round(v.detach() / box)


def _angle(a, b):
    return torch.arccos((a * b).sum(1) / (a.norm(dim=1) * b.norm(dim=1)))


def _dihedral(v1, v2, v3):
    """atan2 form for successive vectors v1 (to the axis), v2 (axis), v3."""
    m, n = torch.linalg.cross(v1, v2), torch.linalg.cross(v2, v3)
    return torch.atan2((v1 * n).sum(1) * v2.norm(dim=1), (m * n).sum(1))


def _pairs(x, box, rc):
    """Index pairs i < j closer than rc."""
    out = []
    for s in range(0, len(x), 1000):
        d = x[s: s + 1000, None] - x[None]
        if box is not None:
            d = d - box * torch.round(d / box)
        i, j = torch.nonzero(d.square().sum(2) < rc * rc, as_tuple=True)
        i = i + s
        out.append(torch.stack([i, j])[:, i < j])
    return torch.cat(out, 1)


_TYPES = {"GC": ("GC", 0), "AU": ("AU", 0), "GU": ("GU", 0), "CG": ("GC", 1), "UA": ("AU", 1), "UG": ("GU", 1)}


def _stack(p, five, three):
    """(dH, dS) of the stack 5'-five-3' / 3'-three-5'."""
    for a, b in ((five, three), (three[::-1], five[::-1])):
        if a + "_" + b in NNT_ORDER:
            k = NNT_ORDER.index(a + "_" + b)
            return p["nn_dH"][k], p["nn_dS"][k]
    raise KeyError(five + "_" + three)


def _dg(p, s, i, j, n_i, n_j, same, tempK):
    """Strength of the pair of chain-local i, j (0-based) in sequences s[0]
    and s[1] of lengths n_i and n_j, or None if they may not pair: the
    nearest-neighbour terms of the triplet model, or 1 in model 1."""
    a, b = s[0], s[1]
    if i in (0, n_i - 1) or j in (0, n_j - 1) or a[i] + b[j] not in _TYPES:
        return None
    if same and i + p["bp_min_loop"] >= j:
        return None
    if p["bp_model"] == 1:
        return 1.0
    outer = a[i - 1] + b[j + 1] in _TYPES and i - 1 != 0 and j + 1 != n_j - 1
    inner = a[i + 1] + b[j - 1] in _TYPES and i + 1 != n_i - 1 and j - 1 != 0
    if same and i + 1 + p["bp_min_loop"] >= j - 1:
        inner = False
    if not outer and not inner:
        return None
    h = t = 0.0
    for on, five, three in ((outer, a[i - 1] + a[i], b[j + 1] + b[j]), (inner, a[i] + a[i + 1], b[j] + b[j - 1])):
        if on:
            dh, ds = _stack(p, five, three)
            h += 0.5 * (dh - p["bp_dH0"])
            t += 0.5 * (ds - p["bp_dS0"])
    g = h - tempK * t * 1e-3
    return g if g < 0 else None


def _exact_energy(s, xyz, forces):
    """energies (11,) and, with `forces`, minus their gradient."""
    p, dev = s["params"], torch.device("cuda")
    x = torch.from_numpy(np.array(xyz, np.float64)).to(dev).requires_grad_(forces)
    box = float(p["box"][0]) if p["pbc"] else None
    lens = np.asarray(s["nmp_chain"])
    chain = np.repeat(np.arange(len(lens)), lens)
    first = np.concatenate([[0], np.cumsum(lens)])
    loc = np.arange(len(chain)) - first[chain]

    def runs(m):    # starts of m successive beads of one chain
        k = np.arange(len(chain) - m + 1)
        return torch.from_numpy(k[chain[k] == chain[k + m - 1]]).to(dev)

    e = [torch.zeros((), dtype=torch.float64, device=dev) for _ in range(11)]
    k = runs(2)
    e[1] = (0.5 * p["bond_k"] * (_vec(x[k], x[k + 1], box).norm(dim=1) - p["bond_r0"]) ** 2).sum()
    k = runs(3)
    u, v = _vec(x[k], x[k + 1], box), _vec(x[k + 2], x[k + 1], box)
    if p["angl_reb"]:
        c, c0 = (u * v).sum(1) / (u.norm(dim=1) * v.norm(dim=1)), math.cos(p["angl_t0"])
        e[2] = (0.5 * p["angl_k"] * (c - c0) ** 2 / (1 - c * c)).sum()
    else:
        e[2] = (0.5 * p["angl_k"] * (_angle(u, v) - p["angl_t0"]) ** 2).sum()
    if p["dih_type"] == 2:
        k = runs(4)
        d = _dihedral(_vec(x[k + 1], x[k], box), _vec(x[k + 2], x[k + 1], box), _vec(x[k + 3], x[k + 2], box))
        e[3] = (-p["dih_k"] * torch.exp(-0.5 * p["dih_w"] * (d - p["dih_p0"]) ** 2)).sum()
    # pairs within the largest cutoff of any term
    bp = p["bp"]
    kind = {}
    for name, (of, back) in _TYPES.items():
        q = dict(bp[of])
        if back:
            q.update(angl_k1=q["angl_k2"], angl_k2=q["angl_k1"], angl_k3=q["angl_k4"], angl_k4=q["angl_k3"])
        q["reach"] = 18.0 - 13.8 if p["bp_cutoff_energy"] == 0 else math.sqrt(math.log(abs(10.0 / p["bp_cutoff_energy"])) / q["bond_k"])
        kind[name] = q
    T, salt = p["tempK"], p["ionic_strength"]
    tc = T - 273.15
    eps = 87.740 - 0.40008 * tc + 9.398e-4 * tc ** 2 - 1.410e-6 * tc ** 3
    eps0, ele, kb, na = 8.8541878128e-12, 1.602176634e-19, 1.380649e-23, 6.02214076e23
    bjerrum = ele ** 2 / (4 * math.pi * eps0 * eps * kb * T) * 1e10
    coef = na / 4184.0 * 1e10 * ele ** 2 / (4 * math.pi * eps0 * eps) * (p["length_per_charge"] / bjerrum) ** 2
    lam = 1e10 * math.sqrt(1e-3 * eps0 * eps * kb / (2 * na * ele ** 2)) * math.sqrt(T / salt)
    ij = _pairs(x.detach(), box, max(p["ele_cutoff"], 19.0) + 1e-6)
    i, j = ij[0], ij[1]
    ci, cj = torch.from_numpy(chain).to(dev), torch.from_numpy(loc).to(dev)
    gap = torch.where(ci[i] == ci[j], cj[j] - cj[i], 1 << 20)
    r = _vec(x[i], x[j], box).norm(dim=1)
    m = (gap > 2) & (r < p["wca_sigma"])
    z = (p["wca_sigma"] / r[m]) ** 6
    e[5] = (p["wca_eps"] * (z * z - 2 * z + 1)).sum()
    m = (gap > 2) & (r <= p["ele_cutoff"])
    e[6] = (coef / r[m] * torch.exp(-r[m] / lam)).sum()
    # base pairs
    reach = max(q["bond_r"] + q["reach"] for q in kind.values())
    m = r.detach() < reach
    rows = {}
    for a, b in zip(i[m].tolist(), j[m].tolist()):
        A, B = s["seqs"][chain[a]], s["seqs"][chain[b]]
        g = _dg(p, (A, B), int(loc[a]), int(loc[b]), len(A), len(B), chain[a] == chain[b], T)
        if g is not None:
            rows.setdefault(A[loc[a]] + B[loc[b]], []).append((a, b, g))
    for name, list_ in rows.items():
        q = kind[name]
        t = torch.tensor([(a, b) for a, b, _ in list_], device=dev)
        g = torch.tensor([w for _, _, w in list_], dtype=torch.float64, device=dev)
        a, b = t[:, 0], t[:, 1]
        v12 = _vec(x[a], x[b], box)
        keep = (v12.detach().norm(dim=1) - q["bond_r"]).abs() <= q["reach"]
        a, b, g, v12 = a[keep], b[keep], g[keep], v12[keep]
        v13, v15 = _vec(x[a], x[a - 1], box), _vec(x[a], x[a + 1], box)
        v42, v62 = _vec(x[b - 1], x[b], box), _vec(x[b + 1], x[b], box)
        u = q["bond_k"] * (v12.norm(dim=1) - q["bond_r"]) ** 2
        for w, th, kk in ((v13, "angl_theta2", "angl_k2"), (v42, "angl_theta1", "angl_k1"), (v15, "angl_theta4", "angl_k4"),
                          (v62, "angl_theta3", "angl_k3")):
            if q[kk]:
                u = u + q[kk] * (_angle(v12, w) - q[th]) ** 2
        for w1, w3, kk, ph in ((v42, v13, "dihd_k1", "dihd_phi1"), (v62, v15, "dihd_k2", "dihd_phi2")):
            u = u + q[kk] * (1 + torch.cos(_dihedral(w1, v12, w3) + q[ph]))
        w = q["U0"] * g * torch.exp(-u)
        e[4] = e[4] + w[w.detach() <= p["bp_cutoff_energy"]].sum()
    e[0] = sum(e[1:])
    f = None
    if forces:
        e[0].backward()
        f = -x.grad.cpu().numpy()
    return np.array([float(v.detach()) for v in e]), f


def exact(case, seed):
    """eval and dcd; a run's segment has no value apart from the engine's own
    random streams and limit-MC choices."""
    if case["kind"] not in ("eval", "dcd"):
        return None
    s = _inputs(case, seed)
    if case["kind"] == "eval":
        en, f = _exact_energy(s, s["xyz"][0], True)
        return dict(force=f, energy=en)
    return np.stack([_exact_energy(s, x.astype(np.float32), False)[0] for x in s["xyz"]])
