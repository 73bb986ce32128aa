"""The limit MC of the performance form, choice by choice: the formed pairs
left by one force evaluation equal those of a plain restatement of the
reference's algorithm per conflict component (src/force_bp_limit_triplet.F90:259-330)
on the same Philox draws.  Energies come from the engine; the deletions are
whole-number decisions, so the sets are equal."""
import math

import numpy as np
import pytest

from sis_amd import configs
from sis_amd.configs import _mk, random_seq
from sis_amd.engine import Engine
from sis_amd.forcefield import default_params

pytestmark = pytest.mark.gpu

M32 = 0xFFFFFFFF


def _philox(c, k0, k1):
    c = list(c)
    for _ in range(10):
        p0, p1 = 0xD2511F53 * c[0], 0xCD9E8D57 * c[2]
        c = [(p1 >> 32) ^ c[1] ^ k0, p1 & M32, (p0 >> 32) ^ c[3] ^ k1, p0 & M32]
        k0, k1 = (k0 + 0x9E3779B9) & M32, (k1 + 0xBB67AE85) & M32
    return c


def _uniform(seed, rep, step, root, draw):
    o = _philox([step & M32, (step >> 32) ^ 0x4D43, root, draw], seed & M32,
                (seed >> 32) ^ ((0x5BD1E995 * (rep + 1)) & M32))
    m = ((o[0] << 21) ^ (o[1] >> 11)) & ((1 << 53) - 1)
    return (float(m) + 0.5) * (1.0 / 9007199254740992.0)


def _limit_mc(pairs, ene, beta, seed, rep, step, max_bp):
    """Pairs (n, 2) of 0-based beads in list order; returns who is left and
    the sizes of the components with excess."""
    parent = {}

    def find(x):
        parent.setdefault(x, x)
        while parent[x] != x:
            x = parent[x]
        return x

    for a, b in pairs:
        ra, rb = find(a), find(b)
        parent[max(ra, rb)] = min(ra, rb)
    alive = np.ones(len(pairs), bool)
    comps = {}
    for k, (a, _) in enumerate(pairs):
        comps.setdefault(find(a), []).append(k)
    sizes = []
    for root, ks in comps.items():
        count = {}
        for k in ks:
            for x in pairs[k]:
                count[x] = count.get(x, -max_bp) + 1
        draw, first = 0, True
        while True:
            act = sorted(x for x, c in count.items() if c > 0)
            if not act:
                break
            if first:
                sizes.append(len(ks))
                first = False
            u = [_uniform(seed, rep, step, root, draw)]
            nt = act[math.ceil(u[0] * len(act)) - 1]
            seq = [k for k in ks if alive[k] and nt in pairs[k]]
            ns = len(seq)
            u += [_uniform(seed, rep, step, root, draw + j) for j in range(1, 2 * ns)]
            for i in range(ns):
                s = math.ceil(u[1 + i] * ns) - 1
                seq[i], seq[s] = seq[s], seq[i]
            gone = seq[0]
            for i in range(1, ns):
                if math.log(u[ns + i]) < (ene[seq[i]] - ene[gone]) * beta:
                    gone = seq[i]
            draw += 2 * ns
            alive[gone] = False
            for x in pairs[gone]:
                count[x] -= 1
    return alive, sizes


def _cloud(rng, nmp_chain, radius, centre=(0.0, 0.0, 0.0)):
    """Beads spread through a ball: distances where pairs form are common, so
    the conflict components are as dense as the radius makes them."""
    n = int(np.sum(nmp_chain))
    d = rng.normal(size=(n, 3))
    d *= (radius * rng.random(n) ** (1 / 3) / np.linalg.norm(d, axis=1))[:, None]
    return d + np.asarray(centre)


def _system(case):
    rng = np.random.default_rng(case["seed"])
    p = default_params(tempK=310.0, nl_margin=5.0, max_bp_per_nt=case.get("max_bp", 1))
    if case["kind"] == "coil":
        return configs.hairpin64(case["seed"])
    if case["kind"] == "far":
        # two chains at one place, numbered 60 chains of 40 beads apart: the
        # bead ids of a component span more than 2,048
        lens = [40] * 60
        x = np.concatenate([_cloud(rng, [40], 18.0, (900.0 * (k % 59), 0.0, 0.0)) for k in range(60)])
        return _mk("far", [random_seq(rng, n, 0.5) for n in lens], x, p)
    return _mk("ball", [random_seq(rng, case["n"], 0.5)], _cloud(rng, [case["n"]], case["radius"]), p)


CASES = [
    dict(kind="coil", seed=3),                                   # a few pairs
    dict(kind="ball", seed=1, n=90, radius=60.0),                # pairs of pairs: one lane each
    dict(kind="ball", seed=2, n=130, radius=48.0),               # up to 64 pairs
    dict(kind="ball", seed=3, n=100, radius=30.0),               # 65 to 128 pairs
    dict(kind="ball", seed=4, n=190, radius=45.0),               # about the edges of 128 pairs and nucleotides
    dict(kind="ball", seed=5, n=120, radius=26.0),               # more than 8 pairs a nucleotide
    dict(kind="ball", seed=6, n=130, radius=44.0, max_bp=2),     # two pairs allowed
    dict(kind="far", seed=7),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(v) for v in c.values()))
@pytest.mark.parametrize("prec", [0, 1])
def test_limit_mc_decisions(case, prec):
    s = _system(case)
    print(f"[case] limit MC {case} prec {prec}", flush=True)
    seed = 0x1234567890ABCDEF
    e = Engine(s, precision=prec, mode="phases", seed=seed)
    e.set_step(77)
    e.neighbor_list(0)
    e.force(1, 1)
    b = e.bp(1)
    e.close()
    formed = np.signbit(b["ene"])      # every formed pair has a negative energy, however small
    pairs = [tuple(int(v) for v in q[:2] - 1) for q in b["bp"][formed]]
    beta = 1.0 / (1.380649e-23 * ((1.0 / 4184.0) * 6.02214076e23) * s["params"]["tempK"])
    left, sizes = _limit_mc(pairs, b["ene"][formed], beta, seed, 0, 77, s["params"]["max_bp_per_nt"])
    print(f"[case] {len(pairs)} formed pairs, components with excess: {sorted(sizes)}", flush=True)
    assert sizes
    assert not np.any(b["status"][~formed])
    np.testing.assert_array_equal(b["status"][formed] != 0, left)


def test_batched_form_with_many_components():
    """More wavefront components in a replica than the batched kernel's sorted
    list holds (64): the formed pairs that one step's limit MC leaves are
    those of the per-phase form, whole-number decisions on the same draws."""
    rng = np.random.default_rng(11)
    n, ncl, nrep = 12, 85, 2     # clusters of G and C along one chain, out of each other's reach
    x = np.concatenate([_cloud(rng, [n], 11.0, (60.0 * (k % 10), 60.0 * (k // 10), 0.0)) for k in range(ncl)])
    s = _mk("clusters", [random_seq(rng, n * ncl, 1.0)], x, default_params(tempK=310.0, nl_margin=5.0), nrep=nrep,
            temps=np.array([300.0, 330.0]))
    print("[case] limit MC, batched form, many components", flush=True)
    res = []
    for mode in ("phases", "batched"):
        e = Engine(s, mode=mode, seed=21)
        e.neighbor_list(0)
        if mode == "phases":
            e.force(1, 1)
            b = e.bp(1)
            f = np.signbit(b["ene"])
            pairs = [tuple(int(v) for v in q[:2] - 1) for q in b["bp"][f]]
            _, sizes = _limit_mc(pairs, b["ene"][f], 1.6, 21, 0, 0, 1)
            print(f"[case] components with excess: {sorted(sizes)}", flush=True)
            assert sum(v > 2 for v in sizes) > 64
        e.step(1)
        assert e.info()["mode"] == {"phases": 1, "batched": 3}[mode]
        res.append([e.bp(r) for r in range(1, nrep + 1)])
        e.close()
    for a, b in zip(*res):
        np.testing.assert_array_equal(a["bp"], b["bp"])
        assert np.any(a["status"])
        np.testing.assert_array_equal(a["status"] != 0, b["status"] != 0)
