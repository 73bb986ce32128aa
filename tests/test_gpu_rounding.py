"""Rounding of the pair sums and of the Brownian move.

The force of every pair is rounded before it is added, in FP64 too: one
bead's force from two neighbours that the same lane adds is then exactly the
rounded sum of the two single-pair forces.

Brownian runs at dt 0.05 move a bead by 0.13 of its force, at which a
15 kcal/mol/A^2 bond is past the edge of stability: every last bit grows by
about 7 a step.  Such runs repeat, bit for bit and with the same list rebuilds,
what the library gave before its pair forces and step launches were rewritten.
The digests are of that library's own outputs (`python tests/test_gpu_rounding.py`
prints them), until well after coordinates stop being finite; they hold for
the compiler it was built with (ROCm 7.2)."""
import hashlib
import sys

import numpy as np
import pytest

if __name__ == "__main__":
    sys.path.insert(0, ".")

from sis_amd.configs import _mk, random_coil, random_seq
from sis_amd.engine import Engine
from sis_amd.forcefield import default_params, nht22_params
from sis_amd.serving import DONE, JobPool

pytestmark = pytest.mark.gpu


def _pairs_system(kind, at, only):
    """Single-bead chains: bead 0 at the origin of each replica, neighbours
    1 and 9 at `at[replica]`, and between them seven that stand within the
    list's reach but beyond the cutoff, so that the eight lanes that share a
    bead give neighbours 1 and 9 to one lane.  only: 1 or 9 alone stays."""
    if kind == "ele":    # 12 to 30 A: beyond the WCA reach
        p, far, near = default_params(nl_margin=20.0), 55.0, (12.0, 30.0)
    else:
        p, far, near = default_params(nl_margin=20.0, ele_on=0), 14.0, (7.0, 9.5)
    rng = np.random.default_rng(17)
    nrep = at
    d = rng.normal(size=(nrep, 2, 3))
    d *= (rng.uniform(*near, (nrep, 2)) / np.linalg.norm(d, axis=2))[..., None]
    x = np.zeros((nrep, 10, 3))
    x[:, 1], x[:, 9] = d[:, 0], d[:, 1]
    t = 2 * np.pi * np.arange(7) / 7
    x[:, 2:9] = far * np.stack([np.cos(t), np.sin(t), 0 * t], 1)
    if only == 1:
        x[:, 9] = [0.0, 0.0, -far]
    elif only == 9:
        x[:, 1] = [0.0, 0.0, -far]
    s = _mk("pairs", ["A"] * 10, x[0], p)
    s.update(nrep=nrep, temps=np.full(nrep, 300.0), xyz=x)
    return s


@pytest.mark.parametrize("kind", ["ele", "wca"])
@pytest.mark.parametrize("mode", ["phases", "batched"])
def test_pair_force_is_rounded_before_the_sum(kind, mode):
    nrep = 48
    f = {}
    for only in (0, 1, 9):
        print(f"[case] rounded pair forces {kind} {mode} {only}", flush=True)
        e = Engine(_pairs_system(kind, nrep, only), mode=mode)
        e.neighbor_list(0)
        f[only] = np.stack([e.force(r + 1, 0)[0] for r in range(nrep)])
        e.close()
    assert np.abs(f[1]).min() > 0 and np.abs(f[9]).min() > 0
    np.testing.assert_array_equal(f[0], f[1] + f[9])


# ---------------------------------------------------------------------
def _chains(lens, seed, params):
    rng = np.random.default_rng(seed)
    x = np.concatenate([random_coil(rng, n, start=np.array([0.0, 400.0 * (k % 8), 400.0 * (k // 8)])) for k, n in enumerate(lens)])
    return _mk("chains", [random_seq(rng, n, 0.5) for n in lens], x, params)


def _brownian(case, prec):
    """Steps, and everything the run leaves."""
    p = (nht22_params if case == "model 1" else default_params)(nl_margin=5.0, integrator=2, dt=0.05)
    if "job" in case:
        s = _chains([300, 20] if case == "job" else [800] * 3, 2, p)
        with JobPool() as pool:
            j = pool.submit(s, 60, seed=6, precision=prec)
            st = -1
            while st != DONE:
                st, _, x = pool.poll(j, want_xyz=True)
        return [x]
    kw = dict(mode="phases")
    if case in ("ladder", "ladder, 512 threads"):
        s = _chains([300], 9, p)
        s.update(nrep=4, temps=290.0 * 1.3 ** (np.arange(4) / 3), xyz=np.repeat(s["xyz"], 4, axis=0))
        kw = dict(mode="batched", exchange_every=50, block=512 if "512" in case else 0)
    elif case == "model 1":
        s = _chains([97, 60], 4, p)
    else:
        s = _chains([150], 6, p)
        kw = dict(mode="persistent" if case == "persistent" else "phases", no_graph=case == "no graph")
    e = Engine(s, precision=prec, seed=99, **kw)
    e.init_velocities()
    e.neighbor_list(0)
    rebuilds = e.step(120)
    x, v, _ = e.get_state()
    e.close()
    return [x, v, np.array([rebuilds])]


def _digest(arrays):
    h = hashlib.sha256()
    for a in arrays:
        a = np.array(a)
        if a.dtype.kind == "f":
            a[np.isnan(a)] = np.nan   # one NaN
        h.update(np.ascontiguousarray(a).tobytes())
    return h.hexdigest()[:20]


DIGESTS = {
    ("chain", 0): "6e922836599731dbb7e2",
    ("chain", 1): "b1e68d9d4084a50ae2b7",
    ("no graph", 0): "6e922836599731dbb7e2",
    ("no graph", 1): "b1e68d9d4084a50ae2b7",
    ("model 1", 0): "338fa3ec446b1083a269",
    ("model 1", 1): "c83632bc404e7afff558",
    ("persistent", 0): "0a7fcda323def42f3d69",
    ("persistent", 1): "e24efd3a79255f7f060b",
    ("ladder", 0): "208e0645617363166670",
    ("ladder", 1): "8be83cb1026f487dd6ec",
    ("ladder, 512 threads", 0): "208e0645617363166670",
    ("ladder, 512 threads", 1): "8be83cb1026f487dd6ec",
    ("job", 0): "b7a585f32aafebe271c9",
    ("job", 1): "3ab300a22b1c21bb3d61",
    ("large job", 0): "442b2307beb9ce1dec67",
    ("large job", 1): "10c9ed7043e0d5a5b40e",
}


@pytest.mark.parametrize("case,prec", list(DIGESTS))
def test_brownian_runs_repeat(case, prec):
    print(f"[case] Brownian, dt 0.05: {case}, prec {prec}", flush=True)
    assert _digest(_brownian(case, prec)) == DIGESTS[case, prec]


if __name__ == "__main__":
    for case in ("chain", "no graph", "model 1", "persistent", "ladder", "ladder, 512 threads", "job", "large job"):
        for prec in (0, 1):
            print(f'    ("{case}", {prec}): "{_digest(_brownian(case, prec))}",', flush=True)
