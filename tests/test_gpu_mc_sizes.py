"""The limit MC at the edges of its forms (64 pairs: one a lane; 128 and 256:
two and four a lane; above: global memory), choice by choice against the
restatement of the reference's algorithm in test_gpu_mc, in the per-phase and
the batched kernels.  Every case states the component it is about."""
import numpy as np
import pytest

from sis_amd.configs import _mk, random_seq
from sis_amd.engine import Engine
from sis_amd.forcefield import default_params
from tests import test_gpu_mc as ref

pytestmark = pytest.mark.gpu

# beads, radius of the ball, seed, pairs of the largest component
BALLS = [(100, 34.0, 195, 64), (100, 34.0, 109, 65), (110, 31.0, 230, 128), (110, 31.0, 252, 129), (190, 37.0, 112, 256),
         (200, 40.0, 189, 257), (200, 36.0, 8, 355)]


def _components(pairs):
    """Bead sets and pair counts of the components."""
    parent = {}

    def find(x):
        parent.setdefault(x, x)
        while parent[x] != x:
            x = parent[x]
        return x

    for a, b in pairs:
        a, b = find(a), find(b)
        parent[max(a, b)] = min(a, b)
    beads, count = {}, {}
    for x in list(parent):
        beads.setdefault(find(x), []).append(x)
    for a, _ in pairs:
        count[find(a)] = count.get(find(a), 0) + 1
    return beads, count


def _check(s, mode, prec):
    """(formed pairs, components) after comparing one evaluation's choices."""
    seed, rep, step = 0x1234567890ABCDEF, 0, 77
    if mode == "batched":     # a second replica, whose evaluation is of the step to come
        s.update(nrep=2, temps=np.full(2, 310.0), xyz=np.repeat(s["xyz"].reshape(1, -1, 3), 2, axis=0))
        rep = 1
    e = Engine(s, precision=prec, mode=mode, seed=seed)
    e.set_step(step)
    e.neighbor_list(0)
    e.force(rep + 1, 1)
    b = e.bp(rep + 1)
    e.close()
    formed = np.signbit(b["ene"])
    pairs = [tuple(int(v) for v in q[:2] - 1) for q in b["bp"][formed]]
    beta = 1.0 / (1.380649e-23 * ((1.0 / 4184.0) * 6.02214076e23) * 310.0)
    left, _ = ref._limit_mc(pairs, b["ene"][formed], beta, seed, rep, step + rep, s["params"]["max_bp_per_nt"])
    assert not np.any(b["status"][~formed])
    np.testing.assert_array_equal(b["status"][formed] != 0, left)
    return pairs, _components(pairs)


@pytest.mark.parametrize("n,radius,seed,size", BALLS)
@pytest.mark.parametrize("mode", ["phases", "batched"])
@pytest.mark.parametrize("prec", [0, 1])
def test_component_sizes(n, radius, seed, size, mode, prec):
    print(f"[case] limit MC, {size} pairs, {mode}, prec {prec}", flush=True)
    rng = np.random.default_rng(seed)
    s = _mk("ball", [random_seq(rng, n, 0.5)], ref._cloud(rng, [n], radius), default_params(tempK=310.0, nl_margin=5.0))
    _, (_, count) = _check(s, mode, prec)
    assert max(count.values()) == size


def test_many_pairs_a_nucleotide():
    print("[case] limit MC, more than eight pairs a nucleotide", flush=True)
    pairs, _ = _check(ref._system(dict(kind="ball", seed=5, n=120, radius=26.0)), "phases", 0)
    assert np.bincount(np.ravel(pairs)).max() > 8


def test_beads_numbered_far_apart():
    print("[case] limit MC, bead numbers of a component 2,048 apart", flush=True)
    _, (beads, _) = _check(ref._system(dict(kind="far", seed=7)), "phases", 0)
    assert max(max(v) - min(v) for v in beads.values()) > 2048
