"""Device-driven batches of steps (four launches a step) against the general
path that launches every phase by itself, which a context with external
terms takes: here an Rg bias of strength zero.  Same lists, draws and
limit-MC choices, sums in another order: FP64 differences of a few 1e-16 a
term that 40 steps of smooth dynamics carry along, so coordinates of up to
1,000 A agree within 1e-9 A (and velocities of about 0.1 within 1e-12)."""
import numpy as np
import pytest

from sis_amd import configs
from sis_amd.abi import MOLT_CIRCRNA
from sis_amd.configs import _mk, random_coil, random_seq
from sis_amd.engine import Engine
from sis_amd.forcefield import default_params, nht22_params

pytestmark = pytest.mark.gpu


def _chains(lens, seed, params, circular=()):
    rng = np.random.default_rng(seed)
    x = np.concatenate([random_coil(rng, n, start=np.array([0.0, 400.0 * (k % 8), 400.0 * (k // 8)])) for k, n in enumerate(lens)])
    s = _mk("chains", [random_seq(rng, n, 0.5) for n in lens], x, params)
    for k in circular:
        s["moltype"][k] = MOLT_CIRCRNA
    return s


def _ring(n, bond=5.9):
    t = 2 * np.pi * np.arange(n) / n
    return np.stack([np.cos(t), np.sin(t), 0.15 * np.cos(3 * t)], 1) * bond / (2 * np.sin(np.pi / n))


def _system(case):
    if case == "short chains":        # 1 to 5 beads: terms that do not exist
        return _chains([1, 2, 3, 4, 5, 30], 1, default_params(nl_margin=5.0))
    if case in ("252", "253", "254", "257"):   # edges of the bead tiles and of the update's blocks
        return _chains([int(case)], 2, default_params(nl_margin=5.0))
    if case == "513 in chains":
        return _chains([255, 1, 257], 3, default_params(nl_margin=5.0))
    if case == "no MC, model 1":
        return _chains([97, 60], 4, nht22_params(nl_margin=5.0))
    if case == "MC every 3, cosine":
        return _chains([120], 5, default_params(nl_margin=1.0, nstep_bp_mc=3, dih_type=1, dih_k=1.0, dih_p0=0.3))
    if case == "Brownian":
        return _chains([150], 6, default_params(nl_margin=5.0, integrator=2, dt=0.005))   # the Brownian tests' step: stable
    if case == "circular":
        rng = np.random.default_rng(7)
        s = _mk("circular", [random_seq(rng, 40, 0.5), random_seq(rng, 33, 0.5)],
                np.concatenate([_ring(40), random_coil(rng, 33, start=np.array([300.0, 0.0, 0.0]))]), default_params(nl_margin=5.0))
        s["moltype"][0] = MOLT_CIRCRNA
        return s
    if case == "box":
        return configs.cag_system(40, 47, 1.0, 310.0, margin=1.0)
    if case == "replicas":
        return configs.remd_c3(nrep=3, n=64, seed=3, margin=1.0)
    s = _chains([600, 520], 8, default_params(nl_margin=0.5))      # "replicas, many blocks"
    s.update(nrep=2, temps=np.array([300.0, 330.0]), xyz=np.repeat(s["xyz"], 2, axis=0))
    return s


CASES = ["short chains", "252", "253", "254", "257", "513 in chains", "no MC, model 1", "MC every 3, cosine", "Brownian",
         "circular", "box", "replicas", "replicas, many blocks"]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("prec", [0, 1])
def test_batched_steps_match_single_launches(case, prec):
    s = _system(case)
    print(f"[case] step batches: {case}, prec {prec}", flush=True)
    out = []
    for general in (False, True):
        e = Engine(s, mode="phases", precision=prec, seed=99)
        if general:
            e.set_external(dict(rg=1, rg_k=0.0, rg_0=10.0))
        e.init_velocities()
        e.neighbor_list(0)
        reb = e.step(7) + e.step(33)
        out.append((*e.get_state(), reb, e.bp(1)["status"]))
        e.close()
    (xa, va, ba, ra, sa), (xb, vb, bb, rb, sb) = out
    assert ra == rb
    np.testing.assert_array_equal(sa, sb)
    np.testing.assert_array_equal(ba, bb)      # noise terms: the same draws
    assert np.abs(xa - xb).max() < 1e-9
    assert np.abs(va - vb).max() < 1e-12 or s["params"]["integrator"] == 2
