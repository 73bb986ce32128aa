"""Device-driven batches of steps at the places where the device and the
host agree on how far a batch got: halts for a rebuild, the stop, and a
conflict component above the bucket capacity (256 pairs), whose step waits
for the host.  Compared with the general path, which launches every phase by
itself (taken with external terms: here an Rg bias of strength zero): the
same lists, draws and limit-MC choices, sums in another order, so coordinates
of up to 1,000 A agree within 1e-9 A over these smooth runs."""
import time

import numpy as np
import pytest
import torch

from sis_amd import configs
from sis_amd.engine import Engine
from sis_amd.forcefield import default_params
from sis_amd.serving import RUNNING, JobPool

pytestmark = pytest.mark.gpu


def _largest(e):
    """Pairs of the largest component of the formed pairs (before deletions)."""
    b = e.bp(1)
    pairs = b["bp"][np.signbit(b["ene"])][:, :2].astype(int)
    parent = {}

    def find(x):
        parent.setdefault(x, x)
        while parent[x] != x:
            x = parent[x]
        return x

    for i, j in pairs:
        i, j = find(i), find(j)
        parent[max(i, j)] = min(i, j)
    return max(np.unique([find(i) for i, _ in pairs], return_counts=True)[1])


def _chain(nstep_mc, **over):
    rng = np.random.default_rng(11)
    seq = configs.random_seq(rng, 2048, 0.6)
    return configs._mk("chain2048", [seq], configs.random_coil(rng, 2048),
                       default_params(tempK=300.0, nl_margin=15.0, nstep_bp_mc=nstep_mc, **over))


@pytest.fixture(scope="module")
def large_state():
    """A state of a 2,048-nt chain with a component of about 320 pairs."""
    e = Engine(_chain(1), mode="phases", seed=9)
    e.init_velocities()
    e.neighbor_list(0)
    e.step(100)
    st = e.get_state()
    n = _largest(e)
    e.close()
    print(f"[case] largest component {n}", flush=True)
    assert n > 280
    return st


def _run(state, every, at, n, general=False, no_graph=False, **over):
    """n steps whose at-th is the first with a limit MC."""
    e = Engine(_chain(every, **over), mode="phases", seed=9, no_graph=no_graph)
    if general:
        e.set_external(dict(rg=1, rg_k=0.0, rg_0=10.0))
    e.set_state(*state)
    e.neighbor_list(0)
    e.set_step(every - at)
    rebuilds = e.step(n)
    out = (*e.get_state(), e.info()["istep"], rebuilds, e.bp(1)["status"])
    if general and n == at:
        assert _largest(e) > 256
    e.close()
    return out


def _same(a, b, end):
    assert a[3] == b[3] == end
    assert a[4] == b[4] == 0
    np.testing.assert_array_equal(a[2], b[2])      # noise terms: the same draws
    np.testing.assert_array_equal(a[5], b[5])
    assert np.abs(a[0] - b[0]).max() < 1e-9


@pytest.mark.parametrize("every", [1000, 40])
def test_first_large_component_at_every_place_of_a_batch(large_state, every):
    """The first component above the bucket capacity at the edges of a run's
    first and third batch of 16 steps and at every place of its second, the
    run ending there or later; every = 40: met again after the hand-over.
    Replayed from a graph and issued directly."""
    for at in (1, 2, 15, *range(16, 34), 47, 48, 49) if every > 49 else (1, 16, 31, 32, 33):
        for n in (at, at + 20) if at in (1, 16, 32, 33) else (at + 20,):
            want = _run(large_state, every, at, n, general=True)
            for no_graph in (False, True):
                print(f"[case] first large component at step {at} of {n}, every {every}, no_graph {no_graph}", flush=True)
                _same(_run(large_state, every, at, n, no_graph=no_graph), want, every - at + n)


@pytest.mark.parametrize("at", [31, 32, 33])
def test_first_large_component_brownian(large_state, at):
    print(f"[case] first large component at step {at}, Brownian", flush=True)
    kw = dict(integrator=2, dt=0.005)
    _same(_run(large_state, 1000, at, at + 20, **kw), _run(large_state, 1000, at, at + 20, general=True, **kw), 1020)


@pytest.mark.parametrize("case", ["chain, MC every step", "ladder, MC every 3", "box"])
def test_batches_with_rebuilds_match_single_launches(case):
    """200 steps with halts for rebuilds inside the batches (0.3 to 1 A
    skins), the limit MC after them, and exchanges: replayed and issued
    directly they give the same bits, and the general path the same labels,
    rebuilds, noise and formed pairs.  Coordinates within 1e-6 A, as other
    forms agree over hundreds of steps."""
    nex = 0
    if case == "chain, MC every step":
        s = configs.remd_c3(nrep=1, n=128, seed=3, margin=0.3)
    elif case == "ladder, MC every 3":
        s, nex = configs.remd_c3(nrep=4, n=128, seed=3, margin=1.0), 25
        s["params"] = dict(s["params"], nstep_bp_mc=3)
    else:
        s = configs.cag_system(40, 47, 1.0, 310.0, margin=1.0)
    out = []
    for general, no_graph in ((True, False), (False, False), (False, True)):
        print(f"[case] batches with rebuilds: {case}, general {general}, no_graph {no_graph}", flush=True)
        e = Engine(s, mode="phases", precision=1, seed=4242, exchange_every=nex, no_graph=no_graph)
        if general:
            e.set_external(dict(rg=1, rg_k=0.0, rg_0=10.0))
        e.init_velocities()
        e.neighbor_list(0)
        reb = e.step(37) + e.step(163)
        out.append((*e.get_state(), reb, e.labels(), [e.bp(r + 1)["status"] for r in range(s["nrep"])]))
        e.close()
    for a in out[1:]:
        assert a[3] == out[0][3] > 2
        np.testing.assert_array_equal(a[4], out[0][4])
        np.testing.assert_array_equal(a[2], out[0][2])
        for u, v in zip(a[5], out[0][5]):
            np.testing.assert_array_equal(u, v)
        assert np.abs(a[0] - out[0][0]).max() < 1e-6
    for u, v in zip(out[1][:3], out[2][:3]):
        np.testing.assert_array_equal(u, v)


def _lattice(nch, n=100):
    """Zigzag chains on a lattice, 50 A apart."""
    k = np.arange(n)
    one = np.stack([5.7 * k, 1.5 * (k % 2), 0.0 * k], 1)
    at = np.array([[0.0, 50.0 * (c // 40), 50.0 * (c % 40)] for c in range(nch)])
    rng = np.random.default_rng(5)
    return configs._mk("lattice", [configs.random_seq(rng, n, 0.5)] * nch, (one + at[:, None]).reshape(-1, 3),
                       default_params(nl_margin=5.0))


@pytest.mark.parametrize("nch,prec", [(204, 0), (205, 0), (205, 1)])
def test_pair_tiles_without_limit_mc(nch, prec):
    """Both sides of the rule that gives the pair tiles a launch of their own
    when the limit MC is off (640 tiles of 32 beads)."""
    print(f"[case] pair tiles without limit MC, {100 * nch} beads, prec {prec}", flush=True)
    s = _lattice(nch)
    s["params"]["nstep_bp_mc"] = 0
    out = []
    for general in (True, False):
        e = Engine(s, mode="phases", precision=prec, seed=4)
        if general:
            e.set_external(dict(rg=1, rg_k=0.0, rg_0=10.0))
        e.init_velocities()
        e.neighbor_list(0)
        e.step(20)
        out.append(e.get_state())
        e.close()
    np.testing.assert_array_equal(out[0][2], out[1][2])
    assert np.abs(out[0][0] - out[1][0]).max() < 1e-9
    assert np.abs(out[0][1] - out[1][1]).max() < 1e-12


def test_pool_counts_what_a_large_job_steps_with():
    """A job above one workgroup's size is charged for the buffers of its
    step batches (64 B a bead, 7.7 MB here) when it is admitted: as much as
    an engine of the same system holds after its first steps.  2 MB: the
    granularity of the card's memory count."""
    small, big = _lattice(30), _lattice(1200)
    for _ in range(5):     # what the kernels themselves need, on every queue
        e = Engine(small, mode="phases", no_graph=True)
        e.neighbor_list(0)
        e.step(20)
        e.close()
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    e = Engine(big, mode="phases", no_graph=True)
    e.neighbor_list(0)
    e.init_velocities()
    e.step(20)
    held = free - torch.cuda.mem_get_info()[0]
    e.close()
    with JobPool(quantum_bead_steps=big["xyz"].size) as pool:
        j = pool.submit(big, 10 ** 6, seed=3)
        until = time.time() + 60
        while pool.poll(j)[1][3] < 10 and time.time() < until:
            time.sleep(0.01)
        assert pool.poll(j)[0] == RUNNING
        charged = pool.stats()["bytes"]
    print(f"[case] large job: engine holds {held}, pool charges {charged}", flush=True)
    assert charged > held - (2 << 20)


def test_step_time_without_graph():
    """sis_gpu_last_kernel_ms 3 and 4 of a context without graphs: a figure
    for one step of every batch that ran that far (a skin of 0.3 A: steps
    issued after a halt do not count), together no longer than the call."""
    s = configs.remd_c3(nrep=1, n=128, seed=3, margin=0.3)
    e = Engine(s, mode="phases", seed=1, no_graph=True)
    e.init_velocities()
    e.neighbor_list(0)
    rebuilds = e.step(90)
    ms, n = e.last_ms(3), e.last_ms(4)
    print(f"[case] step time without graph {ms} x {n}, call {e.last_ms(0)}, {rebuilds} rebuilds", flush=True)
    assert rebuilds > 2
    assert 1 <= n <= 90 // 16 + rebuilds + 1
    assert 0.0 < ms * n < e.last_ms(0)
    e.step(1)
    assert e.last_ms(4) == 1
    e.close()


@pytest.mark.parametrize("integrator", [1, 2])
@pytest.mark.parametrize("pairs,bad", [(64, 47), (512, 383), (1200, 1151), (9000, 8959)])
def test_a_nan_bead_does_not_hide_the_others(integrator, pairs, bad):
    """Two-bead chains out of each other's reach, the first ones stretched
    (Brownian) or fast (Langevin) so that they move furthest by far, one in
    the middle with a NaN coordinate (the last bead of a block of 32 and of
    256, whose maximum stays NaN): the run rebuilds where it does with that
    chain at rest, over few, tens and hundreds of blocks of maxima."""
    print(f"[case] NaN bead, {pairs} pairs, integrator {integrator}", flush=True)
    k = np.arange(pairs)
    x = np.zeros((pairs, 2, 3))
    x[:, 0] = np.stack([90.0 * (k % 30), 90.0 * (k // 30 % 30), 90.0 * (k // 900)], 1)
    x[:, 1] = x[:, 0] + [5.9, 0.0, 0.0]
    v = np.zeros_like(x)
    if integrator == 2:
        x[:3, 1, 0] += 40.0
    else:
        v[:3] = 10.0
    out = []
    for nan in (False, True):
        if nan:
            x[bad, 1, 0] = np.nan
        s = configs._mk("pairs", ["AA"] * pairs, x.reshape(-1, 3),
                        default_params(nl_margin=10.0, integrator=integrator, dt=0.05 if integrator == 1 else 0.005, ele_on=0))
        e = Engine(s, mode="phases", seed=4)
        e.set_state(None, v.reshape(1, -1, 3), 0.0 * v.reshape(1, -1, 3))
        e.neighbor_list(0)
        out.append([e.step(6) for _ in range(10)])
        e.close()
    print(f"[case] rebuilds {out}", flush=True)
    assert sum(out[0]) > 0
    assert out[0] == out[1]
