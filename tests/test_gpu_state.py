"""Bead state in and out, packed by the host for small systems and on the
device for large ones: the same values on both sides of the rule."""
import numpy as np
import pytest

from sis_amd.configs import _mk
from sis_amd.engine import Engine
from sis_amd.forcefield import default_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nrep", [(1, 1), (257, 3), (19999, 1), (20000, 1), (6667, 3)])
def test_state_round_trip(n, nrep):
    print(f"[case] state {n} beads x {nrep}", flush=True)
    rng = np.random.default_rng(n)
    x, v, a = rng.normal(scale=300.0, size=(3, nrep, n, 3))
    s = _mk("beads", ["A"] * n, x[0], default_params())
    s.update(nrep=nrep, temps=np.full(nrep, 300.0), xyz=x)
    e = Engine(s, mode="phases")
    e.set_state(None, v, a)
    for got, want in zip(e.get_state(), (x, v, a)):
        np.testing.assert_array_equal(got, want)
    e.set_state(2.0 * x)
    for got, want in zip(e.get_state(), (2.0 * x, v, a)):
        np.testing.assert_array_equal(got, want)
    e.close()
