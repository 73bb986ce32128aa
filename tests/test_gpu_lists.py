"""Neighbour lists of the cell search (periodic box) against the all-pairs
search (no box) on the same coordinates, a bead cloud in the middle of a box
too wide for any image: the same pairs and candidates in the same order.
Dense enough for beads with more base-pair partners than a wavefront's
buffer (64), more incidences than the sort's LDS rows (32), and neighbour
counts on both sides of 64; the sizes sit at the edges of a wavefront's and
a block's share."""
import numpy as np
import pytest

from sis_amd.configs import _mk, random_seq
from sis_amd.engine import Engine
from sis_amd.forcefield import default_params

pytestmark = pytest.mark.gpu


def _cloud(rng, n, radius):
    d = rng.normal(size=(n, 3))
    return d * (radius * rng.random(n) ** (1 / 3) / np.linalg.norm(d, axis=1))[:, None]


@pytest.mark.parametrize("lens,radius", [([1024], 60.0), ([1025], 200.0), ([700, 1, 326], 40.0), ([513, 514], 130.0), ([1030], 24.0)])
def test_cell_lists_equal_all_pairs(lens, radius):
    rng = np.random.default_rng(sum(lens) + int(radius))
    n = sum(lens)
    x = _cloud(rng, n, radius) + 600.0
    seqs = [random_seq(rng, k, 0.5) for k in lens]
    out = []
    for box in (1200.0, 0.0):
        over = dict(pbc=1, box=[box] * 3) if box else {}
        e = Engine(_mk("cloud", seqs, x, default_params(nl_margin=5.0, **over)), mode="phases")
        e.neighbor_list(0)
        out.append(e.lists(1))
        e.close()
    print(f"[case] lists {lens} {radius}: " + ", ".join(f"{k} {len(v)}" for k, v in out[0].items()), flush=True)
    for k in ("wca", "ele", "bp", "bpcoef"):
        np.testing.assert_array_equal(out[0][k], out[1][k])
    if radius <= 24.0:
        assert np.bincount(out[0]["bp"][:, 0]).max() > 64
