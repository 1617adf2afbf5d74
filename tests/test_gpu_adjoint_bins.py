"""The FP64 adjoint on tile bins against the unsorted engine (the same arithmetic per particle,
another order of the current and field-adjoint sums): tile edges, ragged boxes, segments that do
not divide the run, the current filter, and what it refuses or leaves to the unsorted engine."""
import numpy as np
import pytest

from pictor_amd import Simulation, setup_weibel
from pictor_amd._lib import PictorError

from _util import say

pytestmark = pytest.mark.gpu

ARGS = ("q", "x", "y", "z", "u", "v", "w", "flv")


def _gradient(P, n, tile, engine, nsteps, segment, filt=0):
    with Simulation(*n, epc=8, form="fp64", tile=tile, curr_filter=filt) as sim:
        sim.adjoint_engine(engine)
        L = sim.adjoint_forward(*[P[k] for k in ARGS], nsteps, segment)
        g = sim.adjoint_backward(2.0)
        return L, np.stack(g), sim.adjoint_stats()["engine"]


@pytest.mark.parametrize("n,tile", [((8, 8), 8), ((24, 40), 8), ((16, 16), 16), ((48, 16), 16)])
@pytest.mark.parametrize("nsteps,segment,filt", [(1, 1, 0), (7, 3, 0), (12, 12, 2), (9, 1, 0)])
def test_bins_match_unsorted(n, tile, nsteps, segment, filt):
    say(n, tile, nsteps, segment, filt)
    P = setup_weibel(*n, epc=8, drift=0.5, uth=0.2, seed=9)
    rng = np.random.default_rng(3)
    keep = rng.permutation(len(P["x"]))[: len(P["x"]) - 77]     # any order, a ragged count
    P = {k: np.ascontiguousarray(v[keep]) for k, v in P.items()}
    L1, g1, e1 = _gradient(P, n, tile, "sorted", nsteps, segment, filt)
    L2, g2, e2 = _gradient(P, n, tile, "unsorted", nsteps, segment, filt)
    assert (e1, e2) == (0.0, 1.0)
    assert abs(L1 - L2) <= 1e-12 * abs(L2)
    # FP64 sums in another order, amplified over the steps (1e-13 over 100 steps)
    assert np.linalg.norm(g1 - g2) <= 1e-12 * np.linalg.norm(g2)


def test_tile_32_uses_the_unsorted_engine():
    P = setup_weibel(32, 32, epc=8, drift=0.5, uth=0.2, seed=9)
    assert _gradient(P, (32, 32), 32, "sorted", 3, 2)[2] == 1.0


@pytest.mark.parametrize("column,value", [("x", 2.5), ("y", 3.0 + 16), ("z", 2.0), ("z", 0.5), ("x", np.nan)])
def test_bins_refuse_particles_outside(column, value):
    P = setup_weibel(16, 16, epc=8, drift=0.5, uth=0.2, seed=9)
    P[column][5] = value
    for engine in ("sorted", "unsorted"):
        with pytest.raises(PictorError):
            _gradient(P, (16, 16), 8, engine, 2, 1)
