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


@pytest.mark.parametrize("n", [(8, 8), (8, 24), (40, 8), (24, 16)])
@pytest.mark.parametrize("filt", [0, 1])
def test_gradient_is_the_difference_quotient(n, filt):
    # the field part of the reverse step reads across the boundary from both sides at the smallest
    # boxes; central difference along a random direction of all momenta: the quotient carries
    # rounding of about 1e-16 / h of L and h^2 of its third derivative.  The zigzag current jumps where
    # a particle's cell crossing changes between the two ends: about 2 h c particles steps axes of
    # them, 0.07 at h = 1e-6 and 6144 particles (two of nine boxes met one) and 0.0007 at 1e-8, where
    # the rounding is 1e-7 of the quotient
    say(n, filt)
    P = setup_weibel(*n, epc=8, drift=0.5, uth=0.2, seed=11)
    rng = np.random.default_rng(6)
    d = [rng.standard_normal(len(P["x"])) for _ in range(3)]
    h, L = 1e-8, []
    g = _gradient(P, n, 8, "sorted", 6, 4, filt)[1] / 2.0
    for sign in (1.0, -1.0):
        Q = {k: v + sign * h * d["uvw".index(k)] if k in "uvw" else v for k, v in P.items()}
        L.append(_gradient(Q, n, 8, "sorted", 6, 4, filt)[0])
    want = sum((a * b).sum() for a, b in zip(g, d))
    scale = np.linalg.norm(g) * np.sqrt(sum((a * a).sum() for a in d) / g.size)
    assert abs((L[0] - L[1]) / (2 * h) - want) <= 1e-5 * max(abs(want), scale)


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
