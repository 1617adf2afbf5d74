"""The split form's reverse step recomputes the push that the forward pass ran, so the two have to
round alike: the tile-sorted engine runs the production push, the unsorted engine the push of the
reverse step (push_fwd), and the current of both is exact, so whole runs give the same bits."""
import numpy as np
import pytest

from pictor_amd import Simulation, setup_weibel

from _util import say

pytestmark = pytest.mark.gpu

ARGS = ("q", "x", "y", "z", "u", "v", "w", "flv")


@pytest.mark.parametrize("n,tile", [((8, 8), 8), ((24, 40), 8), ((48, 16), 16), ((32, 32), 32)])
@pytest.mark.parametrize("nsteps,segment,filt", [(2, 1, 0), (12, 5, 0), (30, 30, 1)])
def test_forward_of_both_engines_has_the_same_bits(n, tile, nsteps, segment, filt):
    say(n, tile, nsteps, segment, filt)
    P = setup_weibel(*n, epc=8, drift=0.5, uth=0.2, seed=9)
    L = {}
    for engine in ("sorted", "unsorted"):
        with Simulation(*n, epc=8, form="fp32_split", tile=tile, curr_filter=filt) as sim:
            sim.adjoint_engine(engine)
            L[engine] = sim.adjoint_forward(*[P[k] for k in ARGS], nsteps, segment)
            g = np.stack(sim.adjoint_backward(1.0))
        assert np.isfinite(g).all()
    assert L["sorted"] > 0.0
    assert L["sorted"] == L["unsorted"]
