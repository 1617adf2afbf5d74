"""A particle that a push refuses (outside its tile window) keeps its place beside the error.

A reflecting face deep inside the box throws a particle in front of it several tiles away: the first
push reports it and stores it in its old tile, the second finds it outside that tile's window."""
import numpy as np
import pytest

from pictor_amd import PictorError, Simulation
from pictor_amd._lib import PICTOR_ERR_BOUNDS

from _util import say

pytestmark = pytest.mark.gpu

COLS = ("q", "x", "y", "z", "u", "v", "w")


def _push(sim):
    sim.ResetCurrent()
    sim.MoveDepositPrtl()
    with pytest.raises(PictorError) as e:
        sim.ExchangePrtl()
    assert e.value.args and str(PICTOR_ERR_BOUNDS) in str(e.value)


@pytest.mark.parametrize("n,tile", [((64, 32, 1), 8), ((32, 16, 16), 4)])
def test_refused_particle_keeps_its_place(n, tile):
    ndim = 2 if n[2] == 1 else 3
    say("refused particle", n, "tile", tile)
    wall = 9.5 if ndim == 3 else 13.5           # physical cells from the box's corner
    P = {"q": np.ones(1), "x": np.array([4.25]), "y": np.array([7.5]), "z": np.array([6.75 if ndim == 3 else 1.5]),
         "u": np.array([0.125]), "v": np.array([-0.25]), "w": np.array([0.0625])}
    with Simulation(*n, ndim=ndim, epc=1, form="fp64", tile=tile) as sim:
        sim.SetBC_Prtl("x", wall, "refl", "lower")
        sim.upload_particles(**P, flv=np.ones(1, np.int32))
        _push(sim)
        a = sim.download_particles()
        assert len(a["x"]) == 1 and a["x"][0] > 3.0 + 2 * tile   # thrown more than a tile away
        _push(sim)
        b = sim.download_particles()
    for k in COLS:
        assert np.array_equal(a[k], b[k]), (k, a[k], b[k])
