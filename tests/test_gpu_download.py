"""Downloads through the pinned ring: results on both sides of the size from which host threads
copy (6 MiB: 288 x 288 and 288 x 296), arrays of less and more than one 1 MiB piece, more pieces than the ring holds,
arrays left out, and several contexts from several threads."""
import ctypes
import threading

import numpy as np
import pytest
import torch

from pictor_amd import Simulation, setup_weibel
from pictor_amd._lib import check, lib

from _util import say

pytestmark = pytest.mark.gpu

F = ("Ex", "Ey", "Ez", "Bx", "By", "Bz")


def _fields(sim, seed):
    rng = np.random.default_rng(seed)
    return [np.asfortranarray(rng.standard_normal(sim.shape)) for _ in F]


def _expect(form, name, f):
    if form == "fp64":
        return f
    hi = f.astype(np.float32)
    if name[0] == "B":
        return hi.astype(np.float64)
    return hi.astype(np.float64) + (f - hi.astype(np.float64)).astype(np.float32).astype(np.float64)


@pytest.mark.parametrize("form", ["fp32_split", "fp64"])
@pytest.mark.parametrize("n", [(8, 8), (160, 160), (168, 160), (288, 288), (288, 296), (368, 360), (1024, 704)])
def test_fields(form, n):
    say(form, n)
    with Simulation(*n, form=form) as sim:
        src = _fields(sim, 3)
        sim.upload_fields(*src)
        for _ in range(2):
            out = sim.download_fields()
            for name, f in zip(F, src):
                assert np.array_equal(out[name], _expect(form, name, f)), name
            assert all(not out[j].any() for j in ("Jx", "Jy", "Jz"))
        # only Ey and Bz
        ey, bz = (np.full(sim.shape, np.nan, order="F") for _ in range(2))
        ptr = [None] * 9
        ptr[1], ptr[5] = (a.ctypes.data_as(ctypes.POINTER(ctypes.c_double)) for a in (ey, bz))
        check(lib().pictor_download_fields(sim._ctx, *ptr))
        assert np.array_equal(ey, out["Ey"]) and np.array_equal(bz, out["Bz"])


@pytest.mark.parametrize("form", ["fp32_split", "fp64"])
@pytest.mark.parametrize("n,epc", [((16, 16), 2), ((128, 128), 4), ((256, 192), 8)])
def test_particles(form, n, epc):
    say(form, n, epc)
    P = setup_weibel(*n, epc=epc, drift=0.5, uth=0.2, seed=5)
    m = len(P["x"])
    with Simulation(*n, epc=epc, form=form) as sim:
        sim.upload_particles(**P, tag=np.arange(m, dtype=np.int32))
        out = sim.download_particles(with_tile=True, with_tag=True)
    o = np.argsort(out["tag"])
    assert np.array_equal(out["tag"][o], np.arange(m))
    assert np.array_equal(out["flv"][o], P["flv"])
    for k in ("u", "v", "w"):
        want = P[k] if form == "fp64" else P[k].astype(np.float32).astype(np.float64)
        assert np.array_equal(out[k][o], want), k
    # split positions: a 24-bit offset in the cell
    for k in ("x", "y"):
        assert np.abs(out[k][o] - P[k]).max() <= (0.0 if form == "fp64" else 2.0 ** -24), k
    assert out["tile"].min() >= 0 and out["tile"].max() > 0


@pytest.mark.parametrize("form", ["fp32_split", "fp64"])
def test_pinned_destination(form):
    # the caller's pinned arrays take the results without the ring, beside pageable ones
    say(form)
    with Simulation(168, 160, form=form) as sim:
        sim.upload_fields(*_fields(sim, 4))
        want = sim.download_fields()
        n = int(np.prod(sim.shape))
        pin = [torch.full((n,), float("nan"), dtype=torch.float64, pin_memory=True) for _ in range(4)]
        page = np.full(sim.shape, np.nan, order="F")
        dp = ctypes.POINTER(ctypes.c_double)
        ptr = [ctypes.cast(t.data_ptr(), dp) for t in pin] + [page.ctypes.data_as(dp)] + [None] * 4
        check(lib().pictor_download_fields(sim._ctx, *ptr))
        for name, t in zip(F, pin):
            assert np.array_equal(t.numpy().reshape(sim.shape, order="F"), want[name]), name
        assert np.array_equal(page, want["By"])


def test_threads():
    """Contexts share nothing: four threads, each with its own, download at once."""
    bad = []

    def work(seed):
        with Simulation(368, 360, form="fp64") as sim:
            src = _fields(sim, seed)
            sim.upload_fields(*src)
            for _ in range(3):
                out = sim.download_fields()
                bad.extend((seed, k) for k, f in zip(F, src) if not np.array_equal(out[k], f))

    t = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    [x.start() for x in t]
    [x.join() for x in t]
    assert not bad
