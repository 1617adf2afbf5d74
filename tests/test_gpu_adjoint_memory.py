"""The adjoint engines' memory: bins that overflow, one context over passes of changing size and
engine (memory kept from one pass must not show in the next), and a card with little room left."""
import numpy as np
import pytest
import torch

from pictor_amd import PictorError, Simulation, setup_weibel
from pictor_amd._lib import PICTOR_ERR_CAPACITY

from _util import say

pytestmark = pytest.mark.gpu

ARGS = ("q", "x", "y", "z", "u", "v", "w", "flv")
# gradients of two engines: FP64 sums in another order, amplified over the steps; the split form
# gives 32-bit gradients of one forward run
CLOSE = {"fp64": 1e-12, "fp32_split": 1e-5}


def _pass(sim, engine, P, nsteps, segment):
    sim.adjoint_engine(engine)
    L = sim.adjoint_forward(*[P[k] for k in ARGS], nsteps, segment)
    g = np.stack(sim.adjoint_backward(1.0))
    return L, g, sim.adjoint_stats()


def _fresh(form, n, engine, P, nsteps, segment, tile=8):
    with Simulation(*n, epc=8, form=form, tile=tile) as sim:
        return _pass(sim, engine, P, nsteps, segment)


def _same(form, a, b):
    say(form, "L", a[0], b[0], "gradients", np.linalg.norm(a[1] - b[1]) / np.linalg.norm(b[1]))
    assert abs(a[0] - b[0]) <= (1e-12 if form == "fp64" else 0.0) * abs(b[0])
    assert np.linalg.norm(a[1] - b[1]) <= CLOSE[form] * np.linalg.norm(b[1])


@pytest.mark.parametrize("form", ["fp64", "fp32_split"])
def test_overflowing_bins_repeat_the_pass(form):
    # two halves of the box run into each other: the tiles between them take 2.4 times their first count
    n = (64, 16)
    P = setup_weibel(*n, epc=8, drift=0.0, uth=0.05, seed=4)
    P["u"] += np.where(P["x"] < 35.0, 0.9, -0.9)
    a = _fresh(form, n, "sorted", P, 28, 7)
    assert a[2]["engine"] == 0.0 and a[2]["relayouts"] >= 1.0
    b = _fresh(form, n, "unsorted", P, 28, 7)
    assert b[2]["engine"] == 1.0
    _same(form, a, b)


def test_bins_that_never_fit():
    # every particle in one tile: what leaves it finds bins sized for empty neighbours.  FP64 goes on
    # with the unsorted engine, the split form reports it; both engines of that context still work
    n = (32, 16)
    P = setup_weibel(*n, epc=64, drift=0.0, uth=0.05, seed=4)
    keep = (P["x"] >= 11.0) & (P["x"] < 19.0) & (P["y"] < 11.0)
    P = {k: np.ascontiguousarray(v[keep]) for k, v in P.items()}
    P["u"] += 0.9
    with Simulation(*n, epc=8, form="fp64", tile=8) as sim:
        a = _pass(sim, "sorted", P, 6, 3)
        assert a[2]["engine"] == 1.0
    _same("fp64", a, _fresh("fp64", n, "unsorted", P, 6, 3))
    Q = setup_weibel(*n, epc=8, drift=0.5, uth=0.05, seed=5)
    with Simulation(*n, epc=8, form="fp32_split", tile=8) as sim:
        with pytest.raises(PictorError) as e:
            _pass(sim, "sorted", P, 6, 3)
        assert str(PICTOR_ERR_CAPACITY) in str(e.value)
        b = _pass(sim, "sorted", Q, 6, 3)
    _same("fp32_split", b, _fresh("fp32_split", n, "sorted", Q, 6, 3))


def test_bins_that_grow_too_little():
    # a dense tile flows into one with a dozen particles: its centre overflows at 12 times that count too
    n = (32, 16)
    dense, thin = setup_weibel(*n, epc=10, drift=0.0, uth=0.05, seed=4), setup_weibel(*n, epc=2, drift=0.0, uth=0.05, seed=5)
    tile = (dense["x"] >= 11.0) & (dense["x"] < 19.0) & (dense["y"] < 11.0)
    some = np.random.default_rng(3).random(len(thin["x"])) < 0.06
    P = {k: np.concatenate([dense[k][tile], thin[k][some]]) for k in dense}
    P["u"] += 0.3
    a = _fresh("fp64", n, "sorted", P, 30, 7)
    assert a[2]["engine"] == 1.0
    _same("fp64", a, _fresh("fp64", n, "unsorted", P, 30, 7))


@pytest.mark.parametrize("form", ["fp64", "fp32_split"])
def test_passes_of_one_context(form):
    n = (48, 40)
    full = setup_weibel(*n, epc=16, drift=0.5, uth=0.2, seed=6)
    rng = np.random.default_rng(2)
    order = rng.permutation(len(full["x"]))

    def load(count):
        return {k: np.ascontiguousarray(v[order[:count]]) for k, v in full.items()}
    small, most, some = load(901), load(len(order)), load(len(order) // 3)
    passes = [("sorted", small, 4, 2), ("sorted", most, 9, 4), ("sorted", small, 7, 1), ("unsorted", most, 5, 5),
              ("sorted", some, 12, 3), ("unsorted", small, 3, 2), ("sorted", most, 9, 4)]
    with Simulation(*n, epc=8, form=form, tile=8) as sim:
        for p in passes:
            a = _pass(sim, *p)
            _same(form, a, _fresh(form, n, *p))


# ---- little room on the card ----

N, COUNT, STEPS = (512, 512), 40 << 20, (2, 1)     # 630 MB an FP64 array of the bins


def _random_load():
    """A quiet plasma of COUNT particles as device arrays."""
    g = torch.Generator(device="cuda").manual_seed(7)
    real = dict(device="cuda", dtype=torch.float64)
    at = [torch.rand(COUNT // 2, generator=g, **real) for _ in range(2)]
    P = {"q": torch.ones(COUNT, **real), "x": (3.0 + N[0] * at[0]).repeat(2), "y": (3.0 + N[1] * at[1]).repeat(2),
         "z": torch.full((COUNT,), 1.5, **real)}
    P["q"][COUNT // 2:] = -1.0
    for k in "uvw":
        P[k] = 0.1 * torch.randn(COUNT, generator=g, **real)
    P["flv"] = torch.ones(COUNT, device="cuda", dtype=torch.int32)
    P["flv"][COUNT // 2:] = 2
    return P


def _device_pass(sim, P, out, nsteps, segment, engine="sorted"):
    torch.cuda.synchronize()
    sim.adjoint_engine(engine)
    L = sim.adjoint_forward_device(P["x"].numel(), *[P[k].data_ptr() for k in ARGS], nsteps, segment)
    sim.adjoint_backward_device(*[t.data_ptr() for t in out])
    torch.cuda.synchronize()
    return L, sim.adjoint_stats()


class _Card:
    """The load, the gradient of the unsorted engine, the need of a sorted pass, and the rest of the card held."""

    def __init__(self):
        self.P = _random_load()
        self.want, self.out = ([torch.empty(COUNT, device="cuda", dtype=torch.float64) for _ in range(3)] for _ in range(2))
        with Simulation(*N, epc=8, form="fp64", tile=16) as sim:
            self.need = _device_pass(sim, self.P, self.out, *STEPS)[1]["device_bytes"]
            self.L, stats = _device_pass(sim, self.P, self.want, *STEPS, engine="unsorted")
        self.least = stats["device_bytes"]
        third = [slice(0, COUNT // 3), slice(COUNT // 2, COUNT // 2 + COUNT // 3)]
        self.part = {k: torch.cat([v[a] for a in third]) for k, v in self.P.items()}
        self.part_out = [[torch.empty_like(self.part["x"]) for _ in range(3)] for _ in range(2)]
        self.most = int(1.3 * self.need)
        torch.cuda.empty_cache()
        free = torch.cuda.mem_get_info()[0]
        say("sorted pass: %.2f GiB, unsorted: %.2f; %.2f of the card free" % tuple(b / 2**30 for b in (self.need, self.least, free)))
        self.held = torch.empty(free - self.most, dtype=torch.uint8, device="cuda")

    def leave(self, room):
        """Holds what is free beyond `room` bytes."""
        return torch.empty(max(1, torch.cuda.mem_get_info()[0] - int(room)), dtype=torch.uint8, device="cuda")

    def right(self, L):
        assert abs(L - self.L) <= 1e-12 * abs(self.L)
        for a, b in zip(self.out, self.want):
            for p in range(0, COUNT, 4 << 20):     # in pieces: the card is full
                d = (a[p:p + (4 << 20)] - b[p:p + (4 << 20)]).norm()
                assert float(d) <= 1e-11 * float(b[p:p + (4 << 20)].norm())


@pytest.fixture(scope="module")
def card():
    c = _Card()
    yield c
    del c.held, c.P, c.part, c.want, c.out, c.part_out
    torch.cuda.empty_cache()


@pytest.mark.parametrize("room", [0.7, 1.07, 1.2])
def test_pass_with_little_room(card, room):
    # below the sorted engine's need the unsorted one runs; above it no room may be lost
    with Simulation(*N, epc=8, form="fp64", tile=16) as sim:
        assert room * card.need > card.least
        hold = card.leave(room * card.need + (192 << 20))     # and the runtime's own
        for _ in range(2):
            L, stats = _device_pass(sim, card.P, card.out, *STEPS)
            say("room", room, "engine", stats["engine"], "free", torch.cuda.mem_get_info()[0] >> 20, "MiB")
            assert stats["engine"] == (1.0 if room < 1.0 else 0.0)
        del hold
        torch.cuda.empty_cache()
        card.right(L)


def test_kept_memory_makes_room(card):
    # a pass of two thirds of the particles in more states, then the full one, then the first again:
    # the memory of two of them doesn't fit
    with Simulation(*N, epc=8, form="fp64", tile=16) as sim:
        hold = card.leave(1.12 * card.need)
        La, stats = _device_pass(sim, card.part, card.part_out[0], 4, 2)
        assert stats["engine"] == 0.0 and stats["device_bytes"] > 0.6 * card.need
        L, stats = _device_pass(sim, card.P, card.out, *STEPS)
        assert stats["engine"] == 0.0
        Lb, stats = _device_pass(sim, card.part, card.part_out[1], 4, 2)
        assert stats["engine"] == 0.0
        del hold
        torch.cuda.empty_cache()
        card.right(L)
        assert Lb == pytest.approx(La, rel=1e-12)
        for a, b in zip(*card.part_out):
            assert float((a - b).norm()) <= 1e-11 * float(b.norm())


def test_fields_count_as_used(card):
    # a large grid with few particles: the field checkpoints that the pass already holds are no room for
    # its bins, and the unsorted engine runs where those do not fit
    n, count = (2048, 2048), 100000
    P = {k: v[:: COUNT // count][:count].contiguous() for k, v in card.P.items()}
    out = [[torch.empty_like(P["x"]) for _ in range(3)] for _ in range(2)]
    with Simulation(*n, epc=8, form="fp64", tile=16) as sim:
        L, stats = _device_pass(sim, P, out[0], 8, 1)
        assert stats["engine"] == 0.0
    with Simulation(*n, epc=8, form="fp64", tile=16) as sim:
        hold = card.leave(0.96 * stats["device_bytes"])
        Lb, least = _device_pass(sim, P, out[1], 8, 1)
        say("sorted %.2f GiB, unsorted %.2f" % (stats["device_bytes"] / 2**30, least["device_bytes"] / 2**30))
        assert least["engine"] == 1.0
        del hold
        torch.cuda.empty_cache()
    assert Lb == pytest.approx(L, rel=1e-12)
    for a, b in zip(*out):
        assert float((a - b).norm()) <= 1e-11 * float(b.norm())
