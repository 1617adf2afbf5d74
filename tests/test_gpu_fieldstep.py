"""Runs of fused steps (several enqueued together, the field work of a step in one launch) against
the phase calls: sizes around the field kernel's tiles, every scheme, runs longer than the number
of steps enqueued at once, and bins that overflow in the middle of a run."""
import numpy as np
import pytest

from pictor_amd import Simulation, setup_weibel

from _util import say

pytestmark = pytest.mark.gpu

F = ("Ex", "Ey", "Ez", "Bx", "By", "Bz", "Jx", "Jy", "Jz")


def _run(form, n, ndim, fdtd, filt, cap, calls, phases):
    P = setup_weibel(*n, ndim=ndim, epc=4, drift=0.5, uth=0.2, seed=5)
    rng = np.random.default_rng(1)
    with Simulation(*n, ndim=ndim, epc=4, form=form, fdtd=fdtd, curr_filter=filt, capacity_factor=cap) as sim:
        F0 = []
        for _ in range(6):
            f = np.zeros(sim.shape, order="F")
            inner = tuple(slice(2, -3) if m > 1 else slice(None) for m in sim.shape)
            f[inner] = 0.02 * rng.standard_normal(f[inner].shape)
            F0.append(f)
        sim.upload_fields(*F0)
        sim.SendRecvFlds("E")
        sim.SendRecvFlds("B")
        sim.upload_particles(**P)
        for k in calls:
            if phases:
                for _ in range(k):
                    sim.step_phases()
            else:
                sim.step(k)
        out = sim.download_fields()
        count = sim.particle_count()
        stats = sim.relayout_stats()
        timers = [sim.timer(w)[1] for w in ("push", "fields", "step")]
        diag = sim.diagnostics()
    return out, count, stats, timers, diag, len(P["x"])


@pytest.mark.parametrize("form", ["fp32_split", "fp64"])
@pytest.mark.parametrize("ndim,n", [(2, (8, 8, 1)), (2, (72, 24, 1)), (2, (64, 8, 1)), (2, (136, 40, 1)),
                                    (3, (8, 8, 8)), (3, (72, 12, 8)), (3, (16, 20, 12))])
@pytest.mark.parametrize("fdtd,filt", [("yee", 0), ("lehe", 0), ("yee", 1), ("lehe", 3)])
def test_fused_run_equals_phases(form, ndim, n, fdtd, filt):
    say(form, n, fdtd, filt)
    a, na, _, timers, da, np_ = _run(form, n, ndim, fdtd, filt, 0.0, (1, 5), False)
    b, nb, _, _, db, _ = _run(form, n, ndim, fdtd, filt, 0.0, (1, 5), True)
    assert na == nb == np_
    assert timers == [6, 6, 6]
    for k in F:
        if form == "fp32_split":
            assert np.array_equal(a[k], b[k]), k
        else:
            # FP64 current: the order of the LDS and global adds varies between runs
            assert np.abs(a[k] - b[k]).max() <= 1e-12 * max(np.abs(b[k]).max(), 1e-300), k
    assert abs(da["B_energy"] - db["B_energy"]) <= 1e-11 * abs(db["B_energy"])


@pytest.mark.parametrize("form", ["fp32_split", "fp64"])
@pytest.mark.parametrize("ndim,n,fdtd", [(2, (48, 24, 1), "yee"), (3, (16, 16, 16), "yee"), (3, (16, 16, 16), "lehe")])
def test_overflow_inside_a_run(form, ndim, n, fdtd):
    """Small bins overflow every few steps: the steps enqueued behind the overflow must wait for
    the re-layout, and the run must end as with one step per call (37 > the steps of one run)."""
    a, na, sa, ta, _, np_ = _run(form, n, ndim, fdtd, 0, 0.6, (37,), False)
    b, nb, sb, _, _, _ = _run(form, n, ndim, fdtd, 0, 0.6, (1,) * 37, False)
    c, nc, sc, _, _, _ = _run(form, n, ndim, fdtd, 0, 4.0, (37,), False)
    say(sa, sb, sc)
    assert na == nb == nc == np_
    assert sa[0] > 0 and sb[0] > 0
    assert ta == [37, 37, 37]
    for k in F:
        if form == "fp32_split":
            assert np.array_equal(a[k], b[k]) and np.array_equal(a[k], c[k]), k
        else:
            assert np.abs(a[k] - b[k]).max() <= 1e-9 * np.abs(b[k]).max(), k


def test_step_without_room_for_second_buffers():
    # a card too full for the second field buffers: the step runs in place, with the same bits
    import torch

    cases = [((1024, 1024, 1), 2, dict()), ((1024, 768, 1), 2, dict(fdtd="lehe", curr_filter=1)), ((96, 96, 96), 3, dict())]

    def start(n, ndim, more):
        sim = Simulation(*n, ndim=ndim, epc=2, form="fp32_split", **more)
        sim.upload_particles(**setup_weibel(*n, ndim=ndim, epc=2, drift=0.5, uth=0.2, seed=8))
        return sim

    want = []
    for c in cases:
        with start(*c) as sim:
            lean = sim.memory_bytes()
            sim.step(5)
            want.append(sim.download_fields())
            assert sim.memory_bytes() > lean
    sims = [start(*c) for c in cases]
    torch.cuda.empty_cache()
    torch.cuda.synchronize()
    held = [torch.empty(torch.cuda.mem_get_info()[0] - (64 << 20), dtype=torch.uint8, device="cuda")]
    try:
        while True:     # more than the runtime says is there
            held.append(torch.empty(22 << 20, dtype=torch.uint8, device="cuda"))
    except torch.OutOfMemoryError:
        held.pop()
        torch.cuda.empty_cache()
    lean = [sim.memory_bytes() for sim in sims]
    for sim in sims:
        sim.step(5)
    assert [sim.memory_bytes() for sim in sims] == lean
    del held
    torch.cuda.empty_cache()
    for sim, F in zip(sims, want):
        G = sim.download_fields()
        sim.close()
        for k in F:
            assert np.array_equal(G[k], F[k]), k
