"""The azimuthal-mode (m = 0, 1) cylinder on the GPU vs its oracle, through the C ABI.

Bars:
  * field updates, axis parity fills, z halos and wall: bit for bit;
  * the plasma loader: the same particles bit for bit (counter-based);
  * one push from identical state: positions and momenta within 1e-13
    relative (device vs host cos, sin, atan2), current within 1e-12 of its
    maximum (atomic order); 20 steps: fields and particles within 1e-9;
  * the moving window: 12 steps with shifts and injection as the oracle's;
  * the GPU run keeps the modal Gauss law node by node (1e-12);
  * a laser pulse in vacuum keeps its energy and moves at the group speed;
    a test electron in a weak pulse quivers with gamma beta_x = a0 (5 %);
  * the Lehe B update: bit for bit with the oracle; a pulse at k0 = 1 rad per cell
    moves at the Lehe group speed (2 %), 15 % faster than the Yee one;
  * a Courant number above the limit of the m = 1 terms next to the axis (and
    above the Lehe rule) is rejected;
  * the split form: the loader gives the FP64 loader's particles rounded to the
    split record; one push from the same (rounded) state matches the oracle to
    4e-6 (positions, momenta) and 2e-5 (J_r, J_z; 1e-4 for J_theta); 20 steps stay within 1e-5 of
    the FP64 form; runs are bitwise deterministic, the moving window included;
    the modal Gauss law holds to 1e-6; a contribution beyond the fixed-point
    range is an error;
  * a window run long enough to compact the particle arrays keeps the live
    particles in order: FP64 equal to the oracle (1e-9), split within 2e-4.
"""
import math

import numpy as np
import pytest

from oracle.pyoracle import CylModalOracle
from pictor_amd import Simulation
from tests._util import say

pytestmark = pytest.mark.gpu

FIELDS = ("Ex", "Ey", "Ez", "Bx", "By", "Bz")


def _pair(nr, nz, dr=1.0, c=0.3, epc=4, cap=4096, fdtd="yee"):
    say(f"[case] cylm nr={nr} nz={nz} dr={dr} c={c} fdtd={fdtd}")
    o = CylModalOracle(nr, nz, dr=dr, c=c, c_ompe=10.0, epc=epc, cap=cap, fdtd=1 if fdtd == "lehe" else 0)
    sim = Simulation(nr, 2, nz, ndim=3, epc=epc, c=c, c_ompe=10.0, form="fp64", geometry="cyl_modal", dr=dr,
                     mi_me=1e30, fdtd=fdtd)
    return o, sim


def _smooth_fields(o, rng, amp=1e-3):
    mx, _, mz = o.shape
    i = np.arange(mx)[:, None] + 1.0
    k = np.arange(mz)[None, :] + 1.0
    F = {}
    for n in FIELDS:
        a = np.zeros(o.shape, order="F")
        for s in range(3):
            p, q, ph = rng.normal(size=3)
            a[:, s, :] = amp * np.cos(0.3 * p * i + 0.2 * q * k + ph) * np.exp(-i / (0.7 * mx))
        F[n] = a
    return F


def _upload_fields(o, sim, F):
    o.set_fields(**F)
    sim.upload_fields(*[np.asfortranarray(F[n]) for n in FIELDS])


@pytest.mark.parametrize("fdtd", ["yee", "lehe"])
def test_field_updates_bitwise(fdtd):
    o, sim = _pair(16, 20, dr=2.0, c=0.5, fdtd=fdtd)
    with sim:
        _upload_fields(o, sim, _smooth_fields(o, np.random.default_rng(1)))
        for _ in range(3):
            sim.UpdateBfieldHalf(); o.b_half()
            sim.UpdateEfield(); o.e_phase(curl=True)
        G = sim.download_fields()
    for n in FIELDS:
        assert np.array_equal(G[n], o.F[n]), f"{n}: max diff {np.abs(G[n] - o.F[n]).max()}"


def test_plasma_loader_bitwise():
    o, sim = _pair(24, 16, dr=1.5, c=0.3)
    with sim:
        sim.cyl_plasma(12, 5, 9, 8, seed=77)
        A = sim.download_particles()
    B = o.load_plasma(12, 5, 9, 8, seed=77)
    assert len(A["x"]) == len(B["x"]) == 12 * 9 * 8
    for k in ("q", "x", "y", "z", "u", "v", "w", "flv"):
        assert np.array_equal(A[k], B[k]), k


def _thermal(o, rng, spread=0.1):
    P = o.particles(live_only=False)
    n = len(P["x"])
    for k in "uvw":
        P[k] = rng.normal(0.0, spread, n)
    return P


def test_push_and_steps_match_oracle():
    o, sim = _pair(24, 24, dr=2.0, c=0.5, epc=4)
    rng = np.random.default_rng(5)
    o.load_plasma(14, 3, 24, 8, seed=5)
    P = _thermal(o, rng)
    o.load_particles(P["q"], P["x"], P["y"], P["z"], P["u"], P["v"], P["w"], P["flv"])
    with sim:
        _upload_fields(o, sim, _smooth_fields(o, rng, amp=5e-3))
        sim.upload_particles(**P)
        sim.ResetCurrent(); o.reset_current()
        sim.MoveDepositPrtl(); sim.ExchangePrtl(); o.move_deposit()
        A, B = sim.download_particles(), o.particles()
        for k in ("x", "y", "z", "u", "v", "w"):
            d = np.abs(A[k] - B[k]) / np.maximum(np.abs(B[k]), 1.0)
            assert d.max() <= 1e-13, (k, d.max())
        G = sim.download_fields()
        for k in ("Jx", "Jy", "Jz"):
            scale = np.abs(o.F[k]).max()
            assert scale > 0 and np.abs(G[k] - o.F[k]).max() <= 1e-12 * scale, k
        # 20 full steps from the same state
        _upload_fields(o, sim, _smooth_fields(o, np.random.default_rng(6), amp=5e-3))
        sim.upload_particles(**B)
        sim.step(20)
        o.run(20)
        G = sim.download_fields()
        for k in FIELDS:
            scale = np.abs(o.F[k]).max()
            d = np.abs(G[k] - o.F[k]).max() / scale
            say(f"{k}: max diff / max {d:.2e}")
            assert d <= 1e-9, k
        A, B = sim.download_particles(), o.particles()
        for k in ("x", "y", "z", "u", "v", "w"):
            assert np.abs(A[k] - B[k]).max() <= 1e-9 * max(np.abs(B[k]).max(), 1.0), k


def test_moving_window_matches_oracle():
    o, sim = _pair(20, 24, dr=2.0, c=0.45, epc=4, cap=20000)
    rng = np.random.default_rng(9)
    o.load_plasma(10, 3, 24, 4, seed=13, cap=20000)
    P = _thermal(o, rng, 0.05)
    o.load_particles(P["q"], P["x"], P["y"], P["z"], P["u"], P["v"], P["w"], P["flv"], cap=20000)
    with sim:
        sim.upload_particles(**P)
        sim.moving_window(True, nr_plasma=10, ppc=4, seed=13)
        o.set_zopen(True)   # the window box has open z ends, as on the GPU
        nsteps, shifts = 12, 0
        sim.step(nsteps)
        for t in range(1, nsteps + 1):
            o.step()
            while t * 0.45 >= shifts + 1:
                shifts += 1
                o.shift(10, 4, 13, shifts)
        G = sim.download_fields()
        A, B = sim.download_particles(), o.particles(live_only=False)
    say(f"window shifts {shifts}")
    assert shifts == 5
    assert len(A["x"]) == len(B["x"])
    assert np.array_equal(A["flv"], B["flv"])
    live = B["flv"] != 0
    for k in ("x", "y", "z", "u", "v", "w"):
        assert np.abs(A[k][live] - B[k][live]).max() <= 1e-9 * max(np.abs(B[k][live]).max(), 1.0), k
    for k in FIELDS:
        scale = np.abs(o.F[k]).max()
        assert scale > 0 and np.abs(G[k] - o.F[k]).max() <= 1e-9 * scale, k


def test_gpu_run_keeps_modal_gauss_law():
    o, sim = _pair(32, 40, dr=2.0, c=0.5, epc=4, cap=60000)
    rng = np.random.default_rng(2)
    o.load_plasma(20, 3, 40, 8, seed=2, cap=60000)
    P = _thermal(o, rng, 0.1)
    o.load_particles(P["q"], P["x"], P["y"], P["z"], P["u"], P["v"], P["w"], P["flv"], cap=60000)
    G0 = o.gauss()
    with sim:
        sim.upload_particles(**P)
        sim.step(40)
        F = sim.download_fields()
        A = sim.download_particles()
    o.set_fields(**{k: F[k] for k in FIELDS})
    o.load_particles(A["q"], A["x"], A["y"], A["z"], A["u"], A["v"], A["w"], A["flv"], cap=60000)
    G1 = o.gauss()
    for s in range(3):
        d = np.abs(G1 - G0)[:, s, :].max() / np.abs(G0[:, s, :]).max()
        say(f"slot {s}: Gauss change / max {d:.2e}")
        assert d <= 1e-12, s


def _laser_run(a0, with_electron, steps, fdtd="yee", omega0=10.0):
    nr, nz, dr, c = 48, 384, 4.0, 0.8
    sim = Simulation(nr, 2, nz, ndim=3, epc=1, c=c, c_ompe=20.0, form="fp64", geometry="cyl_modal", dr=dr, mi_me=1e30,
                     fdtd=fdtd)
    # omega0 = 10 omega_p: k0 = 0.5 rad per axial cell; c tau = 40 cells, w0 = 120 cells
    zc = 110.0
    sim.cyl_laser(a0, omega0, 2.0, 6.0, zc)
    if with_electron:
        P = dict(q=np.array([-1e-9]), x=np.array([3.6]), y=np.array([0.0]), z=np.array([250.0]),
                 u=np.zeros(1), v=np.zeros(1), w=np.zeros(1), flv=np.array([2], dtype=np.int32))
        sim.upload_particles(**P)
    return sim, zc


def test_laser_in_vacuum_keeps_energy_and_moves_forward():
    say("[case] laser in vacuum")
    sim, zc = _laser_run(0.1, False, 0)
    with sim:
        e0 = sim.diagnostics()
        F0 = sim.download_fields()
        sim.step(150)
        e1 = sim.diagnostics()
        F1 = sim.download_fields()
    w0 = e0["B_energy"] + e0["E_energy"]
    w1 = e1["B_energy"] + e1["E_energy"]
    say(f"field energy {w0:.6e} -> {w1:.6e}")
    # a purely forward pulse from the first step (B set half a step behind E): no
    # backward wave, E and B energies stay equal
    assert w0 > 0 and abs(w1 - w0) <= 1e-3 * w0
    assert abs(e1["B_energy"] - e1["E_energy"]) <= 2e-3 * w1
    # envelope centre on the axis row of E_r (m = 1 cos), then the distance moved
    moved = _centre(F1) - _centre(F0)
    # Yee group speed along z for k0 = 0.5 at c = 0.8: d omega/dk of sin(w/2) = c sin(k/2)
    vg = 0.8 * math.cos(0.25) / math.sqrt(1.0 - (0.8 * math.sin(0.25)) ** 2)
    say(f"moved {moved:.2f} cells, group speed x 150 = {150 * vg:.2f}")
    assert abs(moved - 150 * vg) <= 0.03 * 150 * vg


def _centre(F):
    a = F["Ex"][3, 1, :] ** 2 + F["Bx"][3, 2, :] ** 2
    k = np.arange(len(a)) + 1.0
    return float((a * k).sum() / a.sum())


def test_lehe_pulse_moves_at_the_lehe_group_speed():
    # k0 = 1 rad per cell (omega0 = 20 omega_p at c/omega_p = 20 cells, c = 0.8): the Lehe
    # dispersion sin^2(w/2) = c^2 (sin^2(k/2) - 4 d_z sin^4(k/2)) gives the group speed
    # 0.872, the Yee one 0.760
    say("[case] Lehe pulse group speed")
    c = 0.8
    dz = 0.25 * (1.0 - (math.sin(0.5 * math.pi * c) / c) ** 2)

    def w(k, lehe):
        s2 = math.sin(0.5 * k) ** 2
        return 2.0 * math.asin(c * math.sqrt(s2 - (4.0 * dz * s2 * s2 if lehe else 0.0)))
    vg = {f: (w(1.0 + 1e-6, f == "lehe") - w(1.0 - 1e-6, f == "lehe")) / 2e-6 for f in ("yee", "lehe")}
    for fdtd in ("yee", "lehe"):
        sim, _ = _laser_run(0.1, False, 0, fdtd=fdtd, omega0=20.0)
        with sim:
            sim.step(10)
            F0 = sim.download_fields()
            sim.step(120)
            F1 = sim.download_fields()
        moved = _centre(F1) - _centre(F0)
        say(f"{fdtd}: moved {moved:.2f} cells, group speed x 120 = {120 * vg[fdtd]:.2f}")
        assert abs(moved - 120 * vg[fdtd]) <= 0.02 * 120 * vg[fdtd], fdtd


def test_electron_quivers_with_a0():
    say("[case] electron in a weak pulse")
    a0 = 0.02
    sim, _ = _laser_run(a0, True, 0)
    umax = 0.0
    with sim:
        for _ in range(60):
            sim.step(5)
            P = sim.download_particles()
            live = P["flv"] != 0
            ux = P["u"][live] * np.cos(P["y"][live]) - P["v"][live] * np.sin(P["y"][live])
            umax = max(umax, float(np.abs(ux).max()))
    say(f"max |gamma beta_x| {umax:.5f} for a0 {a0}")
    assert abs(umax - a0) <= 0.05 * a0


@pytest.mark.parametrize("dr,c,fdtd", [(1.0, 0.41, "yee"), (4.0, 0.88, "yee"), (4.0, 0.85, "lehe")])
def test_courant_above_the_axis_limit_is_rejected(dr, c, fdtd):
    with pytest.raises(RuntimeError):
        Simulation(16, 2, 16, ndim=3, epc=1, c=c, form="fp64", geometry="cyl_modal", dr=dr, fdtd=fdtd)


def test_courant_below_the_lehe_rule_is_accepted():
    # sin^2(0.42 pi) + 1.25 * 0.84^2 / 16 = 0.994 < 1; Yee accepts 0.85 as well
    Simulation(16, 2, 16, ndim=3, epc=1, c=0.84, form="fp64", geometry="cyl_modal", dr=4.0, fdtd="lehe").close()
    Simulation(16, 2, 16, ndim=3, epc=1, c=0.85, form="fp64", geometry="cyl_modal", dr=4.0, fdtd="yee").close()


# ---- the split form: (cell, FP32 offset) positions, theta in 2^-32 turns, FP32 push,
# fixed-point current (2^-36 counts summed exactly in FP64) ----

TURN = 2.0 * math.pi / 2.0 ** 32


def _split_sim(nr, nz, dr, c, epc=4, fdtd="yee"):
    return Simulation(nr, 2, nz, ndim=3, epc=epc, c=c, c_ompe=10.0, form="fp32_split", geometry="cyl_modal", dr=dr,
                      mi_me=1e30, fdtd=fdtd)


def test_split_loader_is_the_fp64_loader_rounded():
    say("[case] split loader")
    o = CylModalOracle(24, 16, dr=1.5, c=0.3, c_ompe=10.0, epc=5, cap=4096)
    B = o.load_plasma(12, 5, 9, 8, seed=77)
    with _split_sim(24, 16, 1.5, 0.3, epc=5) as sim:
        sim.cyl_plasma(12, 5, 9, 8, seed=77)
        A = sim.download_particles()
    assert np.array_equal(A["flv"], B["flv"])
    for k in ("x", "z"):   # the cell exact, the offset rounded to FP32
        assert np.array_equal(np.floor(A[k]), np.floor(B[k])), k
        assert np.abs(A[k] - B[k]).max() <= 2.0 ** -24, k
    assert np.abs(A["y"] - B["y"]).max() <= TURN
    np.testing.assert_allclose(A["q"], B["q"], rtol=2.0 ** -24, atol=0)


def _split_state(o, rng, spread=0.1):
    """a thermal plasma in the oracle, rounded to what the split record holds"""
    P = _thermal(o, rng, spread)
    P["u"], P["v"], P["w"] = (P[k].astype(np.float32).astype(np.float64) for k in "uvw")
    P["q"] = P["q"].astype(np.float32).astype(np.float64)
    for k in ("x", "z"):
        cell = np.floor(P[k])
        P[k] = cell + (P[k] - cell).astype(np.float32).astype(np.float64)
    P["y"] = np.round(P["y"] / TURN) % 2.0 ** 32 * TURN
    return P


def test_split_push_matches_oracle():
    o = CylModalOracle(24, 24, dr=2.0, c=0.5, c_ompe=10.0, epc=4, cap=8192)
    rng = np.random.default_rng(15)
    o.load_plasma(14, 3, 24, 8, seed=5, cap=8192)
    P = _split_state(o, rng)
    F = _smooth_fields(o, rng, amp=5e-3)
    with _split_sim(24, 24, 2.0, 0.5) as sim:
        sim.upload_particles(**P)
        A0 = sim.download_particles()
        for k in ("x", "y", "z", "u", "v", "w", "q"):   # the upload holds the rounded state exactly
            assert np.array_equal(A0[k], P[k]), k
        o.load_particles(P["q"], P["x"], P["y"], P["z"], P["u"], P["v"], P["w"], P["flv"], cap=8192)
        o.set_fields(**F)
        sim.upload_fields(*[np.asfortranarray(F[n]) for n in FIELDS])
        sim.ResetCurrent(); o.reset_current()
        sim.MoveDepositPrtl(); sim.ExchangePrtl(); o.move_deposit()
        A, B = sim.download_particles(), o.particles()
        G = sim.download_fields()
    assert len(A["x"]) == len(B["x"])
    err = {}
    for k in ("x", "z"):
        err[k] = np.abs(A[k] - B[k]).max()
    err["y"] = np.abs((A["y"] - B["y"] + math.pi) % (2 * math.pi) - math.pi).max()
    for k in "uvw":
        err[k] = np.abs(A[k] - B[k]).max() / np.abs(B[k]).max()
    for k in ("Jx", "Jy", "Jz"):
        err[k] = np.abs(G[k] - o.F[k]).max() / np.abs(o.F[k]).max()
    say("split vs oracle after one push: " + ", ".join(f"{k} {v:.2e}" for k, v in err.items()))
    for k in ("x", "z"):
        assert err[k] <= 4e-6, k          # cells: FP32 offsets and displacement
    assert err["y"] <= 4e-6               # radians
    for k in "uvw":
        assert err[k] <= 4e-6, k
    for k in ("Jx", "Jz"):
        assert err[k] <= 2e-5, k
    # the m = 1 angular current q (sin t1 - sin t0), -q (cos t1 - cos t0) is taken from the
    # FP32 phases of the stored angles (the phases the charge density uses, so continuity
    # stays exact); their difference loses digits for small angular moves
    assert err["Jy"] <= 1e-4


def test_split_steps_stay_close_to_fp64():
    say("[case] split vs FP64, 20 steps")
    o = CylModalOracle(24, 32, dr=2.0, c=0.5, c_ompe=10.0, epc=4, cap=20000)
    rng = np.random.default_rng(21)
    o.load_plasma(16, 3, 32, 8, seed=9, cap=20000)
    P = _split_state(o, rng, 0.05)
    F = _smooth_fields(o, rng, amp=5e-3)
    out = []
    for form in ("fp64", "fp32_split"):
        with Simulation(24, 2, 32, ndim=3, epc=4, c=0.5, c_ompe=10.0, form=form, geometry="cyl_modal", dr=2.0,
                        mi_me=1e30, fdtd="lehe") as sim:
            sim.upload_particles(**P)
            sim.upload_fields(*[np.asfortranarray(F[n]) for n in FIELDS])
            sim.step(20)
            out.append((sim.download_fields(), sim.diagnostics()))
    for k in FIELDS:
        d = np.abs(out[1][0][k] - out[0][0][k]).max() / np.abs(out[0][0][k]).max()
        say(f"{k}: split vs FP64 {d:.2e}")
        assert d <= 1e-5, k
    for k in ("E_energy", "B_energy", "prtl_energy_2"):
        assert abs(out[1][1][k] - out[0][1][k]) <= 1e-6 * out[0][1][k], k


def _window_run(form, nsteps=16):
    with Simulation(20, 2, 24, ndim=3, epc=4, c=0.45, c_ompe=10.0, form=form, geometry="cyl_modal", dr=2.0,
                    mi_me=1e30, fdtd="lehe") as sim:
        sim.cyl_plasma(10, 3, 24, 4, seed=13)
        sim.cyl_laser(0.5, 3.0, 0.8, 2.0, 14.0)
        sim.moving_window(True, nr_plasma=10, ppc=4, seed=13)
        sim.step(nsteps)
        return sim.download_fields(), sim.download_particles(), sim.diagnostics()


def test_split_is_deterministic_and_follows_fp64_with_the_window():
    say("[case] split determinism with the moving window")
    F1, P1, d1 = _window_run("fp32_split")
    F2, P2, d2 = _window_run("fp32_split")
    for k in FIELDS + ("Jx", "Jy", "Jz"):
        assert np.array_equal(F1[k], F2[k]), k
    for k in P1:
        assert np.array_equal(P1[k], P2[k]), k
    F0, P0, d0 = _window_run("fp64")
    assert len(P0["x"]) == len(P1["x"]) and np.array_equal(P0["flv"], P1["flv"])
    for k in FIELDS:
        d = np.abs(F1[k] - F0[k]).max() / np.abs(F0[k]).max()
        say(f"{k}: split vs FP64 with the window {d:.2e}")
        assert d <= 1e-5, k


def test_split_run_keeps_modal_gauss_law():
    say("[case] split Gauss law")
    o = CylModalOracle(32, 40, dr=2.0, c=0.5, c_ompe=10.0, epc=4, cap=60000)
    rng = np.random.default_rng(2)
    o.load_plasma(20, 3, 40, 8, seed=2, cap=60000)
    P = _split_state(o, rng, 0.1)
    o.load_particles(P["q"], P["x"], P["y"], P["z"], P["u"], P["v"], P["w"], P["flv"], cap=60000)
    G0 = o.gauss()
    with _split_sim(32, 40, 2.0, 0.5) as sim:
        sim.upload_particles(**P)
        sim.step(40)
        F = sim.download_fields()
        A = sim.download_particles()
    o.set_fields(**{k: F[k] for k in FIELDS})
    o.load_particles(A["q"], A["x"], A["y"], A["z"], A["u"], A["v"], A["w"], A["flv"], cap=60000)
    G1 = o.gauss()
    for s in range(3):
        d = np.abs(G1 - G0)[:, s, :].max() / np.abs(G0[:, s, :]).max()
        say(f"slot {s}: Gauss change / max {d:.2e}")
        assert d <= 1e-6, s


def test_split_contribution_above_the_fixed_point_range_is_an_error():
    o = CylModalOracle(16, 16, dr=1.0, c=0.3, c_ompe=10.0, epc=4, cap=64)
    with _split_sim(16, 16, 1.0, 0.3) as sim:
        # one particle whose weight makes q * qi * dx far above 64 charge cells
        big = -1e9 / o.m.qi
        sim.upload_particles(q=np.array([big]), x=np.array([8.2]), y=np.array([1.0]), z=np.array([8.5]),
                             u=np.array([0.9]), v=np.zeros(1), w=np.zeros(1), flv=np.array([2], dtype=np.int32))
        with pytest.raises(RuntimeError, match="fixed-point"):
            sim.step(1)


@pytest.mark.parametrize("form", ["fp64", "fp32_split"])
def test_window_run_through_compaction_keeps_order(form):
    # 512 particles, room for 1.25 x 512 + 1024 slots; every shift adds 32 and drops about
    # 32 at the back, so after about 36 shifts the arrays are compacted (live particles
    # moved down in order) at least once in 120 steps
    say(f"[case] window through compaction form={form}")
    nr, nz, c, nrp, ppc = 12, 16, 0.45, 8, 4
    o = CylModalOracle(nr, nz, dr=2.0, c=c, c_ompe=10.0, epc=4, cap=20000)
    rng = np.random.default_rng(31)
    o.load_plasma(nrp, 3, nz, ppc, seed=7, cap=20000)
    P = _split_state(o, rng, 0.05)
    o.load_particles(P["q"], P["x"], P["y"], P["z"], P["u"], P["v"], P["w"], P["flv"], cap=20000)
    nsteps, shifts = 120, 0
    with Simulation(nr, 2, nz, ndim=3, epc=4, c=c, c_ompe=10.0, form=form, geometry="cyl_modal", dr=2.0,
                    mi_me=1e30) as sim:
        sim.upload_particles(**P)
        sim.moving_window(True, nr_plasma=nrp, ppc=ppc, seed=7)
        o.set_zopen(True)   # the window box has open z ends, as on the GPU
        sim.step(nsteps)
        A = sim.download_particles()
        G = sim.download_fields()
    for t in range(1, nsteps + 1):
        o.step()
        while t * c >= shifts + 1:
            shifts += 1
            o.shift(nrp, ppc, 7, shifts)
    B = o.particles(live_only=True)
    say(f"shifts {shifts}, slots on the GPU {len(A['x'])}, live {int((A['flv'] != 0).sum())}, oracle live {len(B['x'])}")
    assert shifts == 54
    assert len(A["x"]) < 512 + shifts * nrp * ppc      # the holes were squeezed out
    live = A["flv"] != 0
    if form == "fp64":
        assert live.sum() == len(B["x"])
    else:   # FP32 rounding may move a particle at the back across its cell face when a shift drops the row
        assert abs(int(live.sum()) - len(B["x"])) <= 2
    if live.sum() == len(B["x"]):
        tol = 1e-9 if form == "fp64" else 2e-4
        for k in ("x", "z", "u", "v", "w"):
            d = np.abs(A[k][live] - B[k]).max() / max(np.abs(B[k]).max(), 1.0)
            assert d <= tol, (k, d)
    for k in FIELDS:
        d = np.abs(G[k] - o.F[k]).max() / np.abs(o.F[k]).max()
        say(f"{k}: max diff / max {d:.2e}")
        assert d <= (1e-9 if form == "fp64" else 1e-3), k


@pytest.mark.parametrize("form", ["fp64", "fp32_split"])
def test_sorting_by_cell_keeps_the_physics(form):
    # sorting every 5 steps (stable, by cell, holes dropped) changes only the order: the
    # fields follow the oracle's unsorted run and the particle sets agree; after a sort the
    # arrays hold no holes and run in cell order (k-major, i fastest)
    say(f"[case] sort by cell form={form}")
    nr, nz, c, nrp, ppc = 12, 16, 0.45, 8, 4
    o = CylModalOracle(nr, nz, dr=2.0, c=c, c_ompe=10.0, epc=4, cap=20000)
    rng = np.random.default_rng(41)
    o.load_plasma(nrp, 3, nz, ppc, seed=9, cap=20000)
    P = _split_state(o, rng, 0.2)
    o.load_particles(P["q"], P["x"], P["y"], P["z"], P["u"], P["v"], P["w"], P["flv"], cap=20000)
    nsteps, shifts = 20, 0
    with Simulation(nr, 2, nz, ndim=3, epc=4, c=c, c_ompe=10.0, form=form, geometry="cyl_modal", dr=2.0,
                    mi_me=1e30) as sim:
        sim.upload_particles(**P)
        sim.moving_window(True, nr_plasma=nrp, ppc=ppc, seed=9)
        o.set_zopen(True)   # the window box has open z ends, as on the GPU
        sim.cyl_sort_period(5)
        sim.step(nsteps)
        A = sim.download_particles()
        G = sim.download_fields()
    for t in range(1, nsteps + 1):
        o.step()
        while t * c >= shifts + 1:
            shifts += 1
            o.shift(nrp, ppc, 9, shifts)
    B = o.particles(live_only=True)
    assert np.all(A["flv"] != 0) and len(A["x"]) == len(B["x"])
    key = np.floor(A["z"]) * 4096 + np.floor(A["x"])
    assert np.all(np.diff(key) >= 0)
    ia = np.lexsort((A["y"], A["x"], A["z"]))
    ib = np.lexsort((B["y"], B["x"], B["z"]))
    tol = 1e-9 if form == "fp64" else 2e-4
    for k in ("x", "z", "u", "v", "w"):
        d = np.abs(A[k][ia] - B[k][ib]).max() / max(np.abs(B[k]).max(), 1.0)
        assert d <= tol, (k, d)
    for k in FIELDS:
        d = np.abs(G[k] - o.F[k]).max() / np.abs(o.F[k]).max()
        say(f"{k}: max diff / max {d:.2e}")
        assert d <= (1e-9 if form == "fp64" else 1e-3), k


def _back_state(o, rng):
    """fields in the back rows only (k = 3..5) and electrons at the back moving backwards,
    plus a few slow ones in the middle of the box"""
    mx, _, mz = o.shape
    F = _smooth_fields(o, rng, amp=1e-2)
    for n in FIELDS:
        F[n][:, :, 5:] = 0.0            # python index 5 = Fortran k = 6
        F[n][:, :, :2] = 0.0
    n_back, n_mid = 8, 8
    x = np.concatenate([rng.uniform(5.0, mx - 6.0, n_back + n_mid)])
    z = np.concatenate([rng.uniform(3.05, 3.4, n_back), rng.uniform(8.0, 12.0, n_mid)])
    w = np.concatenate([np.full(n_back, -3.0), np.zeros(n_mid)])
    n = n_back + n_mid
    P = {"q": np.full(n, -1.0), "x": x, "y": rng.uniform(0.0, 2 * np.pi, n), "z": z,
         "u": np.zeros(n), "v": np.zeros(n), "w": w, "flv": np.full(n, 2, dtype=np.int32)}
    return F, P


@pytest.mark.parametrize("form", ["fp64", "fp32_split"])
def test_window_back_does_not_reappear_at_front(form):
    # open z under the moving window: fields of the back rows and electrons leaving through
    # the back must not show up at the front of the box (periodic z would copy the back rows
    # into the front ghosts and wrap the electrons to the front)
    say(f"[case] window open z form={form}")
    # nz = 32: nothing from the back rows or the electrons at rest reaches the front
    # rows in 6 steps (the stencils spread a field by one cell per step)
    nr, nz, c = 12, 32, 0.45
    o = CylModalOracle(nr, nz, dr=2.0, c=c, c_ompe=10.0, epc=4, cap=1024)
    o.set_zopen(True)
    rng = np.random.default_rng(17)
    F, P = _back_state(o, rng)
    if form == "fp32_split":
        cell = np.floor(P["x"]); P["x"] = cell + (P["x"] - cell).astype(np.float32).astype(np.float64)
        cell = np.floor(P["z"]); P["z"] = cell + (P["z"] - cell).astype(np.float32).astype(np.float64)
        P["y"] = np.round(P["y"] / TURN) % 2.0 ** 32 * TURN
    o.set_fields(**F)
    o.load_particles(P["q"], P["x"], P["y"], P["z"], P["u"], P["v"], P["w"], P["flv"], cap=1024)
    nsteps, shifts = 6, 0
    with Simulation(nr, 2, nz, ndim=3, epc=4, c=c, c_ompe=10.0, form=form, geometry="cyl_modal", dr=2.0,
                    mi_me=1e30) as sim:
        sim.upload_fields(*[np.asfortranarray(F[n]) for n in FIELDS])
        sim.upload_particles(**P)
        sim.moving_window(True, nr_plasma=0, ppc=0, seed=1)
        sim.step(nsteps)
        G = sim.download_fields()
        A = sim.download_particles()
    for t in range(1, nsteps + 1):
        o.step()
        while t * c >= shifts + 1:
            shifts += 1
            o.shift(0, 0, 1, shifts)
    assert shifts == 2
    mz = o.shape[2]
    front = slice(mz - 8, mz)     # Fortran rows mz-7 .. mz: the front physical rows and ghosts
    for n in FIELDS:
        assert np.all(G[n][:, :, front] == 0.0), n
        assert np.all(o.F[n][:, :, front] == 0.0), n
        assert np.abs(G[n]).max() > 0.0, n
    live = A["flv"] != 0
    B = o.particles(live_only=True)
    say(f"live particles GPU {int(live.sum())}, oracle {len(B['x'])}")
    assert int(live.sum()) == len(B["x"]) == 8        # the 8 backward electrons left the box
    assert np.all(A["z"][live] < 13.0)
    for n in FIELDS:
        d = np.abs(G[n] - o.F[n]).max() / np.abs(o.F[n]).max()
        assert d <= (1e-9 if form == "fp64" else 1e-4), (n, d)


@pytest.mark.parametrize("form", ["fp32_split", "fp64"])
@pytest.mark.parametrize("n", [1, 16, 17, 255, 257, 4000, 30000])
def test_current_does_not_depend_on_the_particle_order(form, n):
    # in cell order most blocks deposit through one window, over the end of a row of cells two; shuffled
    # ones go through boxes and what is left through direct adds; "packed" crowds a few cells
    say(f"[case] cylm order {form} n={n}")
    nr, nz = 90, 48
    rng = np.random.default_rng(n)
    x, z = rng.uniform(4.0, nr - 8.0, n), rng.uniform(3.0, nz + 2.9, n)
    packed = rng.random(n) < 0.3
    x[packed], z[packed] = 20.0 + 2.0 * rng.random(packed.sum()), 11.0 + rng.random(packed.sum())
    P = dict(q=rng.uniform(0.5, 2.0, n) * rng.choice([-1.0, 1.0], n), x=x, y=rng.uniform(0.0, 2.0 * np.pi, n), z=z,
             u=rng.normal(0.0, 0.4, n), v=rng.normal(0.0, 0.4, n), w=rng.normal(0.0, 0.6, n),
             flv=rng.integers(1, 3, n).astype(np.int32))
    cells = np.lexsort((np.floor(x), np.floor(z)))
    J = []
    for order in (cells, cells[::-1], rng.permutation(n)):
        with Simulation(nr, 2, nz, ndim=3, epc=4, c=0.3, c_ompe=10.0, form=form, geometry="cyl_modal") as sim:
            sim.upload_particles(**{k: a[order] for k, a in P.items()})
            sim.ResetCurrent()
            sim.MoveDepositPrtl()
            out = sim.download_fields()
            J.append([out[k] for k in ("Jx", "Jy", "Jz")])
    for other in J[1:]:
        for a, b in zip(J[0], other):
            if form == "fp32_split":
                assert np.array_equal(a, b)
            else:
                # the crowded nodes take up to 0.3 n contributions in another order: 2^-53 of each partial sum
                assert np.abs(a - b).max() <= max(n, 10) * 2.0 ** -53 * 20.0 * np.abs(a).max()
    assert np.abs(J[0][0]).max() > 0.0


@pytest.mark.parametrize("form", ["fp32_split", "fp64"])
@pytest.mark.parametrize("fdtd", ["yee", "lehe"])
@pytest.mark.parametrize("nr,nz", [(8, 8), (24, 13), (70, 41)])
def test_open_run_equals_phases_and_shifts(form, fdtd, nr, nz):
    # steps of a window run enqueued together against the phase calls, with the window's shift made by
    # hand: every row moves one cell back, the front and the z ghosts restart at zero, J is cleared,
    # E's axis rows follow from the fourth column.  The first fields fill ghosts and wall, too.
    say(f"[case] cylm open run {form} {fdtd} {nr}x{nz}")
    c, steps = 0.4, 7
    rng = np.random.default_rng(nr + nz)

    def make():
        sim = Simulation(nr, 2, nz, ndim=3, epc=4, c=c, c_ompe=10.0, form=form, geometry="cyl_modal", fdtd=fdtd)
        sim.moving_window(True)
        return sim

    with make() as sim:
        shape = sim.shape
    n = 40 * nz
    P = dict(q=rng.uniform(0.5, 1.0, n), x=rng.uniform(4.0, nr - 0.5, n),
             y=rng.uniform(0.0, 2.0 * np.pi, n), z=rng.uniform(3.0, nz + 2.9, n), u=rng.normal(0.0, 0.02, n),
             v=rng.normal(0.0, 0.2, n), w=rng.normal(0.0, 0.3, n), flv=np.full(n, 2, np.int32))
    F0 = [np.asfortranarray(1e-3 * rng.standard_normal(shape)) for _ in FIELDS]
    with make() as a, make() as b:
        for sim in (a, b):
            sim.upload_fields(*F0)
            sim.upload_particles(**P)
        a.step(steps)
        got = a.download_fields()
        pa = a.download_particles()
        shift = 0
        for t in range(1, steps + 1):
            b.step_phases()
            if t * c < shift + 1:
                continue
            shift += 1
            f, p = b.download_fields(), b.download_particles()
            mx, mz = shape[0], shape[2]
            for k in FIELDS:
                g = np.zeros(shape, order="F")
                g[:, :, :mz - 4] = f[k][:, :, 1:mz - 3]
                f[k] = g
            par = np.array([1.0, -1.0, -1.0])[:, None]
            four = {k: f[k][3].copy() for k in ("Ex", "Ey", "Ez")}
            f["Ex"][2], f["Ex"][1] = 0.5 * (four["Ex"] - par * four["Ex"]), -par * four["Ex"]
            f["Ey"][2], f["Ez"][2] = -par * four["Ey"], par * four["Ez"]
            for k in FIELDS:
                f[k][2:mx - 3, :, :2] = 0.0
                f[k][2:mx - 3, :, mz - 3:] = 0.0
                f[k][mx - 3:] = 0.0
            p["z"] = np.where(p["flv"] != 0, p["z"] - 1.0, p["z"])
            p["flv"] = np.where(p["z"] < 3.0, 0, p["flv"]).astype(np.int32)
            b.upload_fields(*[f[k] for k in FIELDS])
            b.upload_particles(**p)
            b.ResetCurrent()
        want, pb = b.download_fields(), b.download_particles()
    live = pa["flv"] != 0
    assert live.sum() == (pb["flv"] != 0).sum()
    for k in ("Ex", "Ey", "Ez", "Bx", "By", "Bz", "Jx", "Jy", "Jz"):
        if form == "fp32_split":
            assert np.array_equal(got[k], want[k]), k
        else:   # the order of the current's FP64 adds
            assert np.abs(got[k] - want[k]).max() <= 1e-12 * max(np.abs(want[k]).max(), 1e-300), k
    for k in ("x", "z", "u", "w"):
        assert np.abs(pa[k][live] - pb[k][pb["flv"] != 0]).max() <= (0.0 if form == "fp32_split" else 1e-12), k


@pytest.mark.parametrize("form", ["fp32_split", "fp64"])
def test_error_inside_an_open_run_stops_behind_that_push(form):
    # a particle that reaches the wall in step 4: the same error and state as steps one at a time
    say(f"[case] cylm open run error {form}")
    P = dict(q=[1.0, 1.0], x=[19.5, 9.5], y=[0.0, 1.0], z=[20.5, 20.5], u=[3.0, 0.0], v=[0.0, 0.0], w=[0.0, 0.1],
             flv=np.array([2, 2], np.int32))
    out = []
    for one in (False, True):
        with Simulation(18, 2, 32, ndim=3, epc=4, c=0.4, c_ompe=10.0, form=form, geometry="cyl_modal") as sim:
            sim.moving_window(True)
            sim.upload_particles(**P)
            with pytest.raises(RuntimeError, match="outer wall"):
                for _ in range(12 if one else 1):
                    sim.step(1 if one else 12)
            out.append((sim.download_fields(), sim.download_particles(), sim.timer("step")[1]))
    (fa, pa, na), (fb, pb, nb) = out
    assert na == nb and 0 < na < 12
    for k in fa:
        assert np.array_equal(fa[k], fb[k]), k
    for k in pa:
        assert np.array_equal(pa[k], pb[k]), k


@pytest.mark.parametrize("form", ["fp32_split", "fp64"])
def test_memory_report_counts_the_window_run(form):
    # the moving window's run keeps a second set of E and B: six FP64 arrays
    say(f"[case] cylm memory report {form}")
    with Simulation(18, 2, 32, ndim=3, epc=4, c=0.4, c_ompe=10.0, form=form, geometry="cyl_modal") as sim:
        sim.moving_window(True)
        before = sim.memory_bytes()
        sim.step(3)
        assert sim.memory_bytes() == before + 6 * 8 * int(np.prod(sim.shape))


def test_window_run_without_room_for_second_fields():
    # a card with room for some of the second E and B: none of them stays, the steps run one at a time
    # with the same bits, and the run takes them when there is room again
    import torch

    say("[case] cylm window run on a full card")

    def make():
        sim = Simulation(500, 2, 4000, ndim=3, epc=4, c=0.4, c_ompe=10.0, form="fp32_split", geometry="cyl_modal", dr=2.0)
        sim.cyl_plasma(100, 3, 200, 4, seed=3)
        sim.moving_window(True)
        sim.cyl_laser(0.5, 8.0, 2.0, 3.0, 150.0)
        sim.ResetCurrent()
        sim.MoveDepositPrtl()      # allocates the push's node copy
        sim.ExchangePrtl()
        return sim

    with make() as sim:
        lean, array = sim.memory_bytes(), 8 * int(np.prod(sim.shape))
        sim.step(7)
        want, full = sim.download_fields(), sim.memory_bytes()
    assert full == lean + 6 * array
    with make() as sim:
        torch.cuda.empty_cache()
        held = [torch.empty(torch.cuda.mem_get_info()[0] - (256 << 20), dtype=torch.uint8, device="cuda")]
        try:
            while True:     # more than the runtime says is there
                held.append(torch.empty(22 << 20, dtype=torch.uint8, device="cuda"))
        except torch.OutOfMemoryError:
            del held[-(3 * array // (22 << 20)):]
            torch.cuda.empty_cache()
        sim.step(7)
        assert sim.memory_bytes() == lean
        del held
        torch.cuda.empty_cache()
        got = sim.download_fields()
        sim.step(1)
        assert sim.memory_bytes() == full
    for k in want:
        assert np.array_equal(got[k], want[k]), k
