"""The fixed-point current of the split forms, bit for bit: a contribution is the FP64 product of a
flux and a weight rounded to an integer count (of 2^-30 or 2^-36 charge cells), both computed from
the stored old and new positions.  Large charges make the products inexact, so that a count made
with one rounding instead of two (a fused multiply-add) differs for one in some ten thousand; the sums of
counts are exact in any order, so one such count changes a node."""
import numpy as np
import pytest

from pictor_amd import Simulation

from _util import say

pytestmark = pytest.mark.gpu


def _relay(p0, p1, c0, c1):
    return np.minimum(np.minimum(c0, c1) + 1.0, np.maximum(np.maximum(c0, c1), 0.5 * (p0 + p1)))


@pytest.mark.parametrize("tile", [8, 16, 32])
def test_cartesian_counts(tile):
    nx, ny, n = 64, 96, 150000
    say("2-D split counts, tile", tile)
    rng = np.random.default_rng(tile)
    flv = rng.integers(1, 3, n).astype(np.int32)
    wt = rng.uniform(500.0, 3000.0, n).astype(np.float32).astype(np.float64)
    P = {"q": np.where(flv == 1, wt, -wt), "x": rng.uniform(6.0, nx - 1.0, n), "y": rng.uniform(6.0, ny - 1.0, n),
         "z": np.full(n, 1.5), "u": rng.normal(0, 0.7, n), "v": rng.normal(0, 0.7, n), "w": rng.normal(0, 0.7, n)}
    with Simulation(nx, ny, epc=8, form="fp32_split", tile=tile) as sim:
        sim.upload_particles(**P, flv=flv, tag=np.arange(n, dtype=np.int32))
        was = sim.download_particles(with_tag=True)
        sim.ResetCurrent()
        sim.MoveDepositPrtl()
        sim.ExchangePrtl()
        now = sim.download_particles(with_tag=True)
        F = sim.download_fields()
        scale = sim.qi / 2.0 ** 30
    a, b = np.argsort(was["tag"]), np.argsort(now["tag"])
    x0, y0, x1, y1 = was["x"][a], was["y"][a], now["x"][b], now["y"][b]
    assert np.abs(x1 - x0).max() < 0.5 and (np.floor(x1) != np.floor(x0)).sum() > 1000   # some leave their cell
    qs = was["q"][a] * 2.0 ** 30
    i0, j0, i1, j1 = (np.floor(p) for p in (x0, y0, x1, y1))
    # positions in their old cells, as the kernel holds them
    X0, Y0, X1, Y1 = x0 - i0, y0 - j0, (x1 - i1) + (i1 - i0), (y1 - j1) + (j1 - j0)
    xr, yr = _relay(X0, X1, 0.0 * i0, i1 - i0), _relay(Y0, Y1, 0.0 * j0, j1 - j0)
    Jx, Jy = np.zeros((nx + 5, ny + 5)), np.zeros((nx + 5, ny + 5))
    for xa, ya, xb, yb, di, dj, i, j in ((X0, Y0, xr, yr, 0.0, 0.0, i0, j0), (xr, yr, X1, Y1, i1 - i0, j1 - j0, i1, j1)):
        Fx, Fy = qs * (xb - xa), qs * (yb - ya)
        Wx, Wy = 0.5 * (xa + xb) - di, 0.5 * (ya + yb) - dj
        i, j = i.astype(int) - 1, j.astype(int) - 1
        np.add.at(Jx, (i, j), np.rint(Fx * (1.0 - Wy)))
        np.add.at(Jx, (i, j + 1), np.rint(Fx * Wy))
        np.add.at(Jy, (i, j), np.rint(Fy * (1.0 - Wx)))
        np.add.at(Jy, (i + 1, j), np.rint(Fy * Wx))
    assert np.abs(Jx).max() > 0
    for name, want in (("Jx", Jx), ("Jy", Jy)):
        got = F[name].reshape(want.shape)
        assert np.array_equal(got, want * scale), (name, np.count_nonzero(got != want * scale))


@pytest.mark.parametrize("shuffled", [False, True])
def test_modal_counts(shuffled):
    nr, nz, n = 48, 96, 60000
    say("modal split counts, shuffled", shuffled)
    rng = np.random.default_rng(5)
    x, z = rng.uniform(8.0, nr - 4.0, n), rng.uniform(10.0, nz - 8.0, n)
    if not shuffled:
        o = np.lexsort((x, np.floor(x), np.floor(z)))
        x, z = x[o], z[o]
    P = {"q": -rng.uniform(1e5, 4e5, n).astype(np.float32).astype(np.float64), "x": x,
         "y": rng.uniform(0.0, 2 * np.pi, n), "z": z, "u": rng.normal(0, 0.7, n), "v": rng.normal(0, 0.7, n),
         "w": rng.normal(0, 0.7, n)}
    with Simulation(nr, 2, nz, ndim=3, epc=16, c=0.8, c_ompe=20.0, mi_me=1e30, form="fp32_split", geometry="cyl_modal",
                    dr=4.0) as sim:
        sim.upload_particles(**P, flv=np.full(n, 2, np.int32))
        was = sim.download_particles()
        sim.ResetCurrent()
        sim.MoveDepositPrtl()
        sim.ExchangePrtl()
        now = sim.download_particles()     # the array order of the particles is kept
        F = sim.download_fields()
        qi = sim.qi
    x0, z0, x1, z1 = was["x"], was["z"], now["x"], now["z"]
    assert np.abs(x1 - x0).max() < 1.0 and np.abs(z1 - z0).max() < 1.0
    i0, k0, i1, k1 = (np.floor(p) for p in (x0, z0, x1, z1))
    assert ((i0 != i1) | (k0 != k1)).any() and ((i0 == i1) & (k0 == k1)).any()
    qs = was["q"] * qi * 2.0 ** 36
    xr, zr = _relay(x0, x1, i0, i1), _relay(z0, z1, k0, k1)
    Jr, Jz = np.zeros((nr + 5, nz + 5)), np.zeros((nr + 5, nz + 5))
    for xa, za, xb, zb, i, k in ((x0, z0, xr, zr, i0, k0), (xr, zr, x1, z1, i1, k1)):
        Fx, Fz = qs * (xb - xa), qs * (zb - za)
        Wx, Wz = 0.5 * (xa + xb) - i, 0.5 * (za + zb) - k
        i, k = i.astype(int) - 1, k.astype(int) - 1
        np.add.at(Jr, (i, k), np.rint(Fx * (1.0 - Wz)))
        np.add.at(Jr, (i, k + 1), np.rint(Fx * Wz))
        np.add.at(Jz, (i, k), np.rint(Fz * (1.0 - Wx)))
        np.add.at(Jz, (i + 1, k), np.rint(Fz * Wx))
    for name, want in (("Jx", Jr), ("Jz", Jz)):
        got = F[name][:, 0, :] * 2.0 ** 36      # slot 0: mode m = 0
        assert np.array_equal(got, want), (name, np.count_nonzero(got != want))


@pytest.mark.parametrize("n", [1, 7, 64])
def test_modal_fp64_sums_in_order(n):
    # FP64 sums show their order.  One wave of particles has one: lane l adds into copy l % 4, one node
    # after the other, first and second half of the move apart, and the copies are added 0 to 3
    say("modal FP64 sums,", n, "particles")
    nr = nz = 32
    rng = np.random.default_rng(n)
    P = {"q": -rng.uniform(1.0, 400.0, n), "x": 12.0 + rng.uniform(0.0, 2.0, n), "y": rng.uniform(0.0, 2 * np.pi, n),
         "z": 14.0 + rng.uniform(0.0, 2.0, n), "u": rng.normal(0, 0.7, n), "v": rng.normal(0, 0.7, n),
         "w": rng.normal(0, 0.7, n)}
    with Simulation(nr, 2, nz, ndim=3, epc=16, c=0.8, c_ompe=20.0, mi_me=1e30, form="fp64", geometry="cyl_modal",
                    dr=4.0) as sim:
        sim.upload_particles(**P, flv=np.full(n, 2, np.int32))
        sim.ResetCurrent()
        sim.MoveDepositPrtl()
        sim.ExchangePrtl()
        now = sim.download_particles()
        F = sim.download_fields()
        qi = sim.qi
    x0, z0, x1, z1 = P["x"], P["z"], now["x"], now["z"]
    i0, k0, i1, k1 = (np.floor(p).astype(int) for p in (x0, z0, x1, z1))
    qs = P["q"] * qi
    xr, zr = _relay(x0, x1, i0.astype(float), i1.astype(float)), _relay(z0, z1, k0.astype(float), k1.astype(float))
    J = np.zeros((2, 4, nr + 5, nz + 5))
    for xa, za, xb, zb, i, k in ((x0, z0, xr, zr, i0, k0), (xr, zr, x1, z1, i1, k1)):
        Fx, Fz = qs * (xb - xa), qs * (zb - za)
        Wx, Wz = 0.5 * (xa + xb) - i, 0.5 * (za + zb) - k
        for c, di, dk, v in ((0, 0, 0, Fx * (1.0 - Wz)), (0, 0, 1, Fx * Wz), (1, 0, 0, Fz * (1.0 - Wx)), (1, 1, 0, Fz * Wx)):
            for l in range(n):
                J[c, l % 4, i[l] + di - 1, k[l] + dk - 1] += v[l]
    for c, name in enumerate(("Jx", "Jz")):
        want = ((J[c, 0] + J[c, 1]) + J[c, 2]) + J[c, 3]
        assert np.count_nonzero(want) > 0
        assert np.array_equal(F[name][:, 0, :], want), np.abs(F[name][:, 0, :] - want).max()
