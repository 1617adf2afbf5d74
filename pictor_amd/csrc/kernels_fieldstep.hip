// kernels_fieldstep.hip -- the field work between two pushes of a periodic box in one launch.
//
// Between the push of step t and the push of step t + 1, MAIN.F90:51-251 runs the second B
// half step, the current halo, UpdateEfield + AddCurrent, ResetCurrent and the first B half
// step, each followed by its halo exchange: eleven launches over arrays that a small grid
// keeps in cache, and six passes over them on a large one.  k_field_step does the same
// arithmetic, term by term in the same order, in one pass: a workgroup computes B after the
// half step on its tile and the surrounding cells it needs (from E and B in memory), the new
// E on its tile and the cells above it, and the next half step of B on its tile, handing the
// values on through LDS.  What a tile recomputes of its neighbours is bitwise what they
// compute.  E, B and J go to second buffers, because the neighbours still read the first.
// Every physical cell writes itself and its ghost images; the current of the ghost layers is
// added to its owners as it is read.  The other current buffer is cleared for the next push.
//
// Bound: HBM, and at small sizes the launch.  In the split form a cell reads E (hi, lo), B and
// J and writes E, B and zeros: 120 B, against 280 B over the separate kernels.  Field work of a
// step, before and after: 2048 x 2048 split 204 -> 135 us, 128^3 split 171 -> 135 us, 256 x 256
// FP64 46 -> 13.5 us, 32 x 32 FP64 40 -> 12 us.  64 cells along x make a row's segment 256 or
// 512 B (32 x 8 tiles: 152 us at 2048 x 2048), and consecutive tiles run on one XCD, whose L2
// then holds the halos and the lines that two tiles share (172 us with the tiles dealt round).
//
// A step after one that spilled particles or failed must not run: its launches find `gate`
// closed and return, so that the host can enqueue many steps before it looks.
#include "fieldstep.h"

namespace pictor {
namespace {

__device__ inline int wrapc(int c, int n) { return c < 3 ? c + n : (c > n + 2 ? c - n : c); }

// F at an offset from the cell, read from memory or from a workgroup's LDS block
template <typename R>
struct MemAcc {
    const R *p;
    long long sy, sz;
    __device__ R operator()(int x, int y, int z) const { return p[x + y * sy + z * sz]; }
};
template <typename R>
struct LdsAcc {
    const R *p;
    int sy, sz;
    __device__ R operator()(int x, int y, int z) const { return p[x + y * sy + z * sz]; }
};

// gradX, gradY, gradZ of em_update_lehe.F90:120-155, term order kept
template <typename R, int DIM, typename A>
__device__ inline R lehe_x(const LeheP<R> &L, R d, const A &f)
{
    R v = L.ax * d * (f(1, 0, 0) - f(0, 0, 0)) + L.bxy * d * (f(1, 1, 0) - f(0, 1, 0)) +
          L.bxy * d * (f(1, -1, 0) - f(0, -1, 0));
    if (DIM == 3) v = v + L.bxz * d * (f(1, 0, 1) - f(0, 0, 1)) + L.bxz * d * (f(1, 0, -1) - f(0, 0, -1));
    return v + L.dx * d * (f(2, 0, 0) - f(-1, 0, 0));
}
template <typename R, int DIM, typename A>
__device__ inline R lehe_y(const LeheP<R> &L, R d, const A &f)
{
    R v = L.ay * d * (f(0, 1, 0) - f(0, 0, 0)) + L.byx * d * (f(1, 1, 0) - f(1, 0, 0)) +
          L.byx * d * (f(-1, 1, 0) - f(-1, 0, 0));
    if (DIM == 3) v = v + L.byz * d * (f(0, 1, 1) - f(0, 0, 1)) + L.byz * d * (f(0, 1, -1) - f(0, 0, -1));
    return v + L.dy * d * (f(0, 2, 0) - f(0, -1, 0));
}
template <typename R, int DIM, typename A>
__device__ inline R lehe_z(const LeheP<R> &L, R d, const A &f)
{
    return L.az * d * (f(0, 0, 1) - f(0, 0, 0)) + L.bzx * d * (f(1, 0, 1) - f(1, 0, 0)) +
           L.bzx * d * (f(-1, 0, 1) - f(-1, 0, 0)) + L.bzy * d * (f(0, 1, 1) - f(0, 1, 0)) +
           L.bzy * d * (f(0, -1, 1) - f(0, -1, 0)) + L.dz * d * (f(0, 0, 2) - f(0, 0, -1));
}

// b after a B half step from the E accessors (em_update.F90:41-77 / em_update_lehe.F90:88-118)
template <typename R, int DIM, bool LEHE, typename A>
__device__ inline void b_half(const FieldC<R> &c, const A &Ex, const A &Ey, const A &Ez, R b[3])
{
    const R hc = c.hc, ix = c.idx, iy = c.idy, iz = c.idz;
    if (LEHE) {
        if (DIM == 2) {
            b[0] = b[0] - hc * lehe_y<R, DIM>(c.L, iy, Ez);
            b[1] = b[1] + hc * lehe_x<R, DIM>(c.L, ix, Ez);
            b[2] = b[2] - hc * lehe_x<R, DIM>(c.L, ix, Ey) + hc * lehe_y<R, DIM>(c.L, iy, Ex);
        } else {
            b[0] = b[0] - hc * lehe_y<R, DIM>(c.L, iy, Ez) + hc * lehe_z<R, DIM>(c.L, iz, Ey);
            b[1] = b[1] - hc * lehe_z<R, DIM>(c.L, iz, Ex) + hc * lehe_x<R, DIM>(c.L, ix, Ez);
            b[2] = b[2] - hc * lehe_x<R, DIM>(c.L, ix, Ey) + hc * lehe_y<R, DIM>(c.L, iy, Ex);
        }
        return;
    }
    const R ex = Ex(0, 0, 0), ey = Ey(0, 0, 0), ez = Ez(0, 0, 0);
    if (DIM == 2) {
        b[0] = b[0] - hc * iy * (Ez(0, 1, 0) - ez);
        b[1] = b[1] + hc * ix * (Ez(1, 0, 0) - ez);
        b[2] = b[2] - hc * ix * (Ey(1, 0, 0) - ey) + hc * iy * (Ex(0, 1, 0) - ex);
    } else {
        b[0] = b[0] - hc * iy * (Ez(0, 1, 0) - ez) + hc * iz * (Ey(0, 0, 1) - ey);
        b[1] = b[1] - hc * iz * (Ex(0, 0, 1) - ex) + hc * ix * (Ez(1, 0, 0) - ez);
        b[2] = b[2] - hc * ix * (Ey(1, 0, 0) - ey) + hc * iy * (Ex(0, 1, 0) - ex);
    }
}

// the current of the physical cell (i, j, k) with what its ghost images received
// (UpdateCurrentAllFaces: x, then y, then z)
template <int DIM>
__device__ inline double folded(const GridP &g, const double *J, int i, int j, int k)
{
    const int di = i <= 5 ? g.nx : (i >= g.mx - 4 ? -g.nx : 0);
    const int dj = j <= 5 ? g.ny : (j >= g.my - 4 ? -g.ny : 0);
    const long long sy = g.mx, sz = (long long)g.mx * g.my;
    auto fx = [&](const double *p) { return di ? p[0] + p[di] : p[0]; };
    auto fy = [&](const double *p) { return dj ? fx(p) + fx(p + dj * sy) : fx(p); };
    const double *p = J + fidx(g, i, j, k);
    if (DIM == 2) return fy(p);
    const int dk = k <= 5 ? g.nz : (k >= g.mz - 4 ? -g.nz : 0);
    return dk ? fy(p) + fy(p + dk * sz) : fy(p);
}

// E after UpdateEfield and AddCurrent from the B accessors; e: E before (FP64 of the pair)
template <typename R, int DIM, typename A>
__device__ inline void e_step(const FieldC<R> &c, const A &Bx, const A &By, const A &Bz, const double j[3], double e[3])
{
    if (sizeof(R) == 8) {
        const R ix = c.idx, iy = c.idy, iz = c.idz, fc = c.fc;
        const R bx = Bx(0, 0, 0), by = By(0, 0, 0), bz = Bz(0, 0, 0);
        R ex = e[0], ey = e[1], ez = e[2];
        if (DIM == 2) {
            ex = ex + fc * iy * (bz - Bz(0, -1, 0));
            ey = ey - fc * ix * (bz - Bz(-1, 0, 0));
        } else {
            ex = ex + fc * iy * (bz - Bz(0, -1, 0)) - fc * iz * (by - By(0, 0, -1));
            ey = ey + fc * iz * (bx - Bx(0, 0, -1)) - fc * ix * (bz - Bz(-1, 0, 0));
        }
        ez = ez + fc * ix * (by - By(-1, 0, 0)) - fc * iy * (bx - Bx(0, -1, 0));
        e[0] = ex - j[0] * iy * iz;
        e[1] = ey - j[1] * ix * iz;
        e[2] = ez - j[2] * iy * ix;
    } else {
        const double ix = c.dix, iy = c.diy, iz = c.diz, fc = c.dfc;
        const double bx = Bx(0, 0, 0), by = By(0, 0, 0), bz = Bz(0, 0, 0);
        double ex = e[0], ey = e[1], ez = e[2];
        if (DIM == 2) {
            ex = ex + fc * iy * (bz - (double)Bz(0, -1, 0));
            ey = ey - fc * ix * (bz - (double)Bz(-1, 0, 0));
        } else {
            ex = ex + fc * iy * (bz - (double)Bz(0, -1, 0)) - fc * iz * (by - (double)By(0, 0, -1));
            ey = ey + fc * iz * (bx - (double)Bx(0, 0, -1)) - fc * ix * (bz - (double)Bz(-1, 0, 0));
        }
        ez = ez + fc * ix * (by - (double)By(-1, 0, 0)) - fc * iy * (bx - (double)Bx(0, -1, 0));
        // through the stored pair between the curl and the current, as the separate phases
        ex = pair_value(ex); ey = pair_value(ey); ez = pair_value(ez);
        e[0] = ex - (j[0] * c.jscale) * iy * iz;
        e[1] = ey - (j[1] * c.jscale) * ix * iz;
        e[2] = ez - (j[2] * c.jscale) * iy * ix;
    }
}

// the flat indices of a physical cell and its ghost images
template <int DIM, typename F>
__device__ inline void for_images(const GridP &g, int i, int j, int k, F f)
{
    const int di = i <= 5 ? g.nx : (i >= g.mx - 4 ? -g.nx : 0);
    const int dj = j <= 5 ? g.ny : (j >= g.my - 4 ? -g.ny : 0);
    const int dk = DIM == 3 ? (k <= 5 ? g.nz : (k >= g.mz - 4 ? -g.nz : 0)) : 0;
    const long long sy = g.mx, sz = (long long)g.mx * g.my, o = fidx(g, i, j, k);
    for (int c = 0; c < (dk ? 2 : 1); c++)
        for (int b = 0; b < (dj ? 2 : 1); b++)
            for (int a = 0; a < (di ? 2 : 1); a++) f(o + a * di + b * dj * sy + c * dk * sz);
}

// tile of cells per workgroup and the halos it recomputes: E on [-EL, +EH] around it (what
// the next B half step reads), B on one cell below that
template <int DIM, bool LEHE>
struct FieldTile {
    static constexpr int TX = 64, TY = DIM == 2 ? 8 : 4, TZ = DIM == 2 ? 1 : 2, BS = 512;
    static constexpr int EL = LEHE ? 1 : 0, EH = LEHE ? 2 : 1;
    static constexpr int EX = TX + EL + EH, EY = TY + EL + EH, EZ = DIM == 2 ? 1 : TZ + EL + EH;
    static constexpr int BX = EX + 1, BY = EY + 1, BZ = DIM == 2 ? 1 : EZ + 1;
    static constexpr int NE = EX * EY * EZ, NB = BX * BY * BZ;
};

template <typename R, int DIM, bool LEHE>
__global__ __launch_bounds__((FieldTile<DIM, LEHE>::BS)) void k_field_step(GridP g, FieldC<R> c, FieldStepP<R> P)
{
    using T = FieldTile<DIM, LEHE>;
    __shared__ R sB[3][T::NB];
    __shared__ R sE[3][T::NE];
    if (gate_closed(P.gate)) return;
    const int tid = threadIdx.x;
    if (P.host && blockIdx.x == 0 && tid == 0) {
        // the push of this step is complete: its spill count, errors and stop step for the host
        volatile int *h = P.host;
        h[0] = *P.spill; h[1] = *P.err; h[2] = *P.gate.stop;
    }
    // consecutive tiles run on one XCD, so that the lines and halos they share meet in its L2
    const int nbx = (g.nx + T::TX - 1) / T::TX, nby = (g.ny + T::TY - 1) / T::TY;
    int bid = blockIdx.x;
    const int per = gridDim.x >> 3;
    if (bid < per * 8) bid = (bid & 7) * per + (bid >> 3);
    const int x0 = 3 + bid % nbx * T::TX, y0 = 3 + bid / nbx % nby * T::TY, z0 = DIM == 3 ? 3 + bid / (nbx * nby) * T::TZ : 1;
    const int hx = g.mx - 3 + T::EH, hy = g.my - 3 + T::EH, hz = DIM == 3 ? g.mz - 3 + T::EH : 1;
    const long long sy = g.mx, sz = (long long)g.mx * g.my;
    for (int e = tid; e < T::NB; e += T::BS) {
        const int i = x0 - T::EL - 1 + e % T::BX, j = y0 - T::EL - 1 + (e / T::BX) % T::BY;
        const int k = DIM == 3 ? z0 - T::EL - 1 + e / (T::BX * T::BY) : 1;
        if (i > hx || j > hy || k > hz) continue;
        const long long o = fidx(g, wrapc(i, g.nx), wrapc(j, g.ny), DIM == 3 ? wrapc(k, g.nz) : 1);
        R b[3] = {P.B[0][o], P.B[1][o], P.B[2][o]};
        b_half<R, DIM, LEHE>(c, MemAcc<R>{P.E[0] + o, sy, sz}, MemAcc<R>{P.E[1] + o, sy, sz},
                             MemAcc<R>{P.E[2] + o, sy, sz}, b);
        sB[0][e] = b[0]; sB[1][e] = b[1]; sB[2][e] = b[2];
    }
    __syncthreads();
    for (int e = tid; e < T::NE; e += T::BS) {
        const int a = e % T::EX, b = (e / T::EX) % T::EY, d = DIM == 3 ? e / (T::EX * T::EY) : 0;
        const int i = x0 - T::EL + a, j = y0 - T::EL + b, k = DIM == 3 ? z0 - T::EL + d : 1;
        if (i > hx || j > hy || k > hz) continue;
        const int wi = wrapc(i, g.nx), wj = wrapc(j, g.ny), wk = DIM == 3 ? wrapc(k, g.nz) : 1;
        const long long o = fidx(g, wi, wj, wk);
        const int q = ((DIM == 3 ? d + 1 : 0) * T::BY + b + 1) * T::BX + a + 1;
        double v[3], J[3];
#pragma unroll
        for (int m = 0; m < 3; m++) {
            v[m] = sizeof(R) == 8 ? (double)P.E[m][o] : (double)P.E[m][o] + (double)P.L[m][o];
            J[m] = P.fold ? folded<DIM>(g, P.J[m], wi, wj, wk) : P.J[m][o];
        }
        e_step<R, DIM>(c, LdsAcc<R>{sB[0] + q, T::BX, T::BX * T::BY}, LdsAcc<R>{sB[1] + q, T::BX, T::BX * T::BY},
                       LdsAcc<R>{sB[2] + q, T::BX, T::BX * T::BY}, J, v);
        const R h[3] = {(R)v[0], (R)v[1], (R)v[2]};
        sE[0][e] = h[0]; sE[1][e] = h[1]; sE[2][e] = h[2];
        const bool own = a >= T::EL && a < T::EL + T::TX && b >= T::EL && b < T::EL + T::TY && i <= g.mx - 3 &&
                         j <= g.my - 3 && (DIM == 2 || (d >= T::EL && d < T::EL + T::TZ && k <= g.mz - 3));
        if (own)
            for_images<DIM>(g, i, j, k, [&](long long t) {
#pragma unroll
                for (int m = 0; m < 3; m++) {
                    P.En[m][t] = h[m];
                    if (sizeof(R) == 4) P.Ln[m][t] = (float)(v[m] - (double)h[m]);
                    if (P.Jz[m]) P.Jz[m][t] = 0.0;
                }
            });
    }
    __syncthreads();
    for (int e = tid; e < T::TX * T::TY * T::TZ; e += T::BS) {
        const int a = e % T::TX, b = (e / T::TX) % T::TY, d = DIM == 3 ? e / (T::TX * T::TY) : 0;
        const int i = x0 + a, j = y0 + b, k = DIM == 3 ? z0 + d : 1;
        if (i > g.mx - 3 || j > g.my - 3 || (DIM == 3 && k > g.mz - 3)) continue;
        const int q = ((DIM == 3 ? d + T::EL + 1 : 0) * T::BY + b + T::EL + 1) * T::BX + a + T::EL + 1;
        const int r = ((DIM == 3 ? d + T::EL : 0) * T::EY + b + T::EL) * T::EX + a + T::EL;
        R n[3] = {sB[0][q], sB[1][q], sB[2][q]};
        if (P.next)
            b_half<R, DIM, LEHE>(c, LdsAcc<R>{sE[0] + r, T::EX, T::EX * T::EY}, LdsAcc<R>{sE[1] + r, T::EX, T::EX * T::EY},
                                 LdsAcc<R>{sE[2] + r, T::EX, T::EX * T::EY}, n);
        for_images<DIM>(g, i, j, k, [&](long long t) {
            P.Bn[0][t] = n[0]; P.Bn[1][t] = n[1]; P.Bn[2][t] = n[2];
        });
    }
}

// The same work in pieces, in place: a B half step (with the current cleared), and the E
// update.  The first half step of a call, and every step of the 3-D Lehe update, whose wide
// stencil would make a tile recompute four times its own cells.
template <typename R, int DIM, bool LEHE>
__global__ __launch_bounds__(256) void k_field_b(GridP g, FieldC<R> c, FieldStepP<R> P)
{
    if (gate_closed(P.gate)) return;
    const long long nt = (long long)g.nx * g.ny * (DIM == 3 ? g.nz : 1);
    const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
    if (t >= nt) return;
    const int i = 3 + (int)(t % g.nx), j = 3 + (int)((t / g.nx) % g.ny), k = DIM == 3 ? 3 + (int)(t / ((long long)g.nx * g.ny)) : 1;
    const long long o = fidx(g, i, j, k), sy = g.mx, sz = (long long)g.mx * g.my;
    R b[3] = {P.B[0][o], P.B[1][o], P.B[2][o]};
    b_half<R, DIM, LEHE>(c, MemAcc<R>{P.E[0] + o, sy, sz}, MemAcc<R>{P.E[1] + o, sy, sz},
                         MemAcc<R>{P.E[2] + o, sy, sz}, b);
    for_images<DIM>(g, i, j, k, [&](long long q) {
#pragma unroll
        for (int m = 0; m < 3; m++) {
            P.Bn[m][q] = b[m];
            if (P.Jz[m]) P.Jz[m][q] = 0.0;
        }
    });
}

template <typename R, int DIM>
__global__ __launch_bounds__(256) void k_field_e(GridP g, FieldC<R> c, FieldStepP<R> P)
{
    if (gate_closed(P.gate)) return;
    const long long nt = (long long)g.nx * g.ny * (DIM == 3 ? g.nz : 1);
    const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
    if (P.host && t == 0) {
        volatile int *h = P.host;
        h[0] = *P.spill; h[1] = *P.err; h[2] = *P.gate.stop;
    }
    if (t >= nt) return;
    const int i = 3 + (int)(t % g.nx), j = 3 + (int)((t / g.nx) % g.ny), k = DIM == 3 ? 3 + (int)(t / ((long long)g.nx * g.ny)) : 1;
    const long long o = fidx(g, i, j, k), sy = g.mx, sz = (long long)g.mx * g.my;
    double v[3], J[3];
#pragma unroll
    for (int m = 0; m < 3; m++) {
        v[m] = sizeof(R) == 8 ? (double)P.E[m][o] : (double)P.E[m][o] + (double)P.L[m][o];
        J[m] = P.fold ? folded<DIM>(g, P.J[m], i, j, k) : P.J[m][o];
    }
    e_step<R, DIM>(c, MemAcc<R>{P.B[0] + o, sy, sz}, MemAcc<R>{P.B[1] + o, sy, sz}, MemAcc<R>{P.B[2] + o, sy, sz}, J, v);
    const R h[3] = {(R)v[0], (R)v[1], (R)v[2]};
    for_images<DIM>(g, i, j, k, [&](long long q) {
#pragma unroll
        for (int m = 0; m < 3; m++) {
            P.En[m][q] = h[m];
            if (sizeof(R) == 4) P.Ln[m][q] = (float)(v[m] - (double)h[m]);
        }
    });
}

template <typename R, int DIM, bool LEHE>
void launch_step(const GridP &g, const FieldC<R> &c, const FieldStepP<R> &P, hipStream_t s)
{
    using T = FieldTile<DIM, LEHE>;
    const dim3 grid((unsigned)(((g.nx + T::TX - 1) / T::TX) * ((g.ny + T::TY - 1) / T::TY) *
                               (DIM == 3 ? (g.nz + T::TZ - 1) / T::TZ : 1)));
    hipLaunchKernelGGL((k_field_step<R, DIM, LEHE>), grid, dim3(T::BS), 0, s, g, c, P);
}

inline dim3 cells_grid(const GridP &g)
{
    return dim3((unsigned)(((long long)g.nx * g.ny * (g.ndim == 3 ? g.nz : 1) + 255) / 256));
}

}  // namespace

template <typename R>
FieldC<R> field_consts(const PhysP &ph, double jscale)
{
    FieldC<R> c{};
    c.hc = (R)ph.fld_halfc; c.fc = (R)ph.fldc;
    c.idx = (R)ph.inv_dx; c.idy = (R)ph.inv_dy; c.idz = (R)ph.inv_dz;
    c.dfc = ph.fldc; c.dix = ph.inv_dx; c.diy = ph.inv_dy; c.diz = ph.inv_dz;
    c.jscale = jscale;
    const double *l = ph.lehe;
    c.L = LeheP<R>{(R)l[0], (R)l[1], (R)l[2], (R)l[3], (R)l[4], (R)l[5], (R)l[6], (R)l[7], (R)l[8], (R)l[9], (R)l[10],
                   (R)l[11]};
    return c;
}

template <typename R>
void launch_field_step(const GridP &g, const PhysP &ph, double jscale, const FieldStepP<R> &P, hipStream_t s)
{
    const FieldC<R> c = field_consts<R>(ph, jscale);
    if (g.ndim == 3) launch_step<R, 3, false>(g, c, P, s);
    else if (ph.fdtd) launch_step<R, 2, true>(g, c, P, s);
    else launch_step<R, 2, false>(g, c, P, s);
}

template <typename R>
void launch_field_b(const GridP &g, const PhysP &ph, const FieldStepP<R> &P, hipStream_t s)
{
    const FieldC<R> c = field_consts<R>(ph, 1.0);
    const dim3 grid = cells_grid(g);
    if (g.ndim == 3 && ph.fdtd) hipLaunchKernelGGL((k_field_b<R, 3, true>), grid, dim3(256), 0, s, g, c, P);
    else if (g.ndim == 3) hipLaunchKernelGGL((k_field_b<R, 3, false>), grid, dim3(256), 0, s, g, c, P);
    else if (ph.fdtd) hipLaunchKernelGGL((k_field_b<R, 2, true>), grid, dim3(256), 0, s, g, c, P);
    else hipLaunchKernelGGL((k_field_b<R, 2, false>), grid, dim3(256), 0, s, g, c, P);
}

template <typename R>
void launch_field_e(const GridP &g, const PhysP &ph, double jscale, const FieldStepP<R> &P, hipStream_t s)
{
    const FieldC<R> c = field_consts<R>(ph, jscale);
    if (g.ndim == 3) hipLaunchKernelGGL((k_field_e<R, 3>), cells_grid(g), dim3(256), 0, s, g, c, P);
    else hipLaunchKernelGGL((k_field_e<R, 2>), cells_grid(g), dim3(256), 0, s, g, c, P);
}

#define INST(R)                                                                                                  \
    template void launch_field_step<R>(const GridP &, const PhysP &, double, const FieldStepP<R> &, hipStream_t); \
    template void launch_field_b<R>(const GridP &, const PhysP &, const FieldStepP<R> &, hipStream_t);           \
    template void launch_field_e<R>(const GridP &, const PhysP &, double, const FieldStepP<R> &, hipStream_t);
INST(float)
INST(double)
#undef INST

}  // namespace pictor
